"""The Jacobi-Davidson driver's device orthonormalisation and Ritz kernels: bases beyond one
launch's coefficients (48 vectors), vectors shorter and longer than a workgroup, constraint
vectors, and a start vector that needs the second Gram-Schmidt pass."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def problems(oracle_engine, gpu_engine):
    from qcmaquis_amd.workload import centre_problem
    out = {}
    for m in (2, 24):
        p = centre_problem(oracle_engine, 8, m=m)
        n = p.psi.to_flat().size
        H = np.stack([oracle_engine.sigma(p.ham.symm, p.psi, p.L, p.R, p.W, x=e)[0] for e in np.eye(n)], 1)
        Lg = gpu_engine.upload_boundary(p.L.layout, p.L.data)
        Rg = gpu_engine.upload_boundary(p.R.layout, p.R.data)
        out[m] = (p, 0.5 * (H + H.T), gpu_engine.sigma_plan(p.ham.symm, p.psi, Lg, Rg, p.W))
    yield out
    for _, _, sp in out.values():
        sp.close()


@pytest.mark.parametrize("m,max_iter,n_ortho", [(2, 3, 0), (24, 10, 0), (24, 70, 0), (24, 70, 3), (24, 130, 1)])
def test_jd_against_dense(problems, gpu_engine, m, max_iter, n_ortho):
    p, H, sp = problems[m]
    n = H.shape[0]
    print(f"m {m} n {n} max_iter {max_iter} ortho {n_ortho}", flush=True)
    rng = np.random.default_rng(m + max_iter)
    w, U = np.linalg.eigh(H)
    live = np.abs(H).sum(0) > 0
    O = [U[:, np.argsort(w)[k]] for k in range(n_ortho)]
    # project the constraints out of H: the driver's Ritz pair minimises over their complement
    Q = np.stack(O, 1) if O else np.zeros((n, 0))
    P = np.eye(n) - Q @ Q.T
    x = np.where(live, rng.standard_normal(n), 0.0)
    its = min(max_iter, n - n_ortho)
    th, u, it = sp.jd(gpu_engine.to_dev(x), its, 1e-11, ortho=O)
    u = u.cpu().numpy()
    assert abs(u @ u - 1) <= 1e-12  # orthonormal basis and unit coefficients
    assert np.abs(Q.T @ u).max(initial=0.0) <= 1e-10
    assert abs(u @ H @ u - th) <= 1e-11 * max(1.0, abs(th))
    r = P @ (H @ u) - th * u
    if it < its:  # converged to the tolerance
        assert np.linalg.norm(r) <= 1.01e-11 * max(1.0, abs(th)) + 1e-12 * np.abs(w).max()
    # the same Krylov space in numpy: Lanczos on P H P from the projected start
    v = P @ x
    K = [v / np.linalg.norm(v)]
    for _ in range(it - 1):
        t = P @ (H @ K[-1])
        for _ in range(2):
            for q in K:
                t = t - (q @ t) * q
        K.append(t / np.linalg.norm(t))
    B = np.stack(K, 1)
    low = np.linalg.eigvalsh(B.T @ H @ B)[0]
    assert abs(low - th) <= 1e-9 * max(1.0, abs(low)), (low, th, it)


def test_start_vector_of_huge_and_tiny_norm(problems, gpu_engine):
    p, H, sp = problems[24]
    x = np.where(np.abs(H).sum(0) > 0, np.random.default_rng(1).standard_normal(H.shape[0]), 0.0)
    ref = sp.jd(gpu_engine.to_dev(x), 12, 0.0)
    for s in (1e-120, 1e120):
        got = sp.jd(gpu_engine.to_dev(s * x), 12, 0.0)
        assert got[2] == ref[2] and abs(got[0] - ref[0]) <= 1e-12 * abs(ref[0])
