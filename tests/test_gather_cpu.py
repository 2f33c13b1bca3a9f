"""The gathered form of a sigma plan (the device's): its lists, executed in numpy, equal
the plain form's C panel products and the oracle, in both symmetries, for sector sizes
around the quads of four K columns, every fuse rule and the chain's ends."""
import numpy as np
import pytest


def _run(hp, L, R, x):
    import emulate
    s, P = hp.sizes, hp.parts
    la, rb, prp = np.zeros(max(s["la"], 1)), np.zeros(max(s["rb"], 1)), np.zeros(max(s["prp"], 1))
    T, y = np.full(max(s["t"], 1), np.nan), np.full(s["vec"], np.nan)
    emulate.copy2d(P["arrL"], L, la)
    emulate.wapply(P["comb_strips"], P["comb_srcs"], la, la)
    emulate.copy2d(P["arrR"], R, rb)
    emulate.copy2d(P["reshape"], x, prp)
    emulate.gemm(P["g1_groups"], P["g1_tiles"], la, prp, T, P["g1_rowmap"])
    emulate.wapply(P["strips"], P["srcs"], T, T)
    for st in P["strips"]:  # only sums of several sources are written, each block contiguous
        assert st["s1"] - st["s0"] >= 2 and st["ldd"] == st["rows"]
    src, quad, row = P["gather_srcs"], P["gather_quads"], P["gather_rows"]
    for g in P["g2_groups"]:
        M, N, K = int(g["M"]), int(g["N"]), int(g["K"])
        assert K % 4 == 0
        A = np.zeros((M, K))
        for q in range(K // 4):
            d = quad[int(g["gq"]) + q]
            k0, n = int(d["k0len"]) >> 3, int(d["k0len"]) & 7
            assert 1 <= n <= 4
            for m in range(M):
                r = row[int(g["grow"]) + m]
                e = src[int(d["desc"]) + int(r["strip"])]
                if e["off"] < 0:
                    continue
                for u in range(n):
                    A[m, 4 * q + u] = e["coef"] * T[int(e["off"]) + int(r["row"]) + (k0 + u) * int(r["ld"])]
        B = emulate._mat(rb, int(g["b"]), K, N, int(g["ldb"]))
        emulate._mat(y, int(g["c"]), M, N, int(g["ldc"]))[...] = A @ B
    assert not np.isnan(y).any()
    return y


@pytest.mark.parametrize("symm,m,site", [("su2u1", 3, 2), ("su2u1", 30, 2), ("su2u1", 21, 0), ("2u1", 20, 2),
                                         ("2u1", 9, 4)])
@pytest.mark.parametrize("fuse", [0, 1, 2])
def test_gathered_plan_matches_oracle(oracle_engine, symm, m, site, fuse):
    from qcmaquis_amd.desc import SiteDesc
    from qcmaquis_amd.gpu import HostPlan
    from qcmaquis_amd.workload import centre_problem
    p = centre_problem(oracle_engine, 6, m=m, symm=symm, site=site)
    sd = SiteDesc(p.ham.symm, p.psi.phys, p.psi.left, p.psi.right, p.W, p.L.layout, p.R.layout)
    plain, hp = HostPlan(sd, "sigma", fuse), HostPlan(sd, "sigma", fuse, gather=True)
    assert hp.exec_flops >= plain.exec_flops and hp.ref_flops == plain.ref_flops
    assert np.array_equal(hp.parts["live"], plain.parts["live"])
    assert len(hp.parts["gather_srcs"]) == len(plain.parts["strips"])
    x = np.random.default_rng(m).standard_normal(hp.sizes["vec"])
    y, _ = oracle_engine.sigma(p.ham.symm, p.psi, p.L, p.R, p.W, x=x)
    ye = _run(hp, p.L.data, p.R.data, x)
    # sums of at most 1e4 products in another order: 1e-13 of the largest element
    assert np.abs(y - ye).max() <= 1e-13 * max(np.abs(y).max(), 1e-300)
