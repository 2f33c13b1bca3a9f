"""BF16x3 sigma vectors of small problems near a chain's end are as exact as with every MPO
term applied on its own: no column is summed on the boundary first whose terms hardly
merge (one bf16 split of a sum has no averaging of the terms' rounding errors)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,site", [(30, 1), (60, 2)])
def test_bf16x3_is_as_exact_as_term_by_term(oracle_engine, gpu_engine, m, site):
    from qcmaquis_amd.desc import MQ_PREC_BF16X3
    from qcmaquis_amd.workload import centre_problem
    print(f"L 8 m {m} site {site}", flush=True)
    p = centre_problem(oracle_engine, 8, m=m, site=site)
    Lg = gpu_engine.upload_boundary(p.L.layout, p.L.data)
    Rg = gpu_engine.upload_boundary(p.R.layout, p.R.data)
    n = p.psi.to_flat().size
    err = {0: 0.0, 1: 0.0}
    for mode in err:
        gpu_engine.set_fuse(mode)
        try:
            sp = gpu_engine.sigma_plan(p.ham.symm, p.psi, Lg, Rg, p.W)
        finally:
            gpu_engine.set_fuse(1)
        for seed in range(4):
            x = np.random.default_rng(seed).standard_normal(n)
            ref, _ = oracle_engine.sigma(p.ham.symm, p.psi, p.L, p.R, p.W, x=x)
            y = sp.apply(gpu_engine.to_dev(x), prec=MQ_PREC_BF16X3)
            gpu_engine.sync()
            err[mode] += np.linalg.norm(y.cpu().numpy() - ref) / np.linalg.norm(ref) / 4
        sp.close()
    print(err, flush=True)
    # two orders of the same sums: their mean errors differ by less than a tenth
    assert err[1] <= 1.1 * err[0]
