"""Split-K of a plan's output GEMM: long K loops of small problems are cut so that the
launch has many tiles, and the chunks cover K."""
import pytest



@pytest.mark.parametrize("m", [16, 64])
def test_long_k_loops_of_small_problems_are_cut(oracle_engine, m):
    import emulate
    import numpy as np
    from qcmaquis_amd.desc import SiteDesc
    from qcmaquis_amd.gpu import HostPlan
    from qcmaquis_amd.workload import centre_problem
    p = centre_problem(oracle_engine, 8, m=m)
    hp = HostPlan(SiteDesc(p.ham.symm, p.psi.phys, p.psi.left, p.psi.right, p.W, p.L.layout, p.R.layout), "sigma")
    g = hp.parts["g2_groups"]
    tiles = -(-g["M"] // g["tm"]) * -(-g["N"] // g["tn"])
    total = int((tiles * g["K"]).sum())
    chunk = min(2048, max(128, (total // 1024 + 15) // 16 * 16))
    for x, t in zip(g, tiles):
        if x["K"] > 2 * chunk and t < 64:
            assert x["split"] > 1 and x["kchunk"] % 16 == 0 and x["split"] <= 64
            assert (x["split"] - 1) * x["kchunk"] < x["K"] <= x["split"] * x["kchunk"]
        else:
            assert x["split"] == 1
    assert (g["split"] > 1).any()
    x = np.random.default_rng(m).standard_normal(hp.sizes["vec"])
    y, _ = oracle_engine.sigma(p.ham.symm, p.psi, p.L, p.R, p.W, x=x)
    ye = emulate.run_sigma(hp, p.L.data, p.R.data, x)
    # sums of at most 1e5 products in another order: 1e-13 of the largest element
    assert np.abs(y - ye).max() <= 1e-13 * np.abs(y).max()
