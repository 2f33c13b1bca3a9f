"""Fused MPO columns: each C row block has one T source, the panels' operands are packed
psi rows, and the plan equals the oracle in both symmetries, off the chain's centre too,
for every fuse rule (including ratios at which only the output-state rule fuses)."""
import numpy as np
import pytest


@pytest.fixture(scope="module")
def problems(oracle_engine):
    from qcmaquis_amd.workload import centre_problem
    return {(symm, site): centre_problem(oracle_engine, 8, m=30, symm=symm, site=site)
            for symm in ("su2u1", "2u1") for site in (2, 4)}


@pytest.mark.parametrize("symm", ["su2u1", "2u1"])
@pytest.mark.parametrize("site", [2, 4])
@pytest.mark.parametrize("fuse,ratio,mn", [(1, 4, 64), (1, 2, 1), (1, 1, 1), (1, 255, 1), (2, 0, 0)])
def test_fused_plans_match_oracle(problems, oracle_engine, symm, site, fuse, ratio, mn):
    import emulate
    from qcmaquis_amd.desc import SiteDesc
    from qcmaquis_amd.gpu import HostPlan
    p = problems[(symm, site)]
    sd = SiteDesc(p.ham.symm, p.psi.phys, p.psi.left, p.psi.right, p.W, p.L.layout, p.R.layout)
    hp = HostPlan(sd, "sigma", fuse, fuse_ratio=ratio, fuse_min=mn)
    g = hp.parts["g1_groups"]
    fused = g["lda"] == g["M"]
    n = hp.parts["strips"]["s1"] - hp.parts["strips"]["s0"]
    if fuse == 2:
        assert fused.all() and n.max() == 1
    if ratio == 255:
        assert len(hp.parts["comb_strips"]) == 0
    # the packed operand of every panel lies behind the right-paired psi
    vec = hp.sizes["vec"]
    packed = hp.parts["comb_strips"].size > 0
    assert (hp.sizes["prp"] > vec) == packed
    x = np.random.default_rng(site).standard_normal(vec)
    y, _ = oracle_engine.sigma(p.ham.symm, p.psi, p.L, p.R, p.W, x=x)
    ye = emulate.run_sigma(hp, p.L.data, p.R.data, x)
    # sums of at most 1e4 products in another order: 1e-13 of the largest element
    assert np.abs(y - ye).max() <= 1e-13 * np.abs(y).max()
