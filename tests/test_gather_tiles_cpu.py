"""The gathered output GEMM as its tiles run it: every tile once, K chunks of whole quads,
split-K partials in disjoint parts of the workspace, their sum equal to the plain form's
product and to the oracle."""
import numpy as np
import pytest


def _tiles(hp, T, rb, y):
    import emulate
    P, G = hp.parts, hp.parts["g2_groups"]
    ws = np.full(max(int(hp.sizes["ws2"]), 1), np.nan)
    src, quad, row = P["gather_srcs"], P["gather_quads"], P["gather_rows"]
    seen = set()
    parts = []
    for gi, g in enumerate(G):
        M, N, K, split, kchunk = (int(g[k]) for k in ("M", "N", "K", "split", "kchunk"))
        assert 0 <= int(g["gq"]) <= len(quad) - K // 4 and 0 <= int(g["grow"]) <= len(row) - M
        if split > 1:
            assert kchunk % 16 == 0 and (split - 1) * kchunk < K <= split * kchunk
            parts.append((int(g["part"]), int(g["part"]) + split * M * N))
    parts.sort()
    assert all(a[1] <= b[0] for a, b in zip(parts, parts[1:])) and (not parts or parts[-1][1] <= ws.size)
    for t in P["g2_tiles"]:
        if t["g"] < 0:
            continue
        key = tuple(int(t[k]) for k in ("g", "mt", "nt", "ks"))
        assert key not in seen
        seen.add(key)
        gi, mt, nt, ks = key
        g = G[gi]
        M, N, K, split, kchunk, tm, tn = (int(g[k]) for k in ("M", "N", "K", "split", "kchunk", "tm", "tn"))
        rows = range(mt * tm, min(M, (mt + 1) * tm))
        cols = slice(nt * tn, min(N, (nt + 1) * tn))
        k0, k1 = (ks * kchunk, min(K, (ks + 1) * kchunk)) if split > 1 else (0, K)
        A = np.zeros((len(rows), k1 - k0))
        for q in range(k0 // 4, k1 // 4):
            d = quad[int(g["gq"]) + q]
            c0, n = int(d["k0len"]) >> 3, int(d["k0len"]) & 7
            for i, m in enumerate(rows):
                r = row[int(g["grow"]) + m]
                e = src[int(d["desc"]) + int(r["strip"])]
                if e["off"] >= 0:
                    at = int(e["off"]) + int(r["row"]) + (c0 + np.arange(n)) * int(r["ld"])
                    A[i, 4 * q - k0:4 * q - k0 + n] = e["coef"] * T[at]
        out = A @ emulate._mat(rb, int(g["b"]), K, N, int(g["ldb"]))[k0:k1, cols]
        if split > 1:
            emulate._mat(ws, int(g["part"]) + ks * M * N, M, N, M)[rows.start:rows.stop, cols] = out
        else:
            emulate._mat(y, int(g["c"]), M, N, int(g["ldc"]))[rows.start:rows.stop, cols] = out
    for gi, g in enumerate(G):
        M, N, split = int(g["M"]), int(g["N"]), int(g["split"])
        want = {(gi, m, n, s) for m in range(-(-M // int(g["tm"]))) for n in range(-(-N // int(g["tn"])))
                for s in range(split)}
        assert want == {k for k in seen if k[0] == gi}
        if split > 1:
            emulate._mat(y, int(g["c"]), M, N, int(g["ldc"]))[...] = sum(
                emulate._mat(ws, int(g["part"]) + s * M * N, M, N, M) for s in range(split))


@pytest.mark.parametrize("symm,L,m,site", [("su2u1", 6, 3, 2), ("su2u1", 6, 30, 2), ("su2u1", 8, 64, 3), ("2u1", 6, 20, 2)])
def test_tiles_of_the_gathered_gemm(oracle_engine, symm, L, m, site):
    import emulate
    from qcmaquis_amd.desc import SiteDesc
    from qcmaquis_amd.gpu import HostPlan
    from qcmaquis_amd.workload import centre_problem
    p = centre_problem(oracle_engine, L, m=m, symm=symm, site=site)
    sd = SiteDesc(p.ham.symm, p.psi.phys, p.psi.left, p.psi.right, p.W, p.L.layout, p.R.layout)
    plain, hp = HostPlan(sd, "sigma"), HostPlan(sd, "sigma", gather=True)
    s, P = hp.sizes, hp.parts
    assert (P["g2_groups"]["split"] > 1).any()
    la, rb, prp = np.zeros(max(s["la"], 1)), np.zeros(max(s["rb"], 1)), np.zeros(max(s["prp"], 1))
    T, y = np.full(max(s["t"], 1), np.nan), np.full(s["vec"], np.nan)
    x = np.random.default_rng(m).standard_normal(s["vec"])
    emulate.copy2d(P["arrL"], p.L.data, la)
    emulate.wapply(P["comb_strips"], P["comb_srcs"], la, la)
    emulate.copy2d(P["arrR"], p.R.data, rb)
    emulate.copy2d(P["reshape"], x, prp)
    emulate.gemm(P["g1_groups"], P["g1_tiles"], la, prp, T, P["g1_rowmap"])
    emulate.wapply(P["strips"], P["srcs"], T, T)
    _tiles(hp, T, rb, y)
    # sums of at most 1e5 products in another order: 1e-13 of the largest element
    for ref in (emulate.run_sigma(plain, p.L.data, p.R.data, x), oracle_engine.sigma(
            p.ham.symm, p.psi, p.L, p.R, p.W, x=x)[0]):
        assert np.abs(y - ref).max() <= 1e-13 * np.abs(ref).max()
