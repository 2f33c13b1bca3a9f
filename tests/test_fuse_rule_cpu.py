"""Which MPO columns a sigma plan sums on the left boundary first (MQ_OPT_FUSE mode 1): a
column's entries against its distinct positions, counted here from the MPO alone; many
entries per output state do not fuse a column.  Plans of one column each: it has
combination strips exactly when it is fused."""
import copy
from collections import Counter

import pytest


class _W:
    pass


def _one_column(a, b2):
    """MPO arrays a with the terms of every other column left out."""
    m = copy.copy(a)
    p0, p1 = int(a.col_ptr[b2]), int(a.col_ptr[b2 + 1])
    m.col_ptr = a.col_ptr * 0
    m.col_ptr[b2 + 1:] = p1 - p0
    m.row_idx = a.row_idx[p0:p1].copy()
    m.term_ptr = a.term_ptr[p0:p1 + 1] - a.term_ptr[p0]
    t0, t1 = int(a.term_ptr[p0]), int(a.term_ptr[p1])
    m.term_op, m.term_scale = a.term_op[t0:t1].copy(), a.term_scale[t0:t1].copy()
    w = _W()
    w._mq_arrays = m
    return w


def _counts(a, b2, phys):
    """(entries, distinct positions, output states) of column b2."""
    ids = {c: i for i, (c, _) in enumerate(phys)}
    n, pos, outs = 0, set(), set()
    for p in range(int(a.col_ptr[b2]), int(a.col_ptr[b2 + 1])):
        for t in range(int(a.term_ptr[p]), int(a.term_ptr[p + 1])):
            o = int(a.term_op[t])
            for b in range(int(a.op_bptr[o]), int(a.op_bptr[o + 1])):
                cin, cout = (tuple(int(v) for v in x[2 * b:2 * b + 2]) for x in (a.opb_in, a.opb_out))
                if cin not in ids or cout not in ids:
                    continue
                for e in range(int(a.opb_eptr[b]), int(a.opb_eptr[b + 1])):
                    out = (cout, int(a.ent_col[e]))
                    n += 1
                    outs.add(out)
                    pos.add((out, cin, int(a.ent_row[e]), int(a.ent_rspin[e]), int(a.ent_cspin[e]),
                             int(a.op_spin[o]), int(a.left_spin[a.row_idx[p]])))
    return n, len(pos), len(outs)


def _kind(n, pos, outs, ratio, least):
    if n < max(least, 1):
        return "few"
    if n >= ratio * pos:
        return "positions"
    return "outputs" if n >= 2 * ratio * outs else "short"


@pytest.mark.parametrize("symm,site,ratio,least,expect", [
    ("su2u1", 3, 4, 64, {"positions", "outputs", "few"}),
    ("su2u1", 1, 4, 64, {"outputs", "few"}),
    ("su2u1", 2, 3, 16, {"outputs", "short", "few"}),
    ("2u1", 3, 4, 64, {"positions", "few"}),
    ("2u1", 3, 6, 16, {"outputs", "few"}),
])
def test_fused_columns(oracle_engine, symm, site, ratio, least, expect):
    from qcmaquis_amd.desc import SiteDesc, mpo_arrays
    from qcmaquis_amd.gpu import HostPlan
    from qcmaquis_amd.workload import centre_problem
    p = centre_problem(oracle_engine, 8, m=20, symm=symm, site=site)
    a = mpo_arrays(p.W)
    seen = Counter()
    for b2 in range(a.col_dim):
        kind = _kind(*_counts(a, b2, p.psi.phys), ratio, least)
        if seen[kind] == 4:
            continue
        sd = SiteDesc(p.ham.symm, p.psi.phys, p.psi.left, p.psi.right, _one_column(a, b2), p.L.layout, p.R.layout)
        if not len(HostPlan(sd, "sigma", 2).parts["comb_strips"]):
            continue  # nothing of this column reaches the site
        seen[kind] += 1
        for gather in (False, True):
            hp = HostPlan(sd, "sigma", 1, fuse_ratio=ratio, fuse_min=least, gather=gather)
            assert (len(hp.parts["comb_strips"]) > 0) == (kind == "positions"), (b2, kind)
    assert expect <= set(seen), seen
