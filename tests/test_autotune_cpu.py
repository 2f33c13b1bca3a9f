"""The tuner does not time a K chunk whose plan is the default's: a launch that does not
fill the GPU gets the same chunk, below all of them."""
import dataclasses
import types

import numpy as np
import pytest


class _Plan:
    def __init__(self, eng, sched):
        self.eng, self.sched = eng, sched
        chunk = min(sched.kchunk, eng.fill)
        other = dataclasses.astuple(dataclasses.replace(sched, kchunk=0))
        self.exec_flops = 1e9 + hash(other) % 1000
        self.workspace_bytes = 10**6 + 4096 // chunk

    def apply(self, x, y, prec=None):
        return y

    def timed(self, x, y, prec=None):
        self.eng.timed.add(self.sched)
        return [0.0, 1.0 / (1 + len(self.eng.timed))], None  # later ones look faster

    def close(self):
        pass


class _Engine:
    torch = types.SimpleNamespace(empty_like=np.empty_like)

    def __init__(self, fill):
        from qcmaquis_amd.autotune import DEFAULT
        self.fill, self.timed, self.schedule = fill, set(), DEFAULT

    def set_schedule(self, s):
        self.schedule = s

    def to_dev(self, x):
        return x

    def sigma_plan(self, *a):
        return _Plan(self, self.schedule)


@pytest.mark.parametrize("fill,timed", [(256, {2048}), (1024, {2048}), (1500, {1024, 2048}), (10**6, {1024, 2048, 4096})])
def test_equal_plans_are_not_timed(fill, timed):
    from qcmaquis_amd.autotune import DEFAULT, candidates, tune
    psi = types.SimpleNamespace(to_flat=lambda: np.ones(4))
    b = types.SimpleNamespace(layout=types.SimpleNamespace(total=3))
    W = types.SimpleNamespace(row_dim=2, col_dim=2)
    eng = _Engine(fill)
    best, table = tune(eng, "su2u1", psi, b, b, W, reps=1)
    assert len(table) == len(candidates())
    rows = {r[0]: r[1:] for r in table}
    chunks = {s.kchunk for s in eng.timed if dataclasses.replace(s, kchunk=DEFAULT.kchunk) == DEFAULT}
    assert chunks == timed
    for s in candidates():
        if dataclasses.replace(s, kchunk=DEFAULT.kchunk) == DEFAULT and s.kchunk not in timed:
            assert rows[s] == rows[DEFAULT]
            assert best != s
