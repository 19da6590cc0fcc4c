"""The walk's wide form (trees that reach beyond 4 GiB of node records) sums the
same sources in the same order as the narrow one: the same bits, at sizes where
each number of waves a group is taken, at both widths and leaf depths, alone and
in a batch."""
import numpy as np
import pytest

import gsim
import helpers as H

pytestmark = pytest.mark.gpu


def _same(a, b):
    assert np.array_equal(a.pos, b.pos)
    assert np.array_equal(a.vel, b.vel)
    assert np.array_equal(a.mass, b.mass)


@pytest.mark.parametrize("bits", [10, 15])
@pytest.mark.parametrize("n,w,debug", [(1, 64, 0), (1_000, 64, 1), (20_000, 64, 0),
                                       (50_000, 64, 1), (140_000, 64, 0), (140_000, 64, 1),
                                       (1_000, 32, 1), (20_000, 32, 0), (50_000, 32, 1),
                                       (140_000, 32, 0), (140_000, 32, 1)])
def test_wide_walk_equals_the_narrow_one(n, w, debug, bits):
    p = gsim.generate("two-exponential-disks", n, 100.0, 1.0, 10.0, seed=n + w)
    out, acc, work = [], [], []
    for wide in (False, True):
        with gsim.Simulation(p, "barnes-hut", group_width=w, accuracy_parameter=0.8) as s:
            s.set_tuning(gsim.TUNE_BH_LEAF_BITS, bits)
            s.set_debug(gsim.DEBUG_ACCEL if debug else 0)
            if wide:
                H.put_narrow_nodes(s, 0)
            s.step(3)
            out.append(s.read())
            work.append(s.dump(gsim.DUMP_COUNTERS))
            acc.append(s.dump(gsim.DUMP_ACCEL) if debug else None)
    _same(*out)
    assert np.array_equal(*work)
    assert not debug or np.array_equal(*acc)


def test_wide_walk_in_a_batch():
    specs = [(300, "direct-sum", {}), (9_000, "barnes-hut", {}),
             (30_000, "barnes-hut", {"group_width": 32}), (64, "barnes-hut", {})]
    ps = [gsim.generate("galaxy", n, 100.0, 1.0, 10.0, seed=n) for n, _, _ in specs]
    want = []
    for p, (_, a, kw) in zip(ps, specs):
        with gsim.Simulation(p, a, **kw) as s:
            s.step(5)
            want.append(s.read())
    with gsim.Batch(60_000, 8) as b:
        ids = [b.add(p, a, **kw) for p, (_, a, kw) in zip(ps, specs)]
        b.step(2)
        H.put_narrow_nodes(b, 0)  # from here on wide
        b.step(3)
        for i, w in zip(ids, want):
            _same(b.read(i), w)
