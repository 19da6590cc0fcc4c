"""Launches that change no result, at sizes where each is taken: the walk's
workgroups heaviest first (more than 2,048 groups), with every unit's cost held
by the plan and with more units than that, and a batch's direct sums by few and
by many workgroups, each taking several blocks."""
import numpy as np
import pytest

import gsim
import helpers as H

pytestmark = pytest.mark.gpu


def _same(a, b):
    assert np.array_equal(a.pos, b.pos)
    assert np.array_equal(a.vel, b.vel)
    assert np.array_equal(a.mass, b.mass)


@pytest.mark.parametrize("n,w", [(131_137, 64), (150_000, 64), (65_600, 32), (150_000, 32),
                                 (600_000, 32)])  # the last: 4,688 units of four groups
def test_heaviest_first_walks_the_same(n, w):
    p = gsim.generate("galaxy", n, 100.0, 1.0, 10.0, seed=n)
    units = (p.padded().n // w + 3) // 4
    out = []
    for order in (0, 1, 2):
        with gsim.Simulation(p, "barnes-hut", group_width=w, accuracy_parameter=0.8) as s:
            s.set_tuning(gsim.TUNE_BH_ORDER, order)
            s.step(10)  # index order, a plan, and a second one; the trial of mode 2
            plan = H.launch_order(s, units)
            assert (plan is None) == (order == 0)
            if order:
                assert np.array_equal(np.sort(plan), np.arange(units))
                assert not np.array_equal(plan, np.arange(units))
            out.append(s.read())
    _same(out[0], out[1])
    _same(out[0], out[2])


@pytest.mark.parametrize("bh,groups", [(0, 1024), (40_000, 1024), (100_000, 256)])
def test_batch_direct_sums_by_few_and_many_workgroups(bh, groups):
    specs = [(9_000, "direct-sum"), (8_990, "direct-sum"), (64, "direct-sum")]
    if bh:
        specs.insert(1, (bh, "barnes-hut"))
    ps = [gsim.generate("galaxy", n, 100.0, 1.0, 10.0, seed=n) for n, _ in specs]
    with gsim.Batch(400_000, 8) as b:
        ids = [b.add(p, a) for p, (_, a) in zip(ps, specs)]
        b.step(3)
        got = [b.read(i) for i in ids]
        taken, blocks = H.direct_sum_launch(b)
    assert taken == groups and blocks > 1024
    for p, (_, a), g in zip(ps, specs, got):
        with gsim.Simulation(p, a) as s:
            s.step(3)
            _same(g, s.read())
