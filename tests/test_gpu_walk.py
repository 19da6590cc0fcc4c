"""The Barnes-Hut walk at the group counts where its launch changes (waves per
group) and on trees that fill its stack of cells and its list of sources: visit
and acceptance counts equal the oracle's on the same tree, and forces within
1e-5 system-relative of the FP32 oracle's, per particle no further from the
same terms in double than 1.5x the oracle's own sums (the walk adds them in
another order)."""
import numpy as np
import pytest

import gsim
import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu

EPS2 = H.sq32(0.2)


def _check(p, W, theta, bits=10):
    with gsim.Simulation(p, "barnes-hut", accuracy_parameter=theta, group_width=W) as s:
        if bits != 10:
            s.set_tuning(gsim.TUNE_BH_LEAF_BITS, bits)
        s.set_debug(gsim.DEBUG_ACCEL)
        s.step(1)
        a = s.dump(gsim.DUMP_ACCEL)
        counts = tuple(int(x) for x in s.dump(gsim.DUMP_COUNTERS))
        t = s.tree()
    pp = p.padded()
    _, _, _, pk, mk = O.bh_build(pp.pos, pp.mass, bits=bits)
    oa, oV, oA, _, _, oa64 = O.bh_traverse(t, pk, mk, EPS2, H.sq32(theta), W=W, f64=True)
    assert counts == (oV, oA)
    inside = t["sorted_src"][t["sorted_src"] < len(mk)]
    a, oa, oa64 = a[inside], oa[inside], oa64[inside]
    assert H.system_rel_err(a, oa) <= 1e-5
    assert H.per_particle_rel(a, oa64).max() <= max(1.5 * H.per_particle_rel(oa, oa64).max(), 1e-6)


@pytest.mark.parametrize("n,W", [(1, 64), (1, 32), (2, 64), (65, 32), (256 * 64, 64),
                                 (256 * 64 + 1, 64), (256 * 32 + 1, 32), (512 * 64 + 1, 64),
                                 (512 * 32 + 1, 32), (2048 * 64 + 1, 64), (2048 * 32 + 1, 32)])
def test_walk_at_every_number_of_waves_per_group(n, W):
    print(f"walk n={n} W={W}", flush=True)
    _check(gsim.generate("exponential-disk", n, 100.0, 1.0, 10.0, seed=n), W, 0.7)


@pytest.mark.parametrize("W", [64, 32])
@pytest.mark.parametrize("bits", [10, 15])
@pytest.mark.parametrize("theta", [0.0, 0.1])
def test_walk_that_opens_almost_every_cell(theta, bits, W):
    """Thousands of cells open at once (the stack's limit), leaves of one and of
    hundreds of particles (lists that end anywhere in a block of 32), and killed
    particles at the end of the order."""
    rng = np.random.default_rng(7)
    pos = rng.uniform(-480, 480, size=(5000, 2)).astype(np.float32)
    pos[:700] = rng.normal(60.3, 0.05, size=(700, 2))
    pos[700:733] = [[900, 0]] * 33
    p = gsim.Particles(pos, np.zeros_like(pos), rng.uniform(1, 10, 5000).astype(np.float32))
    print(f"walk theta={theta} bits={bits} W={W}", flush=True)
    _check(p, W, theta, bits)
