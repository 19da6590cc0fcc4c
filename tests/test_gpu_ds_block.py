"""The direct sum's block form (below 16,384 padded particles) where its split
changes: fewer sixteens of sources than roles, a ragged last round, one and
several rounds in flight, the largest size.  Forces within 1e-5 system-relative
of the FP32 oracle and per particle no further from FP64 than 1.5x the oracle's
own sums, the integration bit-exact on those forces, and the same bits in a
batch."""
import numpy as np
import pytest

import gsim
import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu

EPS2 = H.sq32(0.2)


@pytest.mark.parametrize("rcp", [0, 1])
@pytest.mark.parametrize("n", [1, 64, 250, 256, 300, 1024, 1025, 4160, 16320])
def test_block_forces_and_batch(n, rcp):
    print(f"ds block n={n} rcp={rcp}", flush=True)
    p = gsim.generate("galaxy", n, 50.0, 1.0, 10.0, seed=n)
    with gsim.Simulation(p, "direct-sum") as s:
        s.set_debug(gsim.DEBUG_ACCEL)
        s.set_tuning(gsim.TUNE_DS_RCP, rcp)
        s.step(1)
        a = s.dump(gsim.DUMP_ACCEL)[: p.n]
        g = s.read()
    pp = p.padded()
    ref = O.ds_accel_f32(pp.pos, pp.mass, EPS2)[: p.n]
    ref64 = O.ds_accel_f64(pp.pos, pp.mass, EPS2)[: p.n]
    if n == 1:
        assert np.array_equal(a, np.zeros_like(a))
    else:
        assert H.system_rel_err(a, ref) <= 1e-5
        worst = H.per_particle_rel(ref, ref64).max()
        assert H.per_particle_rel(a, ref64).max() <= max(1.5 * worst, 1e-6)
    nv = (p.vel + a * np.float32(1e-3)).astype(np.float32)
    assert np.array_equal(g.vel, nv)
    assert np.array_equal(g.pos, (p.pos + ((p.vel + nv) * np.float32(0.5)) * np.float32(1e-3))
                          .astype(np.float32))
    if rcp:
        return
    with gsim.Batch(max(8 * pp.n, 65536), 4) as b:  # its direct-sum admission rule needs 8n
        k = b.add(p, "direct-sum")
        b.step(1)
        q = b.read(k)
    assert np.array_equal(q.pos, g.pos) and np.array_equal(q.vel, g.vel)


@pytest.mark.parametrize("n", [28608, 28672, 65473, 131073, 262145])
def test_symmetric_forces_at_every_tile_shape(n):
    """The symmetric form on both sides of the sizes where its tile changes:
    forces of 512 targets within 1e-5 system-relative of the FP64 sum (FP32
    sums of a few hundred terms each, added in order)."""
    print(f"ds symmetric n={n}", flush=True)
    p = gsim.generate("exponential-disk", n, 100.0, 1.0, 10.0, seed=n)
    with gsim.Simulation(p, "direct-sum") as s:
        s.set_debug(gsim.DEBUG_ACCEL)
        s.step(1)
        a = s.dump(gsim.DUMP_ACCEL)[: p.n]
    t = np.sort(np.random.default_rng(n).choice(n, 512, replace=False)).astype(np.uint32)
    t[0], t[-1] = 0, n - 1
    pp = p.padded()
    ref64 = O.ds_accel_f64_at(pp.pos, pp.mass, EPS2, t)
    assert np.isfinite(a).all()
    assert H.system_rel_err(a[t], ref64) <= 1e-5
    # momentum: every pair gave equal and opposite pulls
    f = (a.astype(np.float64) * p.mass[:, None])
    assert np.linalg.norm(f.sum(0)) <= 1e-5 * np.linalg.norm(f, axis=1).sum()


@pytest.mark.parametrize("cols", [1, 2])
@pytest.mark.parametrize("n", [16384, 20000, 28607, 40000])
def test_symmetric_forces_with_the_columns_asked_for(n, cols):
    """As by size, with each number of column blocks a wave."""
    print(f"ds symmetric n={n} cols={cols}", flush=True)
    p = gsim.generate("exponential-disk", n, 100.0, 1.0, 10.0, seed=n)
    with gsim.Simulation(p, "direct-sum") as s:
        s.set_debug(gsim.DEBUG_ACCEL)
        s.set_tuning(gsim.TUNE_DS_SYM_COLS, cols)
        s.step(1)
        a = s.dump(gsim.DUMP_ACCEL)[: p.n]
    pp = p.padded()
    t = np.linspace(0, n - 1, 512).astype(np.uint32)
    assert H.system_rel_err(a[t], O.ds_accel_f64_at(pp.pos, pp.mass, EPS2, t)) <= 1e-5
