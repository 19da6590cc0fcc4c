"""The Barnes-Hut build where its kernels change shape: every node array equals
the oracle's, bit for bit, on the first step and on a third one (whose counters
and look-back words the steps before it have used)."""
import numpy as np
import pytest

import gsim
import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu

TILE = 1000.0 / 32  # edge of a depth-5 cell of the fixed domain


def _same_tree(pos, mass, bits=10, steps=3, boxed=False):
    # padded here: the padding moves with the others, and is read back
    p = gsim.Particles(pos, np.zeros_like(pos), mass).padded()
    with gsim.Simulation(p, "barnes-hut") as s:
        if bits != 10:
            s.set_tuning(gsim.TUNE_BH_LEAF_BITS, bits)
        if boxed:
            s.set_tuning(gsim.TUNE_BH_ADAPTIVE_BOX, 1)
        for k in range(steps):
            pp = s.read() if k else p
            s.step(1)
            if k in (0, steps - 1):
                t = s.tree()
                ot, nn, _, _, _ = O.bh_build(pp.pos, pp.mass, bits=bits,
                                           box=O.bh_box(pp.pos) if boxed else None)
                assert t["total"] == nn, k
                for key in ("sorted_src", "counts", "radii", "node_mass", "node_pos"):
                    assert np.array_equal(t[key], ot[key]), (k, key)


def _tiles(which, per, seed):
    """`per` particles in each depth-5 cell (by its Morton index) of `which`."""
    rng = np.random.default_rng(seed)
    x = np.zeros(len(which), np.int64)
    y = np.zeros(len(which), np.int64)
    for b in range(5):
        x |= ((which >> (2 * b)) & 1) << b
        y |= ((which >> (2 * b + 1)) & 1) << b
    corner = np.stack([x, y], 1) * TILE - 500.0
    pos = np.repeat(corner, per, 0) + rng.uniform(0.05, 0.95, (len(which) * per, 2)) * TILE
    return pos.astype(np.float32), rng.uniform(1, 10, len(pos)).astype(np.float32)


@pytest.mark.parametrize("bits", [10, 15])
@pytest.mark.parametrize("name,which,per", [
    ("one", np.array([1023]), 1), ("one-full", np.array([37]), 1500),
    ("first-of-each-32", np.arange(0, 1024, 32), 3), ("one-32", np.arange(64, 96), 2),
    ("two-of-33", np.array([0, 32]), 5), ("every", np.arange(1024), 1),
    ("every-9", np.arange(1024), 9)])
def test_tree_for_every_pattern_of_occupied_tiles(name, which, per, bits):
    print(f"tiles {name} bits={bits}", flush=True)
    pos, mass = _tiles(which, per, len(which) + per)
    _same_tree(pos, mass, bits)


@pytest.mark.parametrize("bits,boxed", [(10, False), (15, False), (10, True), (15, True)])
@pytest.mark.parametrize("n", [1, 65, 1024, 1025, 5000, 8127, 8192, 8193])
def test_tree_on_both_sides_of_the_one_workgroup_build(n, bits, boxed):
    """Up to 8,192 particles one workgroup sorts and emits them: rows of 64 that
    end anywhere, equal keys, particles outside the domain, and one size more."""
    print(f"small build n={n} bits={bits} boxed={boxed}", flush=True)
    rng = np.random.default_rng(n)
    pos = rng.normal(0, 150, (n, 2)).astype(np.float32)
    pos[: n // 3] = rng.normal(31.2, 0.2, (n // 3, 2))
    pos[n // 3: n // 3 + n // 50] = 7.5
    pos[n // 2: n // 2 + n // 40] = [600, 0]
    _same_tree(pos, rng.uniform(1, 10, n).astype(np.float32), bits, 4, boxed)


@pytest.mark.parametrize("tile", [2048, 3072, 4096])
def test_batch_sorted_by_system_equals_each_system_alone(tile):
    """Systems that end one below, at and one above a radix tile, a group of 16
    tiles, two groups, with particles outside the domain; then members that need
    more sort slots than the first steps' launches had.  Same bits as alone."""
    sizes = [64, tile - 64, tile, tile + 64, 5 * 64, 16 * tile, 16 * tile + 64, 33 * tile, 1]
    batch = gsim.Batch(1400000, 32)
    batch.set_tuning(sort_tile=tile)
    alone, ids = [], []

    def add(n, seed, preset="exponential-disk"):
        p = gsim.generate(preset, n, 120.0, 1.0, 10.0, seed=seed)
        p.pos[: n // 50] = [700, 0]
        alone.append(gsim.Simulation(p, "barnes-hut", accuracy_parameter=1.0))
        ids.append(batch.add(p, "barnes-hut", accuracy_parameter=1.0))

    for k, n in enumerate(sizes):
        print(f"batch tile={tile} n={n}", flush=True)
        add(n, k)
    for extra in ([], [300000, 300000, 200000]):
        for k, n in enumerate(extra):
            add(n, 100 + k, "galaxy")
        batch.step(3)
        for a, k in zip(alone, ids):
            a.step(3)
            x, y = a.read(), batch.read(k)
            assert np.array_equal(x.pos, y.pos) and np.array_equal(x.vel, y.vel)
            assert np.array_equal(x.mass, y.mass)
    for a in alone:
        a.close()
    batch.close()


@pytest.mark.parametrize("bits,boxed", [(10, False), (15, True)])
@pytest.mark.parametrize("n", [131072, 131073, 262144, 262145])
def test_tree_on_both_sides_of_a_change_of_radix_tile(n, bits, boxed):
    print(f"radix tile n={n} bits={bits}", flush=True)
    p = gsim.generate("galaxy-collision", n, 130.0, 1.0, 10.0, seed=n)
    _same_tree(p.pos, p.mass, bits, 2, boxed)


@pytest.mark.parametrize("bh", [0, 64, 16000])
def test_batch_direct_sums_beside_and_without_a_build(bh):
    """The direct-sum launch with all its workgroups taking blocks (no or few
    Barnes-Hut particles) and with one a CU; a system whose budget is spent
    holds its state.  Same bits as alone."""
    print(f"batch direct sums bh={bh}", flush=True)
    batch = gsim.Batch(400000, 32)
    alone, ids = [], []
    for k, n in enumerate([64, 1000, 16 * 257, 6128] + ([bh] if bh else [])):
        p = gsim.generate("random", n, 60.0, 1.0, 10.0, seed=k)
        algo = "barnes-hut" if bh and k == 4 else "direct-sum"
        alone.append(gsim.Simulation(p, algo))
        ids.append(batch.add(p, algo))
    batch.set_steps(ids[0], 2)
    batch.step(3)
    for k, (a, i) in enumerate(zip(alone, ids)):
        a.step(2 if k == 0 else 3)
        x, y = a.read(), batch.read(i)
        assert np.array_equal(x.pos, y.pos) and np.array_equal(x.vel, y.vel)
        a.close()
    batch.close()
