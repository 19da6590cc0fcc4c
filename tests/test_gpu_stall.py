"""A radix sort whose look-back gave up (its counter is set from the host; the
sort itself is whole) leaves a state that no read returns, however many steps
follow, and nothing after it runs out of bounds: every later step ends."""
import pytest

import gsim
import helpers as H

pytestmark = pytest.mark.gpu


def _fails(read):
    with pytest.raises(gsim.GsimError) as e:
        read()
    assert e.value.status == 3 and "gave up" in str(e.value)


@pytest.mark.parametrize("n,kw,bits", [(5_000, {}, 10), (12_000, {}, 10),
                                       (40_000, {"group_width": 32}, 10), (20_000, {}, 15)])
def test_a_given_up_sort_stays_noted(n, kw, bits):
    p = gsim.generate("galaxy", n, 100.0, 1.0, 10.0, seed=n)
    with gsim.Simulation(p, "barnes-hut", **kw) as s:
        s.set_tuning(gsim.TUNE_BH_LEAF_BITS, bits)
        s.step(2)
        s.read()
        H.put_sort_stall(s, 1)
        s.step(3)
        _fails(s.read)
        _fails(s.read)


def test_a_given_up_sort_in_a_batch():
    ps = [gsim.generate("galaxy", n, 100.0, 1.0, 10.0, seed=n) for n in (700, 9_000, 30_000)]
    algos = ["direct-sum", "barnes-hut", "barnes-hut"]
    late = gsim.generate("random", 12_000, 100.0, 1.0, 10.0, seed=4)
    with gsim.Batch(80_000, 8) as b:
        ids = [b.add(p, a) for p, a in zip(ps, algos)]
        b.step(2)
        b.read(ids[1])
        H.put_sort_stall(b, 1)
        b.step(3)
        for i in ids:
            _fails(lambda: b.read(i))
        new = b.add(late, "barnes-hut")
        b.step(2)
        for i in ids:
            _fails(lambda: b.read(i))
        got = b.read(new)
    with gsim.Simulation(late, "barnes-hut") as s:
        s.step(2)
        want = s.read()
    assert (got.pos == want.pos).all() and (got.vel == want.vel).all()
