"""Readback in the caller's order, around the size where it changes from the
pinned block to plain copies, and from the first read (always copies) to the
next: before any step it returns the input, later reads return the same bytes
as the first, and a NULL array is skipped."""
import ctypes as C

import numpy as np
import pytest

import gsim

pytestmark = pytest.mark.gpu


def _same(a, b):
    assert np.array_equal(a.pos, b.pos) and np.array_equal(a.vel, b.vel)
    assert np.array_equal(a.mass, b.mass)


@pytest.mark.parametrize("algorithm", ["direct-sum", "barnes-hut"])
@pytest.mark.parametrize("n", [1, 65, 16383, 16384, 16385, 70001])
def test_reads_agree(n, algorithm):
    print(f"read n={n} {algorithm}", flush=True)
    p = gsim.generate("galaxy", n, 50.0, 1.0, 10.0, seed=n)
    with gsim.Simulation(p, algorithm) as s:
        _same(s.read(), p)
        _same(s.read(), p)
        s.step(2)
        a = s.read()
        _same(s.read(), a)
        vel = np.zeros((n, 2), np.float32)
        assert gsim._lib.gsim_read(s._h, None, gsim._fptr(vel), None) == 0
        assert np.array_equal(vel, a.vel)
    with gsim.Simulation(p, algorithm) as s:  # its first read is after the steps
        s.step(2)
        _same(s.read(), a)


def test_batch_reads_agree():
    ps = [gsim.generate("galaxy", n, 50.0, 1.0, 10.0, seed=n) for n in (300, 16384, 16385, 40001)]
    with gsim.Batch(400000, 8) as b:
        ids = [b.add(p, "direct-sum" if p.n < 8192 else "barnes-hut") for p in ps]
        for k, p in zip(ids, ps):
            _same(b.read(k), p)
        b.step(2)
        got = [b.read(k) for k in ids]
        for k, q in zip(ids, got):
            _same(b.read(k), q)
        mass = np.zeros(ps[0].n, np.float32)
        assert gsim._lib.gsim_batch_read(b._h, C.c_uint32(ids[0]), None, None,
                                         gsim._fptr(mass)) == 0
        assert np.array_equal(mass, ps[0].mass)
