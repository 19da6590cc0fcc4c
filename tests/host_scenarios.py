"""What libgsim's host code does when something fails: each scenario runs in a
process of its own against the HIP runtime of native/fake_hip.cpp, where device
memory is host memory and kernels only leave their names.

    python host_scenarios.py <fake_hip.so> <scenario>
"""
import ctypes as C
import os
import sys
import time

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for sub in ("gravity-sim_amd/python", "tests", "oracle"):
    sys.path.insert(0, os.path.join(ROOT, sub))

fake = None  # the runtime
gsim = None
helpers = None

OUT_OF_MEMORY, DEVICE = 2, 3


def _load(path):
    global fake, gsim, helpers
    fake = C.CDLL(path, mode=C.RTLD_GLOBAL)  # ahead of libgsim.so
    fake.fake_limit.argtypes = [C.c_size_t]
    fake.fake_live.restype = C.c_size_t
    fake.fake_launches.restype = fake.fake_faults.restype = C.c_char_p
    import gsim as g
    import helpers as h
    gsim, helpers = g, h


def _launched(call):
    """The kernels that `call` launches."""
    fake.fake_forget()
    call()
    return fake.fake_launches().decode()


def _refused(status, call):
    try:
        call()
    except gsim.GsimError as e:
        assert e.status == status, e
        return
    raise AssertionError("not refused")


def failed_form_keeps_the_last():
    """A direct-sum form whose partial sums do not fit is refused, and the
    handle goes on in the form it had."""
    for n, kernel, asks in (
            # slices, too large for the default symmetric form
            (600_000, "ds_partial_kernel", lambda s: s.set_tuning(gsim.TUNE_DS_SYMMETRIC, 1)),
            # symmetric; many slices need more
            (20_000, "ds_sym_kernel", lambda s: s.set_ds_shape(4, 256)),
            # blocks, which have no partial sums at all
            (10_000, "ds_block_kernel", lambda s: s.set_ds_shape(1, 100)),
            (10_000, "ds_block_kernel", lambda s: s.set_tuning(gsim.TUNE_DS_SYMMETRIC, 1))):
        with gsim.Simulation(gsim.generate("random", n, 100.0, 1.0, 10.0), "direct-sum") as s:
            before = _launched(lambda: s.step(1))
            assert kernel in before, (n, before)
            fake.fake_limit(fake.fake_live())
            _refused(OUT_OF_MEMORY, lambda: asks(s))
            assert _launched(lambda: s.step(1)) == before
            fake.fake_limit(2 ** 64 - 1)
            assert _launched(lambda: s.step(1)) == before
            asks(s)  # and with memory it is granted
            assert _launched(lambda: s.step(1)) != before
    with gsim.Simulation(gsim.generate("random", 20_000, 100.0, 1.0, 10.0), "direct-sum") as s:
        s.set_ds_shape(4, 200)  # 32 MB of partial sums
        fake.fake_limit(fake.fake_live() + (20 << 20))  # 41 fit, but not beside the 32
        s.set_ds_shape(4, 256)
        fake.fake_limit(2 ** 64 - 1)
        assert "ds_partial_kernel" in _launched(lambda: s.step(1))
    with gsim.Simulation(gsim.generate("random", 20_000, 100.0, 1.0, 10.0), "direct-sum") as s:
        s.set_ds_shape(4, 100)
        fake.fake_limit(0)  # neither the new sums nor the old ones again
        _refused(OUT_OF_MEMORY, lambda: s.set_ds_shape(4, 256))
        _refused(OUT_OF_MEMORY, lambda: s.step(1))
        fake.fake_limit(2 ** 64 - 1)
        s.set_ds_shape(4, 100)
        s.step(1)


def lost_tree_buffers():
    """A leaf depth that does not fit leaves the last one; without memory for
    either the state can still be read, and no step is taken."""
    p = gsim.generate("galaxy", 20_000, 100.0, 1.0, 10.0)  # more than a read stages
    with gsim.Simulation(p, "barnes-hut") as s:
        fake.fake_limit(fake.fake_live())
        _refused(OUT_OF_MEMORY, lambda: s.set_tuning(gsim.TUNE_BH_LEAF_BITS, 15))
        fake.fake_limit(2 ** 64 - 1)
        assert "bh_leaf_kernel" in _launched(lambda: s.step(1))
    with gsim.Simulation(p, "barnes-hut") as s:
        fake.fake_limit(0)
        _refused(OUT_OF_MEMORY, lambda: s.set_tuning(gsim.TUNE_BH_LEAF_BITS, 15))
        q = s.read()
        assert (q.pos == p.pos).all() and (q.vel == p.vel).all() and (q.mass == p.mass).all()
        _refused(OUT_OF_MEMORY, lambda: s.step(1))
        _refused(OUT_OF_MEMORY, lambda: s.dump(gsim.DUMP_CELLS))
        fake.fake_limit(2 ** 64 - 1)
        s.set_tuning(gsim.TUNE_BH_LEAF_BITS, 10)
        assert "bh_walk_kernel" in _launched(lambda: s.step(1))


def given_up_sort_is_never_read():
    """Once a look-back of the sort has given up, every read of the handle
    fails: small and large ones, the first and the later, and after the leaf
    depth's buffers were exchanged.  In a batch it is the systems that had
    stepped."""
    for n in (12_000, 20_000):  # through the pinned block from the second read on, and never
        with gsim.Simulation(gsim.generate("galaxy", n, 100.0, 1.0, 10.0), "barnes-hut") as s:
            s.step(1)
            s.read()
            helpers.put_sort_stall(s, 3)
            for _ in range(3):
                _refused(DEVICE, s.read)
            _refused(DEVICE, lambda: s.dump(gsim.DUMP_CELLS))
            _refused(DEVICE, lambda: s.dump(gsim.DUMP_ACCEL))
            s.set_tuning(gsim.TUNE_BH_LEAF_BITS, 15)
            _refused(DEVICE, s.read)
    with gsim.Batch(100_000, 8) as b:
        old = [b.add(gsim.generate("galaxy", n, 100.0, 1.0, 10.0), "barnes-hut")
               for n in (12_000, 20_000)]
        b.step(2)
        for i in old:
            b.read(i)
        helpers.put_sort_stall(b, 1)
        new = b.add(gsim.generate("galaxy", 9_000, 100.0, 1.0, 10.0), "barnes-hut")
        for i in old + old:
            _refused(DEVICE, lambda: b.read(i))
        b.read(new)
        b.step(1)  # the upload of the new member forgets the count, not what it spoilt
        for i in old:
            _refused(DEVICE, lambda: b.read(i))
        b.read(new)


def new_buffers_are_cleared_before_use():
    """No step starts beside the clearing of the buffers it uses, or beside a
    copy that keeps the state."""
    p = gsim.generate("galaxy", 9_000, 100.0, 1.0, 10.0)
    for algorithm in ("direct-sum", "barnes-hut"):
        with gsim.Simulation(p, algorithm) as s:
            s.step(1)
            if algorithm == "barnes-hut":
                s.set_tuning(gsim.TUNE_BH_LEAF_BITS, 15)
                s.step(1)
    with gsim.Batch(100_000, 8) as b:
        for algorithm in ("direct-sum", "barnes-hut"):
            b.add(p, algorithm)
        b.step(1)
        b.autotune(1)
        b.step(1)


def query_beside_a_capture():
    """A query from a client's thread leaves the worker's capture alone, and
    returns what had been counted."""
    fake.fake_capture_delay(2_000)  # microseconds a captured launch: 30 ms a graph
    budget = 200_000 * gsim.Batch.bytes_per_particle()
    ps = [gsim.generate("galaxy", n, 100.0, 1.0, 10.0) for n in (9_000, 700, 12_000, 300)]
    with gsim.Server(budget, max_systems=64) as srv:
        rids = []
        for p, algorithm in zip(ps, ("barnes-hut", "direct-sum", "barnes-hut", "direct-sum")):
            rids.append(srv.submit(p, 20, algorithm))
            until = time.monotonic() + 0.2
            while time.monotonic() < until:
                srv.stats()
        assert srv.drain(60.0)
        stats = srv.stats()
        assert (stats["completed"], stats["failed"]) == (4, 0), stats
        for r in rids:
            assert srv.wait(r, 1.0)


def walk_form_by_the_members():
    """The batch's walk takes the wide form by what its members can use, not by
    the size of the arena."""
    narrow, wide = "bb_force_kernelILb0E", "bb_force_kernelILb1E"
    with gsim.Batch(100_000_000, 8) as b:  # 300,000,064 node slots
        b.add(gsim.generate("galaxy", 9_000, 100.0, 1.0, 10.0), "barnes-hut")
        names = _launched(lambda: b.step(2))
        assert narrow in names and wide not in names, names
        helpers.put_narrow_nodes(b, b.info()["nodes_reserved"])
        names = _launched(lambda: b.step(2))
        assert wide in names and narrow not in names, names
        helpers.put_narrow_nodes(b, b.info()["nodes_reserved"] + 1)
        assert narrow in _launched(lambda: b.step(1))


def partial_sums_without_room_and_given_back():
    """A large direct sum is one-sided where the symmetric form's partial sums
    do not fit, and gives them back when it is made one-sided."""
    p = gsim.generate("random", 400_000, 100.0, 1.0, 10.0)
    at = fake.fake_live()
    with gsim.Simulation(p, "direct-sum") as s:
        assert "ds_sym_kernel" in _launched(lambda: s.step(1))
        with_sums = fake.fake_live() - at
        s.set_tuning(gsim.TUNE_DS_SYMMETRIC, 0)
        without = fake.fake_live() - at
        assert without < with_sums / 10, (with_sums, without)
        s.step(1)
    assert fake.fake_live() == at
    fake.fake_limit(at + with_sums // 2)
    with gsim.Simulation(p, "direct-sum") as s:
        names = _launched(lambda: s.step(1))
        assert "ds_partial_kernel" in names and "ds_sym_kernel" not in names
        _refused(OUT_OF_MEMORY, lambda: s.set_tuning(gsim.TUNE_DS_SYMMETRIC, 1))
        assert _launched(lambda: s.step(1)) == names


def knob_without_effect_keeps_the_graphs():
    """run_queue shapes no launch any more: setting it captures nothing again."""
    with gsim.Batch(20_000, 8) as b:
        b.add(gsim.generate("galaxy", 9_000, 100.0, 1.0, 10.0), "barnes-hut")
        b.step(2)
        graphs = fake.fake_instantiated()
        b.set_tuning(run_queue=16)
        b.step(2)
        assert b.tuning()["run_queue"] == 16 and fake.fake_instantiated() == graphs
        b.set_tuning(run_queue=32, waves_per_simd=4)
        b.step(2)
        assert b.tuning()["run_queue"] == 32 and fake.fake_instantiated() == graphs + 2


def columns_asked_for_are_taken():
    """Two column blocks a wave need eight row blocks, also where the size alone
    would take four."""
    for n, rows in ((20_000, (4, 4, 8)), (40_000, (8, 8, 8)), (70_000, (16, 16, 16))):
        with gsim.Simulation(gsim.generate("random", n, 100.0, 1.0, 10.0), "direct-sum") as s:
            for cols, r in zip((0, 1, 2), rows):
                s.set_tuning(gsim.TUNE_DS_SYM_COLS, cols)
                assert f"ds_sym_kernelILi{r}E" in _launched(lambda: s.step(1)), (n, cols)


def failed_requests_leave_their_space():
    """Requests that fail with a step, or with the read of their result, say why
    and make room for the next ones."""
    p = gsim.generate("galaxy", 15_000, 100.0, 1.0, 10.0)
    with gsim.Server(20_000 * gsim.Batch.bytes_per_particle(), max_systems=4) as srv:
        fake.fake_refuse_graphs(1)
        for _ in range(2):
            rid = srv.submit(p, 3, "barnes-hut")
            try:
                assert srv.wait(rid, 20.0)
                state = "done"
            except gsim.GsimError as e:
                assert "hipGraphInstantiate" in str(e), e
                state = "failed"
        assert state == "done"
        stats = srv.stats()
        assert (stats["completed"], stats["failed"]) == (1, 1), stats


if __name__ == "__main__":
    _load(sys.argv[1])
    globals()[sys.argv[2]]()
    assert not fake.fake_faults(), fake.fake_faults().decode()
    print("ok")
