"""Submissions whose tickets need most of the ticket ring, one behind the other: each waits until the ring has room for all of
its tickets, and the leader has to find out that it has.  And more submissions of one ticket than the ring holds, handed over
much faster than they are served: the rolling loop fills the ring, and what comes after it must not write beyond that."""
import ctypes
import time

import numpy as np
import pytest

from conftest import GpuBuffers, first_difference, oracle_expected
from test_engine_gpu import Engine, Mapped

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_ticket,counts", [(16, [600000, 600000]), (16, [16, 1 << 20]), (1, [1, 65536, 3, 40000, 40000, 65536]), (31, [1 << 20, 1000000, 5])])
def test_submissions_that_need_most_of_the_ticket_ring(pkg, hip, oracle, per_ticket, counts):
    rng = np.random.default_rng(per_ticket)
    n = sum(counts)
    first = np.cumsum(counts) - counts
    pool = rng.integers(0, 256, 1 << 20, dtype=np.uint8)
    descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"] = rng.integers(0, 65, n)
    descs["src_off"] = rng.integers(0, len(pool) - 64, n)
    descs["dst_off"] = np.cumsum(descs["len"], dtype=np.uint64) - descs["len"]
    total = int(descs["len"].sum())
    expect = oracle_expected(oracle, pool, descs, total)
    g = GpuBuffers(pool, descs, total)
    m = Mapped(pkg, hip, descs[:0], len(counts))
    subs = (pkg.Submission * len(counts))()
    for i in range(len(counts)):
        subs[i] = pkg.Submission(g.pool.data_ptr(), g.dst_base, g.descs.data_ptr() + 16 * int(first[i]), m.flag_dev(i), i + 1, counts[i], 0)
    e = Engine(pkg, hip, descs_per_ticket=per_ticket)
    print("ticket room: %r in tickets of %d" % (counts, per_ticket), flush=True)
    e.start()
    accepted = ctypes.c_uint32()
    pkg.check(hip.tcpxuEngineSubmitMany(e.h, subs, len(counts), ctypes.byref(accepted)), "tcpxuEngineSubmitMany")
    for i in range(len(counts)):
        m.wait(i, i + 1)
    e.stop()
    got = g.result()
    e.destroy()
    m.free()
    assert first_difference(got, expect) is None, repr(first_difference(got, expect))


@pytest.mark.parametrize("workers", [1, 5])
@pytest.mark.parametrize("ring", [0, 65536])
@pytest.mark.parametrize("others", [1, 100])
def test_more_submissions_of_one_ticket_than_the_ring_holds(pkg, hip, oracle, others, ring, workers):
    """Every thousandth submission, and thirty in a row now and then, of `others` descriptors: those of several tickets end the
    rolling loop and go the ordinary way, with the ring full or nearly so."""
    rng = np.random.default_rng(workers)
    count = 250000
    counts = np.ones(count, dtype=np.int64)
    counts[::1000] = others
    for at in range(70000, count, 20000):
        counts[at : at + 30] = others
    first = np.cumsum(counts) - counts
    n = int(counts.sum())
    pool = rng.integers(0, 256, 1 << 20, dtype=np.uint8)
    descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"] = rng.integers(0, 65, n)
    descs["src_off"] = rng.integers(0, len(pool) - 64, n)
    descs["dst_off"] = np.cumsum(descs["len"], dtype=np.uint64) - descs["len"]
    total = int(descs["len"].sum())
    expect = oracle_expected(oracle, pool, descs, total)
    g = GpuBuffers(pool, descs, total)
    m = Mapped(pkg, hip, descs[:0], count)
    flags = np.ctypeslib.as_array(m.flags)
    subs = np.zeros(count, dtype=[("bounce", "<u8"), ("dst", "<u8"), ("descs", "<u8"), ("flag", "<u8"), ("value", "<u8"), ("n", "<u4"), ("bytes", "<u4")])
    assert subs.itemsize == ctypes.sizeof(pkg.Submission)
    subs["bounce"], subs["dst"] = g.pool.data_ptr(), g.dst_base
    subs["descs"] = g.descs.data_ptr() + 16 * first.astype(np.uint64)
    subs["flag"] = m.flag_dev(0) + 8 * np.arange(count, dtype=np.uint64)
    subs["value"] = np.arange(1, count + 1)
    subs["n"] = counts
    e = Engine(pkg, hip, ring_entries=ring, workgroups=workers + 1)
    print("ticket room: %d submissions, every thousandth of %d, %d workers, ring %d" % (count, others, workers, ring), flush=True)
    e.start()
    accepted = ctypes.c_uint32()
    at, deadline, most = 0, time.time() + 60, 0
    while at < count:
        rc = hip.tcpxuEngineSubmitMany(e.h, ctypes.cast(subs.ctypes.data + subs.itemsize * at, ctypes.POINTER(pkg.Submission)), min(count - at, 65536), ctypes.byref(accepted))
        assert rc in (pkg.SUCCESS, pkg.IN_PROGRESS), hip.tcpxuLastError()
        at += accepted.value
        if accepted.value:
            most = max(most, at - int(np.count_nonzero(flags[:at])))
        assert time.time() < deadline, "the submission ring stayed full"
    while not np.array_equal(flags, subs["value"]):
        assert time.time() < deadline, "%d submissions were not completed" % np.count_nonzero(flags != subs["value"])
        time.sleep(0.001)
    e.stop()
    stats = pkg.EngineStats()
    pkg.check(hip.tcpxuEngineGetStats(e.h, ctypes.byref(stats)), "tcpxuEngineGetStats")
    print("ticket room: up to %d at a time not completed, %d of %d polls of 64" % (most, stats.leader_deep_polls, stats.leader_polls), flush=True)
    got = g.result()
    e.destroy()
    m.free()
    assert first_difference(got, expect) is None, repr(first_difference(got, expect))
    assert stats.leader_entries == count and stats.leader_deep_polls > 0
    assert most <= 65536 + (ring or 4096), "more tickets out than the ring holds"
    if workers == 1:
        assert most > 65536 + (ring or 4096) // 2, "the ticket ring was never full"  # (the rest wait in the submission ring)
