"""Entries that become one ticket each where they are looked at, beside entries that do not: sizes around the 16 descriptors
that are one ticket always and the 32 that are while eight submissions are in flight, empty ones and ones of several tickets
among them, one at a time and several to a call, with tickets sized by backlog and of a fixed size.  And long runs of entries
of several tickets, broken at the ends of sixteen and elsewhere by one that is not like them; where they are queued before the
start they are certainly taken 64 at a time, and on rings of 64 and 128 with few workers their job slots come round busy."""
import ctypes
import time

import numpy as np
import pytest

import test_engine_carried_gpu as carried
from conftest import GpuBuffers, first_difference, make_descs, oracle_expected
from test_engine_gpu import Engine, Mapped

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_ticket", [0, 4, 64])
@pytest.mark.parametrize("per_call", [1, 2, 5, 17])
@pytest.mark.parametrize("other", [0, 17, 32, 33, 100])
def test_small_entries_among_others(pkg, hip, oracle, monkeypatch, other, per_call, per_ticket):
    monkeypatch.setattr(carried, "COUNTS", [16, other, 1, 16, 16, 2, other, other, 5, 16, 16, 16, 16, 16, 16, other])
    carried.small_lists(pkg, hip, oracle, "mapped", per_call, descs_per_ticket=per_ticket)


@pytest.mark.parametrize("per_ticket", [0, 3])
@pytest.mark.parametrize("usual", [33, 70, 96, 130])  # (96 in tickets of 3 are the most that an entry's lanes write; 130 go one by one)
@pytest.mark.parametrize("other", [0, 1, 64, 600])
def test_long_runs_of_entries_of_several_tickets(pkg, hip, oracle, monkeypatch, other, usual, per_ticket):
    counts = [usual] * 160
    for at in (5, 31, 32, 63, 90, 111, 159):
        counts[at] = other
    monkeypatch.setattr(carried, "COUNTS", counts)
    for per_call in (160, 48):
        carried.small_lists(pkg, hip, oracle, "mapped", per_call, descs_per_ticket=per_ticket)


@pytest.mark.parametrize("counts", [[5], [100], [100, 100, 100], [100, 0, 100], [1, 1, 100, 100, 100], [1, 100, 1, 100, 100, 1]])
def test_a_poll_of_the_ring_counts_once_whatever_it_shows(pkg, hip, oracle, counts):
    """Everything is queued before the start, so that the first poll shows all of it; then come as many polls that show nothing
    as it takes the kernel to leave, 7/3 of the limit."""
    first = np.cumsum(counts) - counts
    n = sum(counts)
    pool = np.random.default_rng(n).integers(0, 256, 1 << 20, dtype=np.uint8)
    descs = make_descs([((4099 * i) % ((1 << 20) - 1000), 999, 1000 * i) for i in range(n)])
    expect = oracle_expected(oracle, pool, descs, 1000 * n)
    g = GpuBuffers(pool, descs, 1000 * n)
    m = Mapped(pkg, hip, descs, len(counts))
    e = Engine(pkg, hip, spin_limit=3)
    for i in range(len(counts)):
        e.submit(g.pool.data_ptr(), g.dst_base, m.desc_dev(int(first[i])), counts[i], m.flag_dev(i), i + 1)
    e.start()
    for i in range(len(counts)):
        m.wait(i, i + 1)
    deadline = time.time() + 20
    while e.running():  # (a stop would end the polls sooner)
        assert time.time() < deadline
    e.stop()
    stats = pkg.EngineStats()
    pkg.check(hip.tcpxuEngineGetStats(e.h, ctypes.byref(stats)), "tcpxuEngineGetStats")
    got = g.result()
    e.destroy()
    m.free()
    assert first_difference(got, expect) is None, repr(first_difference(got, expect))
    assert stats.launches == 1 and stats.leader_entries == len(counts) and stats.leader_deep_polls == 0
    assert stats.leader_polls == 1 + 7 * 3 // 3


@pytest.mark.parametrize("workers", [2, 40])
@pytest.mark.parametrize("ring", [64, 128])
@pytest.mark.parametrize("usual,per_ticket", [(33, 0), (96, 0), (33, 3), (96, 3)])
@pytest.mark.parametrize("other", [0, 1, 96])
def test_runs_of_several_tickets_on_rings_that_come_round_busy(pkg, hip, oracle, other, usual, per_ticket, ring, workers):
    counts = np.full(600, usual)
    counts[[31, 32, 63, 64, 90, 111, 128, 143, 144, 300, 599]] = other  # (the first sixteen are alike: 64 are asked for next)
    first = np.cumsum(counts) - counts
    n = int(counts.sum())
    rng = np.random.default_rng(ring + workers)
    pool = rng.integers(0, 256, 1 << 20, dtype=np.uint8)
    descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"] = rng.integers(0, 700, n)
    descs["src_off"] = rng.integers(0, len(pool) - 700, n)
    descs["dst_off"] = np.cumsum(descs["len"], dtype=np.uint64) - descs["len"]
    total = int(descs["len"].sum())
    expect = oracle_expected(oracle, pool, descs, total)
    g = GpuBuffers(pool, descs, total)
    m = Mapped(pkg, hip, descs, len(counts))
    subs = (pkg.Submission * len(counts))()
    for i in range(len(counts)):
        subs[i] = pkg.Submission(g.pool.data_ptr(), g.dst_base, m.desc_dev(int(first[i])), m.flag_dev(i), i + 1, int(counts[i]), 0)
    e = Engine(pkg, hip, ring_entries=ring, descs_per_ticket=per_ticket, workgroups=workers + 1)
    print("busy job slots: %d of %d, some %d, tickets of %d, ring %d, %d workers" % (len(counts), usual, other, per_ticket, ring, workers), flush=True)
    accepted = ctypes.c_uint32()
    assert hip.tcpxuEngineSubmitMany(e.h, subs, len(counts), ctypes.byref(accepted)) == pkg.IN_PROGRESS and accepted.value == ring
    e.start()
    at, deadline = ring, time.time() + 20
    while at < len(counts):
        rc = hip.tcpxuEngineSubmitMany(e.h, ctypes.byref(subs[at]), len(counts) - at, ctypes.byref(accepted))
        assert rc in (pkg.SUCCESS, pkg.IN_PROGRESS), hip.tcpxuLastError()
        at += accepted.value
        assert time.time() < deadline, "the submission ring stayed full"
    for i in range(len(counts)):
        m.wait(i, i + 1)
    e.stop()
    stats = pkg.EngineStats()
    pkg.check(hip.tcpxuEngineGetStats(e.h, ctypes.byref(stats)), "tcpxuEngineGetStats")
    print("busy job slots: %d polls, %d of 64" % (stats.leader_polls, stats.leader_deep_polls), flush=True)
    got = g.result()
    e.destroy()
    m.free()
    assert first_difference(got, expect) is None, repr(first_difference(got, expect))
    assert stats.leader_entries == len(counts) and stats.leader_deep_polls > 0
