"""Submissions whose tickets need most of the ticket ring, one behind the other: each waits until the ring has room for all of
its tickets, and the leader has to find out that it has."""
import ctypes

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
