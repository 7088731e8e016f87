"""Descriptors on both sides of a ticket: a busy engine's tickets share destination lines across their ends, and a ticket's own
descriptors and its two neighbours come by one load as far as a wavefront's lanes go.  Tickets of a fixed size around the number
of lanes and around whole lines of descriptors, the last of a submission full, of one descriptor or one short."""
import ctypes

import numpy as np
import pytest

from conftest import GpuBuffers, first_difference, oracle_expected
from test_engine_gpu import Engine, Mapped

pytestmark = pytest.mark.gpu

PAGES = 512
COUNT = 10  # submissions of a call: from eight on tickets look at their neighbours


@pytest.mark.parametrize("per", [1, 2, 8, 31, 32, 61, 62, 63, 64])
@pytest.mark.parametrize("beyond", [-1, 0, 1])
def test_neighbours_of_a_ticket(pkg, hip, oracle, per, beyond):
    n = 3 * per + beyond
    rng = np.random.default_rng(100 * per + beyond + 1)
    lens = rng.integers(130, 700, COUNT * n)
    lens[rng.random(COUNT * n) < 0.05] = 0
    lens[0] = 517
    descs = np.zeros(COUNT * n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"] = lens
    descs["src_off"] = rng.integers(0, (PAGES - 1) * 4096, COUNT * n)
    descs["dst_off"] = np.cumsum(lens) - lens
    total = int(lens.sum())
    pool = rng.integers(0, 256, PAGES * 4096, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, total, 3)
    buffers = [GpuBuffers(pool, descs, total, 3) for _ in range(2)]  # one a turn: what either fails to write shows
    m = Mapped(pkg, hip, descs, COUNT)
    e = Engine(pkg, hip, workgroups=33, descs_per_ticket=per)
    subs = (pkg.Submission * COUNT)()
    print("%d submissions of %d descriptors in tickets of %d" % (COUNT, n, per), flush=True)
    accepted = ctypes.c_uint32()
    try:
        e.start()
        for turn, g in enumerate(buffers, 1):
            for i in range(COUNT):
                subs[i] = pkg.Submission(g.pool.data_ptr(), g.dst_base, m.desc_dev(i * n), m.flag_dev(i), turn, n, 400 * n)
            assert hip.tcpxuEngineSubmitMany(e.h, subs, COUNT, ctypes.byref(accepted)) == pkg.SUCCESS, hip.tcpxuLastError()
            assert accepted.value == COUNT
            for i in range(COUNT):
                m.wait(i, turn)
    finally:
        e.destroy()  # (stops it: nothing may be left running on buffers that go back to the allocator)
    m.free()
    for turn, g in enumerate(buffers, 1):
        difference = first_difference(g.result(), expect)
        assert difference is None, "turn %d, first (index, got, want, count): %r" % (turn, difference)
