"""Descriptors that travel with a submission: lists around the sixteen that do, in memory where the host sees them and where
it does not, with destination offsets that fit and that do not, handed over one at a time and several to a call, on the
smallest ring (every place used many times over) and on one where nothing comes round."""
import ctypes
import time

import numpy as np
import pytest

from conftest import GpuBuffers, first_difference, oracle_expected
from test_engine_gpu import Engine, Mapped

pytestmark = pytest.mark.gpu

PAGES = 1024
COUNTS = [1, 2, 15, 16, 17, 0, 3, 16, 40, 5, 8, 16, 1]


@pytest.mark.parametrize("per_call", [1, 3, 9, 40])
@pytest.mark.parametrize("kind", ["mapped", "device", "offsets beyond 4 GiB"])
@pytest.mark.parametrize("ring", [16, 0])
def test_small_lists(pkg, hip, oracle, ring, kind, per_call):
    small_lists(pkg, hip, oracle, kind, per_call, ring_entries=ring)


@pytest.mark.parametrize("workers", [1, 3])
def test_lists_of_tickets_that_are_there_at_the_first_look(pkg, hip, oracle, workers):
    """More tickets than workers, in bursts with a wait after each: a fetcher's first looks, which do not ask for the list
    that travels, find most of them, and its later looks, which do, the first of a burst."""
    small_lists(pkg, hip, oracle, "mapped", 40, workgroups=workers + 1)


def small_lists(pkg, hip, oracle, kind, per_call, **config):
    rng = np.random.default_rng(per_call)
    counts = np.array([COUNTS[i % len(COUNTS)] for i in range(160)])
    first = np.cumsum(counts) - counts
    n = int(counts.sum())
    lens = np.where(rng.random(n) < 0.5, 4096, rng.integers(0, 4097, n))
    descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"] = lens
    descs["src_off"] = rng.integers(0, (PAGES - 1) * 4096, n)
    descs["dst_off"] = np.cumsum(lens) - lens
    total = int(lens.sum())
    pool = rng.integers(0, 256, PAGES * 4096, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, total, 0)
    far = 2**32 if kind.startswith("offsets") else 0
    descs["dst_off"] += far
    g = GpuBuffers(pool, descs, total)
    m = Mapped(pkg, hip, descs, len(counts))
    e = Engine(pkg, hip, **config)
    subs = (pkg.Submission * len(counts))()
    for i in range(len(counts)):
        at = g.descs.data_ptr() + 16 * int(first[i]) if kind == "device" else m.desc_dev(int(first[i]))
        subs[i] = pkg.Submission(g.pool.data_ptr(), g.dst_base - far, at, m.flag_dev(i), i + 1, int(counts[i]), 0)
    print("small lists: %r, %s, %d a call" % (config, kind, per_call), flush=True)
    e.start()
    accepted = ctypes.c_uint32()
    at, deadline = 0, time.time() + 20
    while at < len(counts):
        take = min(per_call, len(counts) - at)
        rc = hip.tcpxuEngineSubmitMany(e.h, ctypes.byref(subs[at]), take, ctypes.byref(accepted))
        assert rc in (pkg.SUCCESS, pkg.IN_PROGRESS), hip.tcpxuLastError()
        at += accepted.value
        if at % 4 == 0 and at:  # now and then the engine runs empty
            m.wait(at - 1, at)
        assert time.time() < deadline, "the submission ring stayed full"
    for i in range(len(counts)):
        m.wait(i, i + 1)
    e.stop()
    got = g.result()
    e.destroy()
    m.free()
    assert first_difference(got, expect) is None, repr(first_difference(got, expect))
