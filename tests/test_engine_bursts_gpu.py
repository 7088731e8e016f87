"""Bursts: several submissions handed over in one call to an engine of 32 workers, on both sides of the lines where the size
of their tickets changes (three, four and eight submissions, 32 descriptors each, 12 x 32 and 40 x 32 descriptors in all), with
a payload hint that says whole pages, one that says short fragments -- those submissions say how many more of their call
follow -- and none."""
import ctypes

import numpy as np
import pytest

from conftest import GpuBuffers, first_difference, oracle_expected
from test_engine_gpu import Engine, Mapped

pytestmark = pytest.mark.gpu

PAGES = 512
WORKERS = 32


@pytest.mark.parametrize("hint", [4096, 1000, 0])
@pytest.mark.parametrize("subs_n", [(8, 47), (8, 48), (8, 159), (8, 160), (8, 199), (8, 200), (7, 90), (12, 32), (12, 33), (40, 40), (4, 70), (3, 500)])
def test_burst(pkg, hip, oracle, subs_n, hint):
    count, per = subs_n
    rng = np.random.default_rng(count * per)
    n = count * per
    lens = rng.integers(0, 700, n)
    descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"] = lens
    descs["src_off"] = rng.integers(0, (PAGES - 1) * 4096, n)
    descs["dst_off"] = np.cumsum(lens) - lens
    total = int(lens.sum())
    pool = rng.integers(0, 256, PAGES * 4096, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, total, 0)
    g = GpuBuffers(pool, descs, total)
    m = Mapped(pkg, hip, descs, count)
    e = Engine(pkg, hip, workgroups=WORKERS + 1)
    subs = (pkg.Submission * count)()
    print("burst: %d of %d descriptors, hint %d" % (count, per, hint), flush=True)
    e.start()
    accepted = ctypes.c_uint32()
    for turn in (1, 2, 3):  # the first finds the engine idle, the others just emptied
        for i in range(count):
            subs[i] = pkg.Submission(g.pool.data_ptr(), g.dst_base, m.desc_dev(i * per), m.flag_dev(i), turn, per, hint * per)
        assert hip.tcpxuEngineSubmitMany(e.h, subs, count, ctypes.byref(accepted)) == pkg.SUCCESS, hip.tcpxuLastError()
        assert accepted.value == count
        for i in range(count):
            m.wait(i, turn)
    e.stop()
    got = g.result()
    e.destroy()
    m.free()
    assert first_difference(got, expect) is None, repr(first_difference(got, expect))


@pytest.mark.parametrize("subs_n", [(8, 71), (8, 72), (8, 1024), (8, 1025), (8, 1536), (8, 1537), (9, 2048), (8, 3999), (8, 4000)])
def test_burst_of_fragments_of_half_a_page(pkg, hip, oracle, subs_n):
    """The sizes where such submissions change between tickets of 12, 32 and 48, and the leader's way of writing them; 3999
    and 4000: below and at a thousand descriptors per worker."""
    test_burst(pkg, hip, oracle, subs_n, 1800)


@pytest.mark.parametrize("per", [90, 700, 1600])
def test_calls_of_half_page_fragments_behind_one_another(pkg, hip, oracle, per):
    """Calls of eight submissions handed over without a wait: the first finds the engine idle, the others find the ones before
    them queued, and the tickets are of one size or another by that."""
    calls, count = 6, 8
    rng = np.random.default_rng(per)
    n = calls * count * per
    lens = rng.integers(0, 700, n)
    descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"] = lens
    descs["src_off"] = rng.integers(0, (PAGES - 1) * 4096, n)
    descs["dst_off"] = np.cumsum(lens) - lens
    total = int(lens.sum())
    pool = rng.integers(0, 256, PAGES * 4096, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, total, 0)
    g = GpuBuffers(pool, descs, total)
    m = Mapped(pkg, hip, descs, calls * count)
    e = Engine(pkg, hip, workgroups=WORKERS + 1)
    subs = (pkg.Submission * count)()
    print("calls of %d submissions of %d descriptors behind one another" % (count, per), flush=True)
    e.start()
    accepted = ctypes.c_uint32()
    for turn in (1, 2):
        for call in range(calls):
            for k in range(count):
                i = call * count + k
                subs[k] = pkg.Submission(g.pool.data_ptr(), g.dst_base, m.desc_dev(i * per), m.flag_dev(i), turn, per, 1800 * per)
            assert hip.tcpxuEngineSubmitMany(e.h, subs, count, ctypes.byref(accepted)) == pkg.SUCCESS, hip.tcpxuLastError()
            assert accepted.value == count
        for i in range(calls * count):
            m.wait(i, turn)
    e.stop()
    got = g.result()
    e.destroy()
    m.free()
    assert first_difference(got, expect) is None, repr(first_difference(got, expect))
