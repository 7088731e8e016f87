"""The kernels that are launched per list, at the list lengths where their grids and counters change: whole and partial
workgroups of four descriptors, grids rounded up to eight workgroups, one counter up to 64 workgroups of a slot and eight
beyond (tcpxuUnpackBatch, tcpxuUnpackSlotNoAlloc; byte-exact against the CPU oracle)."""
import numpy as np
import pytest

from conftest import GUARD, SENTINEL, GpuBuffers, first_difference, oracle_expected
from test_engine_gpu import Mapped

pytestmark = pytest.mark.gpu

PAGES = 4096


def ragged_list(n, seed):
    """n descriptors back to back in the destination: whole pages, short, tiny and empty ones, one of several rounds."""
    rng = np.random.default_rng(seed)
    lens = np.where(rng.random(n) < 0.5, 4096, rng.integers(0, 4097, n))
    lens[rng.random(n) < 0.1] = rng.integers(0, 32)
    if n > 6:
        lens[n // 2] = 3 * 4096 + 77  # longer than a page: four rounds
    descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"] = lens
    descs["src_off"] = rng.integers(0, PAGES * 4096 - 4 * 4096, n)
    descs["dst_off"] = np.cumsum(lens) - lens
    return descs, int(lens.sum())


@pytest.mark.parametrize("n", [1, 3, 4, 5, 32, 33, 255, 256, 257, 1023, 2047, 2048])
@pytest.mark.parametrize("misalign", [0, 5])
def test_list_lengths(pkg, hip, oracle, n, misalign):
    import torch

    descs, total = ragged_list(n, n)
    pool = np.random.default_rng(n + 1).integers(0, 256, PAGES * 4096, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, total, misalign)
    buf = GpuBuffers(pool, descs, total, misalign)
    mapped = Mapped(pkg, hip, descs, 3)
    print("list of %d descriptors, %d bytes, misaligned by %d" % (n, total, misalign), flush=True)
    pkg.check(hip.tcpxuUnpackBatch(0, buf.pool.data_ptr(), buf.dst_base, buf.descs.data_ptr(), n, None), "tcpxuUnpackBatch")
    torch.cuda.synchronize()
    assert first_difference(buf.result(), expect) is None
    for call in range(3):  # each finds the counters as the one before left them
        buf.reset()
        pkg.check(hip.tcpxuUnpackSlotNoAlloc(0, buf.pool.data_ptr(), buf.dst_base, mapped.desc_dev(0), n, mapped.flag_dev(call), 70 + call, None), "tcpxuUnpackSlotNoAlloc")
        torch.cuda.synchronize()
        assert int(mapped.flags[call]) == 70 + call
        assert first_difference(buf.result(), expect) is None
    mapped.free()


def test_calls_on_two_streams_at_once(pkg, hip, oracle):
    """Every call has counters of its own: slots on two streams complete in whatever order they run."""
    import torch

    descs, total = ragged_list(700, 9)
    pool = np.random.default_rng(10).integers(0, 256, PAGES * 4096, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, total)
    buf = GpuBuffers(pool, descs, total)
    second = torch.full_like(buf.dst, SENTINEL)
    bases = [buf.dst_base, second.data_ptr() + GUARD]
    streams = [torch.cuda.Stream() for _ in range(2)]
    mapped = Mapped(pkg, hip, descs, 2)
    torch.cuda.synchronize()
    for call in range(100):
        for k in range(2):
            pkg.check(
                hip.tcpxuUnpackSlotNoAlloc(0, buf.pool.data_ptr(), bases[k], mapped.desc_dev(0), len(descs), mapped.flag_dev(k), 1 + call, streams[k].cuda_stream),
                "tcpxuUnpackSlotNoAlloc",
            )
        if call % 20 == 19:
            torch.cuda.synchronize()
            assert [int(mapped.flags[k]) for k in range(2)] == [1 + call] * 2
    assert first_difference(buf.result(), expect) is None
    assert first_difference(second.cpu().numpy(), expect) is None
    mapped.free()


def test_every_set_of_counters_is_used_again(pkg, hip, oracle):
    """2100 calls in a row, every one with a completion word of its own: the 1024 sets come round twice, each after lists of
    another length on either side of the line between one counter and nine."""
    import torch

    descs, total = ragged_list(300, 4)
    pool = np.random.default_rng(5).integers(0, 256, PAGES * 4096, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, total)
    buf = GpuBuffers(pool, descs, total)
    calls = 2100
    mapped = Mapped(pkg, hip, descs, calls)
    for call in range(calls):
        n = (300, 3, 257)[call % 3] if call != calls - 1 else 300
        pkg.check(hip.tcpxuUnpackSlotNoAlloc(0, buf.pool.data_ptr(), buf.dst_base, mapped.desc_dev(0), n, mapped.flag_dev(call), 1 + call, None), "tcpxuUnpackSlotNoAlloc")
    torch.cuda.synchronize()
    assert (np.asarray(mapped.flags[:calls]) == np.arange(1, calls + 1)).all()
    assert first_difference(buf.result(), expect) is None
    mapped.free()
