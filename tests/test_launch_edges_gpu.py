"""The kernels that are launched per list, at the list lengths where their grids change: whole and partial workgroups of
four descriptors, grids rounded up to eight workgroups, a slot of one workgroup and of two launches (tcpxuUnpackBatch,
tcpxuUnpackSlotNoAlloc; byte-exact against the CPU oracle)."""
import ctypes

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


@pytest.mark.parametrize("n", [1, 3, 4, 5, 16, 17, 32, 33, 255, 256, 257, 1023, 2047, 2048])
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
    for call in range(3):
        buf.reset()
        pkg.check(hip.tcpxuUnpackSlotNoAlloc(0, buf.pool.data_ptr(), buf.dst_base, mapped.desc_dev(0), n, mapped.flag_dev(call), 70 + call, None), "tcpxuUnpackSlotNoAlloc")
        torch.cuda.synchronize()
        assert int(mapped.flags[call]) == 70 + call
        assert first_difference(buf.result(), expect) is None
    mapped.free()


@pytest.mark.parametrize("n", [15, 18, 23, 24, 25])
@pytest.mark.parametrize("misalign", [0, 5])
def test_list_lengths_around_one_workgroup(pkg, hip, oracle, n, misalign):
    """A slot whose workgroup has a wavefront for every descriptor, two descriptors for some, and two launches."""
    test_list_lengths(pkg, hip, oracle, n, misalign)


@pytest.mark.parametrize("n", [2, 16, 17, 24, 25])
@pytest.mark.parametrize("length", [9000, 70001])
def test_few_descriptors_of_many_rounds_each(pkg, hip, oracle, n, length):
    """Fragments of several pages through one workgroup, a wavefront's second one behind its first, and through two launches."""
    import torch

    rng = np.random.default_rng(n)
    descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"], descs["dst_off"] = length, np.arange(n) * length
    descs["src_off"] = rng.integers(0, PAGES * 4096 - length, n)
    pool = rng.integers(0, 256, PAGES * 4096, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, n * length, 5)
    buf = GpuBuffers(pool, descs, n * length, 5)
    mapped = Mapped(pkg, hip, descs, 1)
    print("slot of %d descriptors of %d bytes" % (n, length), flush=True)
    pkg.check(hip.tcpxuUnpackSlotNoAlloc(0, buf.pool.data_ptr(), buf.dst_base, mapped.desc_dev(0), n, mapped.flag_dev(0), 7, None), "tcpxuUnpackSlotNoAlloc")
    torch.cuda.synchronize()
    assert int(mapped.flags[0]) == 7 and first_difference(buf.result(), expect) is None
    mapped.free()


@pytest.mark.parametrize("n", [2049, 4095, 4096, 4097, 4604, 4607, 4608, 4609, 4613, 6144, 6145, 7001])
def test_lists_around_whole_turns_of_the_xcds(pkg, hip, oracle, n):
    """Beyond 4096 descriptors the XCDs take runs of 24 groups of four descriptors in turn, 768 descriptors a turn: lists of
    whole turns, of one group or descriptor more or less, and of some left over."""
    rng = np.random.default_rng(n)
    lens = rng.choice([0, 20, 100, 300, 1500], size=n)
    descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
    descs["len"], descs["dst_off"] = lens, np.cumsum(lens) - lens
    descs["src_off"] = rng.integers(0, (1 << 20) - 1500, n)
    total = int(lens.sum())
    pool = rng.integers(0, 256, 1 << 20, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, total, 9)
    buf = GpuBuffers(pool, descs, total, 9)
    print("list of %d descriptors" % n, flush=True)
    pkg.check(hip.tcpxuUnpackBatch(0, buf.pool.data_ptr(), buf.dst_base, buf.descs.data_ptr(), n, None), "tcpxuUnpackBatch")
    pkg.check(hip.tcpxuDeviceSynchronize(0), "sync")
    assert first_difference(buf.result(), expect) is None


@pytest.mark.parametrize("n", [7679, 7680, 7681, 8191, 8192, 8193, 8196, 8197, 8447, 8448, 8449, 9217])
def test_lists_around_workgroups_of_one_wavefront_and_of_four(pkg, hip, oracle, n):
    """Up to 8192 descriptors a workgroup is one wavefront, beyond that four; turns of 768 descriptors either way."""
    test_lists_around_whole_turns_of_the_xcds(pkg, hip, oracle, n)


def test_calls_on_two_streams_at_once(pkg, hip, oracle):
    """Calls share nothing: slots on two streams complete in whatever order they run."""
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
    """2100 calls in a row, every one with a completion word of its own, lists on either side of the line between one launch
    and two in turn: no call depends on how many came before."""
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


@pytest.mark.parametrize("n", [16, 700])
def test_replays_of_the_same_call_at_the_same_time(pkg, hip, oracle, n):
    """One call captured into two graphs, arguments and completion word the same, the two replayed on two streams at once
    and an ordinary call after them: every round ends with the bytes and the word."""
    import torch

    descs, total = ragged_list(n, 12)
    pool = np.random.default_rng(13).integers(0, 256, PAGES * 4096, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, total)
    buf = GpuBuffers(pool, descs, total)
    mapped = Mapped(pkg, hip, descs, 2)

    def call(flag, stream):
        rc = hip.tcpxuUnpackSlotNoAlloc(0, buf.pool.data_ptr(), buf.dst_base, mapped.desc_dev(0), n, mapped.flag_dev(flag), 77, ctypes.c_void_p(stream))
        pkg.check(rc, "tcpxuUnpackSlotNoAlloc")

    streams = [torch.cuda.Stream() for _ in range(2)]
    call(0, streams[0].cuda_stream)  # the ordinary call that loads the kernels
    torch.cuda.synchronize()
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    for g, s in zip(graphs, streams):
        with torch.cuda.graph(g, stream=s):
            call(1, torch.cuda.current_stream().cuda_stream)
    for replay in range(20):
        print("replays of the same call: %d descriptors, round %d" % (n, replay), flush=True)
        buf.reset()
        mapped.flags[0] = mapped.flags[1] = 0
        for _ in range(5):
            for g, s in zip(graphs, streams):
                with torch.cuda.stream(s):
                    g.replay()
        torch.cuda.synchronize()
        assert int(mapped.flags[1]) == 77 and first_difference(buf.result(), expect) is None
        buf.reset()
        call(0, streams[0].cuda_stream)
        torch.cuda.synchronize()
        assert int(mapped.flags[0]) == 77 and first_difference(buf.result(), expect) is None
    mapped.free()


@pytest.mark.parametrize("n", [1, 5, 16, 40])
@pytest.mark.parametrize("captured", [False, True])
def test_a_list_rewritten_between_calls_is_read_afresh(pkg, hip, oracle, n, captured):
    """The same slot of mapped memory and the same completion word, another list each time, written as soon as the word
    says that the last one has been copied: the descriptors come through a cache, which must not keep the last list's."""
    import torch

    pool = np.random.default_rng(n).integers(0, 256, PAGES * 4096, dtype=np.uint8)
    room = n * 5000 + 3 * 4096
    lists = [ragged_list(n, 1000 * n + k)[0] for k in range(60)]
    expect = [oracle_expected(oracle, pool, d, room) for d in lists]
    buf = GpuBuffers(pool, lists[0], room)
    mapped = Mapped(pkg, hip, lists[0], 1)
    stream = torch.cuda.Stream()

    def call():
        pkg.check(
            hip.tcpxuUnpackSlotNoAlloc(0, buf.pool.data_ptr(), buf.dst_base, mapped.desc_dev(0), n, mapped.flag_dev(0), 5, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
            "tcpxuUnpackSlotNoAlloc",
        )

    with torch.cuda.stream(stream):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    if captured:
        with torch.cuda.graph(graph, stream=stream):
            call()
    print("lists of %d rewritten, captured: %s" % (n, captured), flush=True)
    for k, d in enumerate(lists):
        buf.reset()
        mapped.flags[0] = 0
        ctypes.memmove(mapped.host.value + mapped.flag_bytes, d.ctypes.data, d.nbytes)
        for _ in range(2):  # the second right behind the first, with the list that the first one has seen
            with torch.cuda.stream(stream):
                graph.replay() if captured else call()
            mapped.wait(0, 5)
            mapped.flags[0] = 0
        assert first_difference(buf.result(), expect[k]) is None, "list %d" % k
    torch.cuda.synchronize()
    mapped.free()
