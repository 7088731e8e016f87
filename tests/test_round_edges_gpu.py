"""Rounds of a wavefront's copy at the lengths where their parts begin and end: 64, 128, 192 and 256 vectors more or less a
vector, where the dword behind the last vector moves to another register or to a load of its own, for every shift of the
source against the destination and boundaries all along a line; and one fragment beyond 2 GiB, whose offsets need all of
their 32 bits.  Byte-exact against the CPU oracle (the long one against the bytes it was cut from)."""
import numpy as np
import pytest

from conftest import GUARD, SENTINEL, GpuBuffers, first_difference, make_descs, oracle_expected
from test_engine_gpu import Engine, Mapped

pytestmark = pytest.mark.gpu

SLOT = 2 * 4096  # of the pool, for one fragment


def run(pkg, hip, kernel, bounce, dst, descs_dev, n, mapped):
    """The list through one kernel; mapped holds it, too, and a completion word."""
    import torch

    if kernel == "batch":
        pkg.check(hip.tcpxuUnpackBatch(0, bounce, dst, descs_dev, n, None), "tcpxuUnpackBatch")
    elif kernel == "noalloc":
        pkg.check(hip.tcpxuUnpackSlotNoAlloc(0, bounce, dst, mapped.desc_dev(0), n, mapped.flag_dev(0), 7, None), "tcpxuUnpackSlotNoAlloc")
    else:
        engine = Engine(pkg, hip)
        engine.start()
        engine.submit(bounce, dst, mapped.desc_dev(0), n, mapped.flag_dev(0), 7)
        mapped.wait(0, 7)
        engine.destroy()
    torch.cuda.synchronize()


@pytest.mark.parametrize("kernel", ["batch", "noalloc", "engine"])
@pytest.mark.parametrize("vectors", [64, 128, 192, 256])
def test_lengths_around_whole_registers(pkg, hip, oracle, kernel, vectors):
    rng = np.random.default_rng(vectors)
    rows, dst = [], 0
    for skew in range(4):
        for start in (0, 1, 16, 63, 112, 127):  # where in a line the first of a run of three starts
            dst = (dst + 127) // 128 * 128 + start
            for extra in rng.permutation([-17, -16, -3, 0, 1, 16, 19, 130])[:4]:
                length = min(16 * vectors + int(extra), SLOT - 16)
                rows.append([len(rows) * SLOT + (dst + skew) % 16, length, dst])
                dst += length
            dst += 1  # a guard byte between runs
    rows[-1][0] = len(rows) * SLOT - rows[-1][1]  # the last one ends with the pool
    descs = make_descs(rows)
    pool = rng.integers(0, 256, len(rows) * SLOT, dtype=np.uint8)
    expect = oracle_expected(oracle, pool, descs, dst)
    buf, mapped = GpuBuffers(pool, descs, dst), Mapped(pkg, hip, descs, 1)
    print("%s: %d descriptors around %d vectors" % (kernel, len(descs), vectors), flush=True)
    run(pkg, hip, kernel, buf.pool.data_ptr(), buf.dst_base, buf.descs.data_ptr(), len(descs), mapped)
    mapped.free()
    assert first_difference(buf.result(), expect) is None


@pytest.mark.parametrize("kernel", ["batch", "noalloc"])
def test_fragment_beyond_2_gib(pkg, hip, kernel):
    """Between two of ordinary size that continue it, so that both of its ends lie in shared lines."""
    import torch

    lens = [1000, (1 << 31) + 4099, 3000]
    srcs = [5, 4097, 4097 + lens[1] + 11]
    dsts = np.cumsum([0] + lens[:-1]) + 3
    descs = make_descs(zip(srcs, lens, dsts))
    pool = torch.randint(-(2**63), 2**63 - 1, ((srcs[2] + lens[2]) // 8 + 1,), dtype=torch.int64, device="cuda:0").view(torch.uint8)
    out = torch.full((GUARD + 3 + sum(lens) + GUARD,), SENTINEL, dtype=torch.uint8, device="cuda:0")
    on_gpu = torch.from_numpy(descs.view(np.uint8).copy()).to("cuda:0")
    mapped = Mapped(pkg, hip, descs, 1)
    torch.cuda.synchronize()
    print("%s: a fragment of %d bytes" % (kernel, lens[1]), flush=True)
    run(pkg, hip, kernel, pool.data_ptr(), out.data_ptr() + GUARD, on_gpu.data_ptr(), len(descs), mapped)
    mapped.free()
    for src, length, dst in zip(srcs, lens, dsts):
        assert torch.equal(out[GUARD + int(dst) :][:length], pool[src : src + length])
    assert bool((out[: GUARD + 3] == SENTINEL).all()) and bool((out[-GUARD:] == SENTINEL).all())


@pytest.mark.parametrize("per_ticket", [0, 8, 16, 17, 24, 33, 64])
def test_rounds_in_pairs(pkg, hip, oracle, per_ticket):
    """Shares of one to eight fragments a wavefront, odd and even, with tiny, empty and several-round fragments first, second
    and last in a pair: requests of one ticket (pairs), of several small ones (one at a time), of several large ones (pairs)."""
    engine = Engine(pkg, hip, descs_per_ticket=per_ticket)
    engine.start()
    for n in (1, 2, 8, 9, 15, 16, 17, 31, 64, 65, 130):
        rng = np.random.default_rng(100 * per_ticket + n)
        lens = rng.choice([0, 1, 29, 31, 700, 2048, 4095, 4096, 4097, 9000], size=n, p=[0.1, 0.05, 0.05, 0.05, 0.2, 0.2, 0.1, 0.1, 0.05, 0.1])
        descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
        descs["len"], descs["dst_off"] = lens, np.cumsum(lens) - lens
        descs["src_off"] = rng.integers(0, (1 << 20) - 9000, n)
        pool = rng.integers(0, 256, 1 << 20, dtype=np.uint8)
        total = int(lens.sum())
        expect = oracle_expected(oracle, pool, descs, total, 5)
        buf, mapped = GpuBuffers(pool, descs, total, 5), Mapped(pkg, hip, descs, 1)
        print("tickets of %d, %d descriptors, %d bytes" % (per_ticket, n, total), flush=True)
        engine.submit(buf.pool.data_ptr(), buf.dst_base, mapped.desc_dev(0), n, mapped.flag_dev(0), 9)
        mapped.wait(0, 9)
        assert first_difference(buf.result(), expect) is None
        mapped.free()
    engine.destroy()


@pytest.mark.parametrize("per_ticket", [18, 19, 24, 32, 33])
def test_rounds_of_fragments_on_lines(pkg, hip, oracle, per_ticket):
    """Fragments of whole destination lines, some of several rounds: in tickets of 19 to 32 one round at a time, in smaller and
    larger ones and in a request's only ticket in pairs; with one fragment off the lines, in pairs as well."""
    engine = Engine(pkg, hip, descs_per_ticket=per_ticket)
    engine.start()
    for n in (per_ticket - 1, per_ticket, per_ticket + 1, 3 * per_ticket + 5):
        for odd in (0, 1):
            rng = np.random.default_rng(100 * per_ticket + 2 * n + odd)
            lens = rng.choice([128, 1024, 2048, 4096, 4096 + 128, 9 * 1024], size=n)
            lens[-1] += 4 * odd
            descs = np.zeros(n, dtype=np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")]))
            descs["len"], descs["dst_off"] = lens, np.cumsum(lens) - lens
            descs["src_off"] = rng.integers(0, (1 << 20) - 9500, n)
            pool = rng.integers(0, 256, 1 << 20, dtype=np.uint8)
            total = int(lens.sum())
            expect = oracle_expected(oracle, pool, descs, total, 0)
            buf, mapped = GpuBuffers(pool, descs, total, 0), Mapped(pkg, hip, descs, 1)
            assert buf.dst_base % 128 == 0
            print("tickets of %d, %d descriptors, %d bytes" % (per_ticket, n, total), flush=True)
            engine.submit(buf.pool.data_ptr(), buf.dst_base, mapped.desc_dev(0), n, mapped.flag_dev(0), 9)
            mapped.wait(0, 9)
            assert first_difference(buf.result(), expect) is None
            mapped.free()
    engine.destroy()
