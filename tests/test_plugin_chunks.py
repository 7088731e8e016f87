"""Chunks that are there whole when their control message is read, there in part, or not there yet: received into the
slot at once, the rest of it by a task, or by a task altogether (no GPU: the emulated device of tests/emu)."""
import numpy as np
import pytest

from plugin_common import expected_bytes
from test_plugin_host import ARENA_BYTES, INTERNAL_ERROR, comm, drive_until_transmitted, env, host_buffer, simple_request  # noqa: F401


def message(env, n, seed):
    """n fragments of 1 to 4096 bytes on pages of their own, every third one empty."""
    rng = np.random.default_rng(seed)
    frags = np.zeros(n, dtype=env.pkg.Workload(1, shrink=6).frag_dtype)
    pages = rng.choice(ARENA_BYTES // 4096, size=n, replace=False)
    frags["frag_size"] = rng.integers(2, 4097, size=n)
    frags["frag_size"][1::3] = 0
    frags["frag_offset"] = pages * 4096 + (rng.integers(0, 4097, size=n) % (4097 - np.maximum(frags["frag_size"], 1)))
    frags["frag_token"] = pages
    return frags


@pytest.mark.parametrize("there", [0, 1, 4, 29, 30])
@pytest.mark.parametrize("cut", [None, 1, 2000])
def test_a_chunk_of_which_only_a_part_has_arrived(env, comm, there, cut):  # noqa: F811
    """Two chunks on one flow and one on another; `there` fragments of the first flow have arrived when the control
    messages are read.  `cut`: the boundary between its two chunks lies that many bytes into a fragment."""
    comm.emu = env.emu
    env.arena_np[:] = np.random.default_rng(1).integers(0, 256, ARENA_BYTES, dtype=np.uint8)
    a, b = message(env, 30, 10 + there), message(env, 7, 500)
    size_a, size_b = int(a["frag_size"].sum()), int(b["frag_size"].sum())
    first = int(a["frag_size"][:15].sum()) + (min(cut, int(a["frag_size"][15]) - 1) if cut else 0)
    total = size_a + size_b
    buf, ptr = host_buffer(total + 16)
    mh = comm.reg(ptr, total)
    env.emu.emu_set_hold(1)
    rc, req = comm.irecv(ptr, total, mh)
    assert rc == 0
    comm.ctrl(0, first, 0, total)
    comm.ctrl(0, size_a - first, first, total)
    comm.ctrl(3, size_b, size_a, total)
    comm.deliver(0, a[:there])
    for _ in range(5):
        assert comm.test(req)[:2] == (0, 0)
    assert env.emu.emu_pending() == 0, "handed over with bytes missing"
    comm.deliver(0, a[there:])
    for _ in range(3):
        assert comm.test(req)[:2] == (0, 0)
    comm.deliver(3, b)
    drive_until_transmitted(comm, req)
    rows, cnt = comm.slot(comm.queue_state()[0] % 16)
    rows = rows[:cnt]
    assert cnt == 37 + (cut is not None)  # the fragment that the boundary cuts has a descriptor in each chunk
    live = rows[rows["len"] != 0]
    order = np.argsort(live["dst_off"])
    assert np.array_equal(np.cumsum(live["len"][order]), np.append(live["dst_off"][order][1:], total))
    assert comm.outstanding_pages() == cnt
    env.emu.emu_release(1)
    assert comm.test(req)[:2] == (0, 1)
    request = np.zeros(1, dtype=env.pkg.Workload(1, shrink=6).req_dtype)
    request["n_descs"] = 37
    want = expected_bytes(env.arena_np, np.concatenate([a, b]), request, total + 16)
    assert np.array_equal(buf, want)
    assert comm.consumed(req) == 0 and comm.outstanding_pages() == 0
    comm.dereg(mh)


@pytest.mark.parametrize("fragments", [2047, 2048])
def test_a_slot_that_is_just_full_and_one_descriptor_more(env, comm, fragments):  # noqa: F811
    """Chunks of 1024 and 1023 fragments fill a slot but for one descriptor; one of two more than that leaves is refused
    before anything is written past the slot's list (src/net_tcpx.cc:1350-1353)."""
    comm.emu = env.emu
    last = fragments - 2047 + 1  # 1: just full; 2: one more than the slot holds
    n = 1024 + 1023 + last
    frags = np.zeros(n, dtype=env.pkg.Workload(1, shrink=6).frag_dtype)
    frags["frag_offset"] = np.arange(n) * 4096
    frags["frag_size"] = 2
    frags["frag_token"] = np.arange(n)
    buf, ptr = host_buffer(2 * n)
    mh = comm.reg(ptr, 2 * n)
    rc, req = comm.irecv(ptr, 2 * n, mh)
    at = 0
    for flow, count in ((0, 1024), (1, 1023), (2, last)):
        comm.ctrl(flow, 2 * count, 2 * at, 2 * n)
        comm.deliver(flow, frags[at : at + count])
        at += count
    for _ in range(20):
        rc, done, _ = comm.test(req)
        if rc or done:
            break
    if last == 2:
        assert rc == INTERNAL_ERROR
        return
    assert (rc, done) == (0, 1) and comm.consumed(req) == 0
    pages = env.arena_np[: 4096 * n].reshape(n, 4096)
    assert np.array_equal(buf, pages[:, :2].reshape(-1))
    comm.dereg(mh)


@pytest.mark.parametrize("there", [0, 1, 1000, 2046, "all"])
@pytest.mark.parametrize("fragments", [2047, 2048])
def test_the_most_fragments_of_one_chunk(env, comm, fragments, there):  # noqa: F811
    """A chunk of 2048 fragments is refused (src/sock/tcpx.h:183-187) and one of 2047 is not, however much of it is there
    when its control message is read."""
    comm.emu = env.emu
    frags = np.zeros(fragments, dtype=env.pkg.Workload(1, shrink=6).frag_dtype)
    frags["frag_offset"] = np.arange(fragments) * 4096
    frags["frag_size"] = 2
    frags["frag_token"] = np.arange(fragments)
    there = fragments if there == "all" else there
    buf, ptr = host_buffer(2 * fragments)
    mh = comm.reg(ptr, 2 * fragments)
    rc, req = comm.irecv(ptr, 2 * fragments, mh)
    comm.ctrl(0, 2 * fragments, 0, 2 * fragments)
    if there:
        comm.deliver(0, frags[:there])
    if there < fragments:
        assert comm.test(req)[:2] == (0, 0)
        comm.deliver(0, frags[there:])
    for _ in range(20):
        rc, done, _ = comm.test(req)
        if rc or done:
            break
    if fragments == 2048:
        assert rc == INTERNAL_ERROR
        return
    assert (rc, done) == (0, 1) and comm.consumed(req) == 0
    assert np.array_equal(buf, env.arena_np[: 4096 * fragments].reshape(fragments, 4096)[:, :2].reshape(-1))
    comm.dereg(mh)


def test_pages_are_given_back_by_the_comm_that_received_them(env, comm):  # noqa: F811
    """Two comms receive from the same pages; each gives back its own references."""
    other = env.driver.RecvComm(0)
    before = comm.outstanding_pages()
    buf, ptr = host_buffer(3 * 8192)
    reqs = []
    for i, c in enumerate((comm, other, other)):
        mh = c.reg(ptr, 3 * 8192)
        rc, req = c.irecv(ptr + i * 8192, 8192, mh)
        assert rc == 0
        c.ctrl(1, 8192, 0, 8192)
        c.deliver(1, simple_request(env, c))
        while not c.test(req)[1]:
            pass
        reqs.append((c, req))
        assert comm.outstanding_pages() == other.outstanding_pages() == before + 2 * (i + 1)
    for i, (c, req) in enumerate(reqs):
        assert c.consumed(req) == 0
        assert comm.outstanding_pages() == before + 4 - 2 * i
    other.close()
    assert comm.outstanding_pages() == before


@pytest.mark.parametrize("token", [ARENA_BYTES // 4096, 2**32 - 1])
def test_a_token_that_names_no_page(env, comm, token):  # noqa: F811
    """It is received like any other (the bytes are where the fragment's offset says) and refused when it is given back;
    its entry, which does not exist, is neither read nor asked for ahead."""
    frags = np.zeros(16, dtype=env.pkg.Workload(1, shrink=6).frag_dtype)
    frags["frag_offset"] = np.arange(16) * 4096
    frags["frag_size"] = 4096
    frags["frag_token"] = np.arange(16) * 3
    frags["frag_token"][12] = token  # (far enough from the first to be asked for ahead)
    before = comm.outstanding_pages()
    buf, ptr = host_buffer(16 * 4096)
    mh = comm.reg(ptr, 16 * 4096)
    rc, req = comm.irecv(ptr, 16 * 4096, mh)
    comm.ctrl(0, 16 * 4096, 0, 16 * 4096)
    comm.deliver(0, frags)
    while not comm.test(req)[1]:
        pass
    assert np.array_equal(buf, env.arena_np[: 16 * 4096])
    assert comm.outstanding_pages() == before + 15
    assert comm.consumed(req) == INTERNAL_ERROR and comm.outstanding_pages() == before + 3
