"""The second copy of a request's descriptors is written by whole lines of four: lists that end within a line, fill it or go one
beyond, small ones and of a request that is alone; and where the engine brings lists of mapped slots along, a small request that is
alone has none (no GPU: the emulated device of tests/emu)."""
import numpy as np
import pytest

from test_plugin_host import ARENA_BYTES, brings_no_lists, comm, env, host_buffer  # noqa: F401  (fixtures)


def receive(env, comm, sizes, seed, copied):
    """Posts a request for each of `sizes` (fragment counts) before any of their bytes is there, and lets the engine have them all
    before it completes one; `copied` of the lists are copied."""
    rng = np.random.default_rng(seed)
    copies, posted, first = env.emu.emu_counter(6), [], 0
    env.arena_np[:] = rng.integers(0, 256, len(env.arena_np), dtype=np.uint8)
    pages = rng.permutation(sum(sizes)) % (ARENA_BYTES // 4096)
    for n in sizes:
        frags = np.zeros(n, dtype=env.pkg.Workload(1, shrink=6).frag_dtype)
        frags["frag_size"] = rng.integers(1, 200, n)
        frags["frag_token"] = pages[first : first + n]
        frags["frag_offset"] = frags["frag_token"] * 4096 + rng.integers(0, 3896, n)
        first += n
        total = int(frags["frag_size"].sum())
        buf, ptr = host_buffer(total)
        mh = comm.reg(ptr, total)
        rc, req = comm.irecv(ptr, total, mh)
        assert rc == 0
        posted.append((frags, total, buf, mh, req))
    for frags, total, buf, mh, req in posted:
        comm.ctrl(0, total, 0, total)
        comm.deliver(0, frags)
    submitted = env.emu.emu_counter(0)
    env.emu.emu_set_hold(1)  # (none is done before all are at the engine)
    for _ in range(100000):
        assert comm.test(posted[0][4])[:2] == (0, 0)
        if env.emu.emu_counter(0) == submitted + len(sizes):
            break
    assert env.emu.emu_counter(6) - copies == copied
    assert env.emu.emu_release(1 << 20) == len(sizes)
    env.emu.emu_set_hold(0)
    for frags, total, buf, mh, req in posted:
        assert comm.test(req)[:2] == (0, 1) and comm.consumed(req) == 0
        comm.dereg(mh)
        assert buf.tobytes() == b"".join(env.arena_np[int(f["frag_offset"]) :][: int(f["frag_size"])].tobytes() for f in frags)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 13, 15, 16, 17, 19, 509, 511, 512])
def test_a_second_copy_of_any_length(env, brings_no_lists, comm, n):  # noqa: F811
    receive(env, comm, [n], n, 1)


@pytest.mark.parametrize("n", [1, 4, 15, 16, 17, 512, 513])
def test_which_lists_are_copied_where_the_engine_brings_them_along(env, comm, n):  # noqa: F811
    receive(env, comm, [n], n, 1 if 16 < n <= 512 else 0)
    receive(env, comm, [n] * 3, n + 1, 3 if n <= 16 else 0)


class Small:
    """A comm with small requests of 3 descriptors that the engine holds."""

    def __init__(self, env, at):
        self.env, self.comm, self.at, self.held = env, env.driver.RecvComm(0), at, []
        self.buf, self.ptr = host_buffer(4096)
        self.mh = self.comm.reg(self.ptr, 4096)

    def post(self):
        """Hands a request to the engine; whether its list was copied."""
        submitted, copied = self.env.emu.emu_counter(0), self.env.emu.emu_counter(6)
        frags = np.zeros(3, dtype=self.env.pkg.Workload(1, shrink=6).frag_dtype)
        frags["frag_size"], frags["frag_token"] = 100, 3 * (8 * self.at + len(self.held)) + np.arange(3)
        frags["frag_offset"] = 4096 * frags["frag_token"]
        rc, req = self.comm.irecv(self.ptr + 300 * len(self.held), 300, self.mh)
        assert rc == 0
        self.held.append((frags, req))
        self.comm.ctrl(0, 300, 0, 300)
        self.comm.deliver(0, frags)
        for _ in range(100000):
            assert self.comm.test(self.held[0][1])[:2] == (0, 0)  # (only the oldest may be asked for)
            if self.env.emu.emu_counter(0) == submitted + 1:
                return self.env.emu.emu_counter(6) - copied
        raise AssertionError("request never reached the engine")

    def finish(self):
        for frags, req in self.held:
            assert self.comm.test(req)[:2] == (0, 1) and self.comm.consumed(req) == 0
        want = b"".join(self.env.arena_np[int(f["frag_offset"]) :][:100].tobytes() for frags, _ in self.held for f in frags)
        assert self.buf.tobytes()[: len(want)] == want
        self.held = []


@pytest.mark.parametrize("others", [0, 1, 3, 4, 5, 16])
def test_lists_travel_while_few_comms_have_requests_at_the_gpu(env, others):  # noqa: F811
    """The engine is the device's: a small request that is alone in its comm counts what all comms have there."""
    env.arena_np[:] = np.random.default_rng(others).integers(0, 256, len(env.arena_np), dtype=np.uint8)
    comms = [Small(env, i) for i in range(others + 1)]
    env.emu.emu_set_hold(1)
    try:
        for _ in range(2):  # (and again once all have been reported done)
            assert [c.post() for c in comms] == [int(i >= 4) for i in range(others + 1)]
            assert env.emu.emu_release(1 << 20) == others + 1
            for c in comms:
                c.finish()
    finally:
        env.emu.emu_set_hold(0)
        env.emu.emu_release(1 << 20)
        for c in comms:
            c.comm.close()


def test_a_comm_with_several_at_the_gpu_is_a_crowd_until_it_is_done_or_closed(env):  # noqa: F811
    env.arena_np[:] = np.random.default_rng(1).integers(0, 256, len(env.arena_np), dtype=np.uint8)
    busy, other = Small(env, 0), Small(env, 1)
    env.emu.emu_set_hold(1)
    try:
        for closed in (False, True):
            assert [busy.post() for _ in range(3)] == [0, 1, 1]
            assert other.post() == 1
            assert env.emu.emu_release(4) == 4
            other.finish()
            assert other.post() == 1  # (done, but not reported yet)
            assert env.emu.emu_release(1) == 1
            other.finish()
            if closed:
                busy.comm.close()
            else:
                busy.finish()
            assert other.post() == 0
            assert env.emu.emu_release(1) == 1
            other.finish()
    finally:
        env.emu.emu_set_hold(0)
        env.emu.emu_release(1 << 20)
        other.comm.close()
