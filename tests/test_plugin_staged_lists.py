"""The second copy of a request's descriptors is written by whole lines of four: lists that end within a line, fill it or go one
beyond, small ones and of a request that is alone (no GPU: the emulated device of tests/emu)."""
import numpy as np
import pytest

from test_plugin_host import ARENA_BYTES, comm, env, host_buffer  # noqa: F401  (fixtures)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 13, 15, 16, 17, 19, 509, 511, 512])
def test_a_second_copy_of_any_length(env, comm, n):  # noqa: F811
    rng = np.random.default_rng(n)
    frags = np.zeros(n, dtype=env.pkg.Workload(1, shrink=6).frag_dtype)
    frags["frag_size"] = rng.integers(1, 200, n)
    frags["frag_token"] = rng.permutation(n) % (ARENA_BYTES // 4096)
    frags["frag_offset"] = frags["frag_token"] * 4096 + rng.integers(0, 3896, n)
    env.arena_np[:] = rng.integers(0, 256, len(env.arena_np), dtype=np.uint8)
    total = int(frags["frag_size"].sum())
    buf, ptr = host_buffer(total)
    mh = comm.reg(ptr, total)
    copies = env.emu.emu_counter(6)
    rc, req = comm.irecv(ptr, total, mh)
    assert rc == 0
    comm.ctrl(0, total, 0, total)
    comm.deliver(0, frags)
    for _ in range(100000):
        rc, done = comm.test(req)[:2]
        assert rc == 0
        if done:
            break
    assert done and env.emu.emu_counter(6) == copies + 1
    assert comm.consumed(req) == 0
    comm.dereg(mh)
    assert buf.tobytes() == b"".join(env.arena_np[int(f["frag_offset"]) :][: int(f["frag_size"])].tobytes() for f in frags)
