"""A comm's first receive does not pay for what accept could have set up (no GPU: the emulated device of tests/emu)."""
import ctypes
import resource

import numpy as np

from plugin_common import load_emu
from test_plugin_host import host_buffer

ARENA_BYTES = 1 << 30  # (virtual: only the pages that fragments lie in are ever read)


def test_page_references_are_touched_when_the_comm_is_accepted(pkg):
    """A chunk of one fragment from each 4 MiB of the arena: 4 bytes of ledger per page of arena, so every fragment's
    reference lies in a host page of its own, and a ledger that nobody has written to costs a page fault each."""
    emu, lib = load_emu(), pkg.plugin_lib()
    assert lib.tcpxSetDeviceOpsForTesting(emu.emu_ops()) == 0
    assert lib.tcpxInit(None) == 0
    assert lib.tcpxSynthArenaCreate(0, ARENA_BYTES, ctypes.byref(ctypes.c_void_p())) == 0
    from nccl_plugin_gpudirecttcpx_amd.synth_driver import RecvComm

    n = ARENA_BYTES >> 22
    frags = np.zeros(n, dtype=pkg.Workload(1, shrink=6).frag_dtype)
    frags["frag_token"] = np.arange(n) << 10
    frags["frag_offset"] = frags["frag_token"] << 12
    frags["frag_size"] = 64
    buf, ptr = host_buffer(64 * n)

    def faults_of_a_receive(c):
        mh = c.reg(ptr, 64 * n)
        rc, req = c.irecv(ptr, 64 * n, mh)
        assert rc == 0
        c.ctrl(0, 64 * n, 0, 64 * n)
        c.deliver(0, frags)
        before = resource.getrusage(resource.RUSAGE_THREAD).ru_minflt
        done = 0
        while not done:
            rc, done, _ = c.test(req)
            assert rc == 0
        after = resource.getrusage(resource.RUSAGE_THREAD).ru_minflt
        assert c.consumed(req) == 0
        c.dereg(mh)
        return after - before

    warm = RecvComm(0)  # (the process's own first times: code, the arena's pages, the destination)
    faults_of_a_receive(warm)
    fresh = RecvComm(0)
    faults = faults_of_a_receive(fresh)
    fresh.close()
    warm.close()
    assert lib.tcpxFinalize() == 0 and lib.tcpxSetDeviceOpsForTesting(None) == 0
    assert faults < n // 2
