"""The time-out of tcpxSynthRunRequests' poll loop, also for waits of more than 2^32 polls (no GPU;
tests/native/quiet_timeout.cc)."""
import os
import subprocess

from plugin_common import ROOT


def test_a_wait_of_more_polls_than_32_bits_count_ends():
    out = os.path.join(ROOT, "tests", "native", "build")
    os.makedirs(out, exist_ok=True)
    exe = os.path.join(out, "quiet_timeout")
    subprocess.check_call(
        ["g++", "-std=c++17", "-O2", "-Wall", "-I" + os.path.join(ROOT, "include"),
         "-I" + os.path.join(ROOT, "nccl-plugin-gpudirecttcpx_amd", "csrc", "plugin"),
         os.path.join(ROOT, "tests", "native", "quiet_timeout.cc"), "-o", exe]
    )  # fmt: skip
    p = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=60)
    assert p.returncode == 0 and "quiet time-out ok" in p.stdout, p.stdout
