"""Control messages and the synthetic socket that writes them, against plain restatements (no GPU;
tests/native/recv_cmsg.cc, under AddressSanitizer)."""
import os
import subprocess

from plugin_common import ROOT
from test_sanitizers import CSRC, SOURCES


def test_control_messages_of_any_kind_and_room(tmp_path):
    exe = str(tmp_path / "recv_cmsg")
    sources = [os.path.join(ROOT, "tests", "native", "recv_cmsg.cc")] + [s for s in SOURCES if os.path.join("csrc", "plugin") in s]
    subprocess.check_call(
        ["g++", "-std=c++17", "-O2", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-I" + os.path.join(ROOT, "include"),
         "-I" + os.path.join(CSRC, "plugin"), *sources, "-o", exe, "-pthread", "-ldl"]
    )  # fmt: skip
    p = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert p.returncode == 0 and "control messages ok" in p.stdout, p.stdout[-3000:]
