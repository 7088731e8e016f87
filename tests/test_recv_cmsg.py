"""Control messages and the synthetic socket that writes them, against plain restatements (no GPU;
tests/native/recv_cmsg.cc, under AddressSanitizer and with the flags that the plugin ships with)."""
import os
import subprocess

import pytest

from plugin_common import ROOT
from test_sanitizers import CSRC, SOURCES


def shipped_flags():
    return subprocess.check_output(["make", "-s", "-C", CSRC, "print-cxxflags"], text=True).split()


@pytest.mark.parametrize("build", ["sanitized", "shipped"])
def test_control_messages_of_any_kind_and_room(tmp_path, build):
    exe = str(tmp_path / "recv_cmsg")
    sources = [os.path.join(ROOT, "tests", "native", "recv_cmsg.cc")] + [s for s in SOURCES if os.path.join("csrc", "plugin") in s]
    sanitized = ["-std=c++17", "-O2", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined"]
    flags = sanitized if build == "sanitized" else shipped_flags()
    subprocess.check_call(
        ["g++", *flags, "-I" + os.path.join(ROOT, "include"),
         "-I" + os.path.join(CSRC, "plugin"), *sources, "-o", exe, "-pthread", "-ldl"]
    )  # fmt: skip
    p = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert p.returncode == 0 and "control messages ok" in p.stdout, p.stdout[-3000:]
