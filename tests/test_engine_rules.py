"""The engine's decisions by numbers (csrc/hip/engine_rules.h), compiled and run on the host (tests/native/engine_rules.cc)."""
import os
import subprocess

from plugin_common import ROOT
from test_sanitizers import CSRC


def test_engine_rules(tmp_path):
    exe = str(tmp_path / "engine_rules")
    subprocess.check_call(
        ["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-function", "-I" + os.path.join(CSRC, "hip"), os.path.join(ROOT, "tests", "native", "engine_rules.cc"), "-o", exe]
    )  # fmt: skip
    p = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert p.returncode == 0 and "engine rules ok" in p.stdout, p.stdout[-3000:]
