"""What kernel launches do once for each GPU of a process (grx_once.h, host
code alone): the second device's first call runs too, a call that failed runs
again, and a device past the table runs every time."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gorelaxor_amd", "csrc")

PROGRAM = r"""
#include "grx_once.h"
#include <cstdio>
int main() {
    static GrxDeviceOnce once;
    int calls = 0;
    auto ok = [&] { ++calls; return true; };
    auto bad = [&] { ++calls; return false; };
    bool r[8];
    int n[8], i = 0;
    auto rec = [&](bool v) { r[i] = v, n[i] = calls, ++i; };
    rec(once.run(0, ok));    // first on device 0
    rec(once.run(0, bad));   // done there
    rec(once.run(1, bad));   // device 1 is another: runs, and fails
    rec(once.run(1, ok));    // again after the failure
    rec(once.run(1, bad));   // done
    rec(once.run(63, ok));
    rec(once.run(64, ok));   // past the table
    rec(once.run(64, bad));
    for (int k = 0; k < i; ++k) printf("%d:%d ", (int)r[k], n[k]);
}
"""


def test_once_for_each_device(tmp_path):
    src, exe = tmp_path / "once.cpp", tmp_path / "once"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["1:1", "1:1", "0:2", "1:3", "1:3", "1:4", "1:5", "0:6"]


@pytest.mark.parametrize("source", sorted(f for f in os.listdir(CSRC) if f.endswith(".hip")))
def test_lds_limits_are_asked_for_each_device(source):
    """No source keeps a raised LDS limit in a flag of the whole process."""
    text = open(os.path.join(CSRC, source)).read()
    for flag in ("static bool raised", "static bool attr", "static const bool ok", "static const hipError_t"):
        assert flag not in text
