"""The device's error word: each cause has its own bit and comes back as its own
status, alone and beside others."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

TU = r"""
#include <cstdio>
#include "errors.hpp"
int main() {
  using namespace evd;
  const unsigned bits[] = {kErrTimeout, kErrNonfinite, kErrNoconverge, kErrRange};
  for (unsigned a : bits) std::printf("%u %d %s\n", a, device_error_code(a), device_error_text(a));
  std::printf("%d %d %d %d\n", device_error_code(kErrRange | kErrNoconverge), device_error_code(kErrRange | kErrNonfinite),
              device_error_code(kErrNoconverge | kErrTimeout), device_error_code(1u << 20));
}
"""


def test_every_cause_is_reported_as_itself(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src = tmp_path / "word.cpp"
    src.write_text(TU)
    exe = tmp_path / "word"
    res = subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", str(ROOT / "evd4sc2025_amd" / "csrc"), str(src),
                          "-o", str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60).stdout.splitlines()
    rows = [line.split(" ", 2) for line in out[:4]]
    words = [int(r[0]) for r in rows]
    assert len({w.bit_length() for w in words}) == 4 and all(w & (w - 1) == 0 for w in words)
    assert [int(r[1]) for r in rows] == [4, 3, 6, 7]  # TIMEOUT, NONFINITE, NOCONVERGE, RANGE
    assert len({r[2] for r in rows}) == 4
    # the cause that others may follow from goes first; no known bit is no cause of the library
    assert out[4] == "6 3 4 1"


def test_kernels_raise_bits_only():
    for f in (ROOT / "evd4sc2025_amd" / "csrc").glob("*.h*"):
        for arg in re.findall(r"atomicOr\(err, ([^)]*)\)", f.read_text()):
            assert arg.startswith("kErr"), (f.name, arg)
