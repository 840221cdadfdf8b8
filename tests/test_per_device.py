"""Settings of a kernel that hold for one device (sa_per_device.hpp): made once on each device,
from several threads, and tried again after a failure.  Host code only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "sa_per_device.hpp"
#define EXPECT(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
  sa::per_device_once once;
  int acts = 0;
  auto ok = [&] { ++acts; return 0; };
  EXPECT(once(0, ok) == 0 && once(0, ok) == 0 && acts == 1);
  EXPECT(once(1, ok) == 0 && once(1, ok) == 0 && once(0, ok) == 0 && acts == 2);  // each device
  EXPECT(once(7, [&] { ++acts; return 5; }) == 5 && acts == 3);                    // reported
  EXPECT(once(7, ok) == 0 && acts == 4 && once(7, ok) == 0 && acts == 4);           // and tried again
  EXPECT(once(63, ok) == 0 && once(63, ok) == 0 && acts == 5);
  EXPECT(once(64, ok) == 0 && once(64, ok) == 0 && acts == 7);  // beyond the bits: every time
  sa::per_device_once shared;
  std::atomic<int> n{0};
  std::vector<std::thread> th;
  for (int t = 0; t < 8; ++t)
    th.emplace_back([&, t] { for (int k = 0; k < 1000; ++k) if (shared((t + k) % 4, [&] { ++n; return 0; })) n += 1000000; });
  for (auto &t : th) t.join();
  EXPECT(n >= 4 && n <= 32);
  return 0;
}
"""


def test_once_on_each_device(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src = tmp_path / "once.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "once"
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-pthread", "-I",
                    os.path.join(ROOT, "simulated_annealing_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
