"""The map of generated kernels that a backward reads on PyTorch's threads while a first call of another element type adds to it: run
under the thread sanitizer (host code only)."""

import shutil
import subprocess
from pathlib import Path

import pytest

HOST = Path(__file__).resolve().parent.parent / "cuequivariance_amd" / "csrc" / "host"
PROGRAM = r"""
#include "shared_map.h"
#include <cstdio>
#include <thread>
#include <vector>
struct Unit { void* entry[6]; long from[3]; };
int main() {
  cueq_host::SharedMap<Unit> units;
  std::vector<std::thread> threads;
  long seen[4] = {0, 0, 0, 0};
  for (int t = 0; t < 4; ++t)
    threads.emplace_back([&, t] {
      for (int i = 0; i < 2000; ++i) {
        if (i % 50 == 0) units.set(t * 64 + i / 50, Unit{{}, {t, i, 1}});
        if (const auto u = units.find((t ^ 1) * 64 + i / 50)) seen[t] += u->from[2];
      }
    });
  for (auto& t : threads) t.join();
  for (int t = 0; t < 4; ++t)
    for (int i = 0; i < 2000; i += 50) {
      const auto u = units.find(t * 64 + i / 50);
      if (!u || u->from[0] != t || u->from[1] != i) return 2;
    }
  std::puts("whole");
}
"""


def test_entries_added_while_others_are_looked_up(tmp_path):
    gxx = shutil.which("g++")
    flags = ["-std=c++17", "-O1", "-g", "-fsanitize=thread", "-pthread", f"-I{HOST}"]

    def build(name, text):
        (tmp_path / f"{name}.cpp").write_text(text)
        subprocess.run([gxx, *flags, str(tmp_path / f"{name}.cpp"), "-o", str(tmp_path / name)], check=True, capture_output=True, timeout=120)
        return subprocess.run([str(tmp_path / name)], capture_output=True, text=True, timeout=120)

    try:
        if gxx is None or build("nothing", "int main() { return 0; }").returncode:
            pytest.skip("no thread sanitizer here")
    except subprocess.CalledProcessError:
        pytest.skip("no thread sanitizer here")
    r = build("map", PROGRAM)
    assert r.returncode == 0 and "whole" in r.stdout and "data race" not in r.stderr, r.stderr[-2000:]
