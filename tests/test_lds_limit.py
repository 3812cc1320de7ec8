"""The LDS limit of a kernel that several threads launch: never set below what a launch has been promised, by device, refusals not
remembered. Host code alone, compiled here."""

from __future__ import annotations

import shutil
import subprocess

import pytest

from pyre_amd.hip import build

SOURCE = r"""
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>
#include "pyre_lds.h"

int main() {
  constexpr size_t kb = 1024;
  for (int round = 0; round < 200; ++round) {
    pyre::LdsLimit limit;
    std::atomic<size_t> device[2] = {};  // what the devices hold, as they were last asked
    std::atomic<int> asked{0}, broken{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
      threads.emplace_back([&, t] {
        for (int i = 0; i < 20; ++i) {
          const size_t want = (64 + (t * 37 + i * 11) % 90) * kb;
          const int d = (t + i) % 2;
          const bool ok = limit.allow(d, want, [&](size_t bytes) {
            ++asked;
            std::this_thread::yield();
            device[d] = bytes;
            return true;
          });
          if (!ok || (want > 64 * kb && device[d] < want)) ++broken;
        }
      });
    for (auto& t : threads) t.join();
    if (broken || asked > 2 * 90) return std::printf("lowered %d times, asked %d times\n", broken.load(), asked.load()), 1;
  }
  pyre::LdsLimit limit;
  int asked = 0;
  auto no = [&](size_t) { return ++asked, false; };
  auto yes = [&](size_t) { return ++asked, true; };
  if (!limit.allow(0, 64 * kb, no) || asked) return std::puts("64 KB need no asking"), 1;
  if (limit.allow(0, 65 * kb, no) || !limit.allow(0, 65 * kb, yes) || !limit.allow(0, 65 * kb, no) || asked != 2) return std::puts("a refusal is asked again"), 1;
  if (limit.allow(1, 65 * kb, no) || limit.allow(-1, 65 * kb, yes) || limit.allow(64, 65 * kb, yes)) return std::puts("another device is asked itself"), 1;
  return 0;
}
"""


def test_never_lowered_by_another_thread(tmp_path):
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("no C++ compiler")
    (tmp_path / "limit.cpp").write_text(SOURCE)
    subprocess.run([compiler, "-std=c++17", "-O1", "-pthread", f"-I{build.CSRC}", str(tmp_path / "limit.cpp"), "-o", str(tmp_path / "limit")], check=True)
    done = subprocess.run([str(tmp_path / "limit")], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout


def test_every_kernel_asks_through_it():
    for source in build.CSRC.glob("*.hip"):
        assert "hipFuncSetAttribute" not in source.read_text(), source.name
