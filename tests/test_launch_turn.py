"""Turns of the calls on one workspace (fast_v2_amd/csrc/launch_turn.h), built for the host."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

PROG = r"""
#include <stdio.h>
#include <thread>
#include <vector>
#include "launch_turn.h"

// two threads "launch" calls of two kernels on one workspace; the stream's order must hold
// each call's kernels next to each other
int main() {
  static char memory[1 << 20];
  std::mutex queue;
  std::vector<int> stream;
  auto kernel = [&](int id) {
    std::lock_guard<std::mutex> g(queue);
    stream.push_back(id);
  };
  auto caller = [&](int id) {
    for (int i = 0; i < 2000; ++i) {
      const fdllm::WorkspaceTurn turn(memory);
      kernel(id);
      std::this_thread::yield();
      kernel(id);
    }
  };
  std::thread a(caller, 1), b(caller, 2);
  a.join();
  b.join();
  for (size_t i = 0; i < stream.size(); i += 2)
    if (stream[i] != stream[i + 1]) return 1;
  // a call without a workspace and one on another workspace do not wait
  const fdllm::WorkspaceTurn held(memory);
  std::thread c([&] {
    const fdllm::WorkspaceTurn none(nullptr);
    const fdllm::WorkspaceTurn other(memory + 4096);
    puts("free");
  });
  c.join();
  return stream.size() == 8000 ? 0 : 2;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_kernels_of_one_call_stay_together(tmp_path):
    src, exe = tmp_path / "turn.cc", tmp_path / "turn"
    src.write_text(PROG)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(ROOT / "fast_v2_amd" / "csrc"), str(src), "-o",
                    str(exe)], check=True, capture_output=True, text=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "free\n", (r.returncode, r.stdout)
