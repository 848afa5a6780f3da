"""Host state that several threads' calls share, under ThreadSanitizer (no GPU)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-kunlun_amd", "csrc")

PROGRAM = r"""
#include <thread>
#include <vector>
#include "asked_once.h"
int main() {
  static kmoe::AskedOnce value;
  std::atomic<int> wrong{0}, asked{0};
  if (value.get([] { return 0; }) != 0 || value.get([] { return -1; }) != -1) return 2;  // not kept
  std::vector<std::thread> threads;
  for (int t = 0; t < 8; ++t)
    threads.emplace_back([&] {
      for (int i = 0; i < 1000; ++i)
        if (value.get([&] { asked.fetch_add(1); return 256; }) != 256) wrong.fetch_add(1);
    });
  for (auto& t : threads) t.join();
  return wrong.load() != 0 || asked.load() < 1 || asked.load() > 8 ? 1 : 0;
}
"""


def test_a_value_asked_for_once_by_many_threads(tmp_path):
    src, exe = tmp_path / "once.cc", tmp_path / "once"
    src.write_text(PROGRAM)
    built = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-pthread", "-I", CSRC, str(src), "-o", str(exe)],
                           capture_output=True, text=True)
    if built.returncode and "tsan" in built.stderr:
        pytest.skip("no ThreadSanitizer runtime")
    assert built.returncode == 0, built.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and "data race" not in run.stderr, run.stderr[-2000:]
