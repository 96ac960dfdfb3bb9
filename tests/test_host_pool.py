"""The threads a context keeps for large host arrays (csrc/host_pool.h), in a program of their own: every part is done once, calls
may follow one another, and a process forked off after the workers started has none of them: it must neither wait for them where
it uses a pool of its parent's nor where it destroys one."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <sys/wait.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <memory>

#include "host_pool.h"

static bool each_once(nnvhip::HostPool& pool, int parts) {
  std::unique_ptr<std::atomic<int>[]> seen(new std::atomic<int>[parts + 1]());
  pool.run(parts, [&](int i) { ++seen[i]; });
  for (int i = 0; i < parts; ++i)
    if (seen[i] != 1) return false;
  return true;
}

int main() {
  std::unique_ptr<nnvhip::HostPool> used(new nnvhip::HostPool()), fresh(new nnvhip::HostPool());
  for (int round = 0; round < 200; ++round)
    for (int parts : {0, 1, 2, 3, 4, 16, 97})
      if (!each_once(*used, parts)) return 1;
  for (bool use : {false, true}) {
    const pid_t child = fork();
    if (child == 0) {
      alarm(20);  // (a child that waits for ever ends by this signal)
      if (use && !(each_once(*used, 16) && each_once(*used, 5) && each_once(*fresh, 16))) _exit(2);
      used.reset();
      fresh.reset();
      _exit(0);
    }
    int status = 0;
    if (waitpid(child, &status, 0) != child || status != 0) return 3 + use;
  }
  return each_once(*used, 16) && each_once(*fresh, 16) ? 0 : 5;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_every_part_once_and_forked_processes(tmp_path):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(PROGRAM)
    p = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", os.path.join(ROOT, "nnv_amd", "csrc"), str(src), "-o", str(exe)],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert p.returncode == 0, p.stdout
    assert subprocess.run([str(exe)], timeout=100).returncode == 0
