"""The threads a context keeps for large host arrays (csrc/host_pool.h), in a program of their own: every part is done once, calls
may follow one another, a process has no more of them than CPUs beside the caller's, and one forked off after the workers started
has none of them: it must neither wait for them where it uses a pool of its parent's nor where it destroys one."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <dirent.h>
#include <sched.h>
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
  const pid_t child = fork();
  if (child == 0) {  // a process that may use one CPU, or two: the caller and so many workers
    alarm(20);
    for (int cpus = 1; cpus <= 2; ++cpus) {
      cpu_set_t all, some;
      if (sched_getaffinity(0, sizeof all, &all) != 0 || CPU_COUNT(&all) < cpus) _exit(0);
      CPU_ZERO(&some);
      for (int i = 0, n = 0; n < cpus; ++i)
        if (CPU_ISSET(i, &all)) CPU_SET(i, &some), ++n;
      if (sched_setaffinity(0, sizeof some, &some) != 0) _exit(0);
      nnvhip::HostPool pool;
      if (!each_once(pool, 16)) _exit(6);
      DIR* tasks = opendir("/proc/self/task");
      int n = 0;
      while (const dirent* e = readdir(tasks)) n += e->d_name[0] != '.';
      closedir(tasks);
      if (n != cpus) _exit(7);
      if (sched_setaffinity(0, sizeof all, &all) != 0) _exit(0);
    }
    _exit(0);
  }
  int status = 0;
  if (waitpid(child, &status, 0) != child || status != 0) return 8;
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
