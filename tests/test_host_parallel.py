"""The host's parallel loop (csrc/mose_host.hpp) covers its range once, also where no thread can be started: a failed
thread must not end the process through the C ABI."""
import os
import resource
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mose-gpu_amd", "csrc")

MAIN = r"""
#include <sys/resource.h>
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "mose_host.hpp"

int main(int argc, char** argv) {
  const size_t n = std::strtoul(argv[1], nullptr, 10);
  std::vector<int> hits(n, 0);
  if (argc > 2) {                       // no room for a thread's stack
    rlimit a{48ul << 20, 48ul << 20};
    if (setrlimit(RLIMIT_AS, &a) != 0) return 3;
    bool started = true;
    try { std::thread([] {}).join(); } catch (...) { started = false; }
    if (started) return 4;
  }
  mose::host_parallel(n, [&](size_t a, size_t b) { for (size_t q = a; q < b; ++q) ++hits[q]; });
  for (int h : hits) if (h != 1) return 5;
  std::puts("covered");
  return 0;
}
"""


def stacks():
    """Threads of the program ask for stacks of 64 MiB."""
    resource.setrlimit(resource.RLIMIT_STACK, (64 << 20, resource.getrlimit(resource.RLIMIT_STACK)[1]))


@pytest.mark.parametrize("starved", [False, True], ids=["threads", "no-threads"])
def test_range_covered_once(tmp_path, starved):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "main.cpp", tmp_path / "main"
    src.write_text(MAIN)
    subprocess.run([cxx, "-O1", "-std=c++17", "-pthread", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    for n in (0, 1, 32767, 32768, 100003):
        r = subprocess.run([str(exe), str(n)] + (["starved"] if starved else []), capture_output=True, text=True,
                           preexec_fn=stacks)
        assert r.returncode == 0 and r.stdout == "covered\n", (n, r.returncode, r.stderr)
