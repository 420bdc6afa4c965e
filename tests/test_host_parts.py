"""Host work split over threads (csrc/host_parts.hpp): every part runs, once, also where
the system refuses threads.  Compiled and run on the CPU."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kore_amd", "csrc")

PROGRAM = r"""
#include "host_parts.hpp"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <sys/resource.h>
#include <unistd.h>
int main(int argc, char** argv) {
  const int n = atoi(argv[1]);
  if (argc > 2) {                        // no thread may be started from here on (root is exempt, so not as root)
    if (geteuid() == 0 && (setgid(65534) || setuid(65534))) return 3;
    const rlimit none{0, 0};
    if (setrlimit(RLIMIT_NPROC, &none)) return 3;
    bool refused = false;
    try { std::thread t([] {}); t.join(); } catch (const std::exception&) { refused = true; }
    if (!refused) return 3;
  }
  std::atomic<int> runs[64] = {};
  auto part = [&](int t) { ++runs[t]; };
  run_parts(n, part);
  for (int t = 0; t < 64; ++t)
    if (runs[t] != (t < n)) return 1;
  puts("all parts ran once");
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("parts")
    (d / "parts.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(d / "parts.cpp"), "-o", str(d / "parts")],
                   check=True)
    return str(d / "parts")


@pytest.mark.parametrize("n", [1, 2, 8, 16])
@pytest.mark.parametrize("refuse", [False, True])
def test_every_part_runs(program, n, refuse):
    r = subprocess.run([program, str(n)] + (["refuse"] if refuse else []), capture_output=True, text=True)
    if r.returncode == 3:
        pytest.skip("this system does not refuse threads")
    assert r.returncode == 0 and "all parts ran once" in r.stdout, r
