"""The wait of a host-controlled step: a number that arrives within the limit is
seen whenever it arrives (the limit is a time, not a count of turns), together
with the values written before it, and one that never arrives ends the wait."""
import os
import subprocess

from tests.test_launch_sizes import CSRC, ROCM

PROGRAM = """
#include <cstdio>
#include <thread>
#include "fv_host.h"
int main() {
  using namespace std::chrono;
  for (int late : {0, 30, 300, 3000}) {  // us
    double h[3] = {0, 0, 0};
    std::thread t([&] {
      std::this_thread::sleep_for(microseconds(late));
      h[0] = late + 1.0;
      std::atomic_thread_fence(std::memory_order_release);
      *(volatile double *)(h + 2) = 7.0;
    });
    const bool seen = fv::watch(h + 2, 7.0, 5e6);
    std::printf("%d %d %g\\n", late, (int)seen, h[0]);
    t.join();
  }
  double never = 0.0;
  const auto t0 = steady_clock::now();
  const bool seen = fv::watch(&never, 1.0, 2000.0);
  const double us = duration<double, std::micro>(steady_clock::now() - t0).count();
  std::printf("never %d %d\\n", (int)seen, (int)(us >= 2000.0));
  std::printf("there %d\\n", (int)fv::watch(&never, 0.0, 0.0));
}
"""


def test_watch(tmp_path):
    src, exe = str(tmp_path / "watch.cpp"), str(tmp_path / "watch")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I",
                           os.path.join(ROCM, "include"), "-I", CSRC, "-o", exe, src])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60, check=True).stdout.split("\n")
    assert out[:6] == ["0 1 1", "30 1 31", "300 1 301", "3000 1 3001", "never 0 1", "there 1"]
