"""csrc/lds_limit.h against a stand-in for the runtime (host code only): a thread that comes back from raise_lds_limit
finds the limit raised, also while another thread is still raising it."""
import subprocess

from conftest import ROOT

SOURCE = r"""
#include "lds_limit.h"
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>

static std::atomic<int> calls{0}, raised{0};
static thread_local int device = 0;
extern "C" hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
extern "C" hipError_t hipGetLastError(void) { return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) {
  const bool first = calls++ == 0;
  if (first) std::this_thread::sleep_for(std::chrono::milliseconds(300));
  ++raised;
  return hipSuccess;
}
static void kernel(int) {}

int main() {
  static uint64_t seen = 0;
  std::thread slow([] { mega::raise_lds_limit(&seen, 1, kernel); });
  while (calls == 0) std::this_thread::yield();
  mega::raise_lds_limit(&seen, 1, kernel);
  const int during = raised;                    // the other thread is still inside its call
  slow.join();
  const int before = calls;
  mega::raise_lds_limit(&seen, 1, kernel);      // known by now
  const int again = calls - before;
  device = 1;
  mega::raise_lds_limit(&seen, 1, kernel);      // another device
  printf("%d %d %d\n", during, again, (int)calls - before);
}
"""


def test_no_thread_overtakes_the_limit(tmp_path):
    (tmp_path / "t.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           f"-I{ROOT}/fairseq-apollo_amd/csrc", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t"), "-lpthread"])
    assert subprocess.check_output([str(tmp_path / "t")], timeout=60, text=True).split() == ["1", "0", "1"]
