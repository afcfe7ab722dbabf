"""The multi-column solver's workspace (multi_state.hpp) with allocation calls
that fail on demand: whichever one fails, the call reports it and nothing is
held, and the next call allocates everything; sizes that fit are kept, others
are allocated anew, and every buffer is freed once."""
import os
import subprocess

import pytest

_CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "wnfea_amd", "csrc")

_PROGRAM = r"""
#include "multi_state.hpp"
#include <cstdio>
#include <cstdlib>
#include <set>
static std::set<void*> live;
static int calls = 0, fail_at = -1, bad = 0;
static hipError_t take(void** p) {
  if (calls++ == fail_at) return hipErrorOutOfMemory;  // *p stays as it was
  *p = std::malloc(1);
  live.insert(*p);
  return hipSuccess;
}
static hipError_t give(void* p) {
  if (!live.erase(p)) ++bad;
  std::free(p);
  return hipSuccess;
}
extern "C" {
hipError_t hipMalloc(void** p, size_t) { return take(p); }
hipError_t hipHostMalloc(void** p, size_t, unsigned int) { return take(p); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipGetLastError() { return hipSuccess; }
}
static bool whole(const wn::MultiState& m, size_t levels, bool cycle64) {
  bool ok = m.r && m.p && m.q && m.zs && m.rp32 && m.zp32 && m.partials && m.sc && m.flags && m.h_sc && m.h_flags &&
            m.lv32.size() == levels && (!cycle64 || m.lv64.size() == levels);
  for (const auto& l : m.lv32)
    for (float* v : l.v) ok = ok && v;
  for (const auto& l : m.lv64)
    for (double* v : l.v) ok = ok && v;
  return ok;
}
#define CHECK(c) if (!(c)) { std::printf("line %d: %s (fail_at %d)\n", __LINE__, #c, fail_at); return 1; }
int main() {
  for (int cycle64 = 0; cycle64 < 2; ++cycle64) {
    const std::vector<int> levels = {300, 60, 6};
    const int total = 11 + 15 * (1 + cycle64);
    for (int f = 0; f < total; ++f) {
      wn::MultiState m;
      calls = 0;
      fail_at = f;
      CHECK(m.ensure(300, 8, levels, cycle64, 4096) == (int)hipErrorOutOfMemory);
      CHECK(live.empty());
      fail_at = -1;
      CHECK(m.ensure(300, 8, levels, cycle64, 4096) == 0);
      CHECK(whole(m, 3, cycle64) && (int)live.size() == total);
      calls = 0;
      CHECK(m.ensure(300, 8, levels, cycle64, 4096) == 0 && calls == 0);  // it fits
      CHECK(m.ensure(200, 8, {200, 60, 6}, cycle64, 100) == 0 && calls == 0);
      CHECK(m.ensure(300, 4, levels, cycle64, 4096) == 0 && calls == total);  // other columns
      calls = 0;
      CHECK(m.ensure(300, 4, {300, 61, 6}, cycle64, 4096) == 0 && calls == total);  // a larger level
      CHECK(m.ensure(300, 4, {300, 61}, cycle64, 4096) == 0 && whole(m, 2, cycle64));
      CHECK(m.ensure(300, 4, {}, 0, 5000) == 0 && whole(m, 0, false));
      m.release();
      CHECK(live.empty() && bad == 0);
    }
  }
  return 0;
}
"""


def test_failed_allocations_leave_nothing_behind(tmp_path):
    if not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"):
        pytest.skip("no HIP headers")
    src, exe = tmp_path / "state.cpp", tmp_path / "state"
    src.write_text(_PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unused-result", "-D__HIP_PLATFORM_AMD__", "-I", _CSRC,
                    "-isystem", "/opt/rocm/include", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
