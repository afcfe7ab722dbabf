// Workspace of the multi-column solver (multi.hip): what it holds, and how it
// grows.  Host code over the HIP runtime's allocation calls alone.
#pragma once
#include <hip/hip_runtime_api.h>
#include <algorithm>
#include <cstddef>
#include <vector>

namespace wn {

enum MsIdx { kMsRho = 0, kMsRhoPrev, kMsBeta, kMsAlpha, kMsGamma, kMsRR, kMsRR0, kMsTol2, kMsCount };

// Per-level column vectors of the multi-column cycle (b, x, tmp, d, res).
template <typename T>
struct MrLevel {
  T* v[5] = {};
};

struct MultiState {
  int nr = 0;
  long long n = 0;
  std::vector<MrLevel<float>> lv32;
  std::vector<MrLevel<double>> lv64;
  std::vector<int> level_n;  // rows the level vectors were sized for
  double *r = nullptr, *p = nullptr, *q = nullptr, *zs = nullptr;  // FP64 n x NR
  float *rp32 = nullptr, *zp32 = nullptr;                           // FP32 n x NR
  double* partials = nullptr;  // NR x max blocks
  int max_blocks = 0;
  double* sc = nullptr;  // per-column scalars: kMs* x NR
  int* flags = nullptr;  // [0] all done, [1] iteration, [2..2+NR) done per column, [2+NR..) iterations per column
  double* h_sc = nullptr;
  int* h_flags = nullptr;
  void release() {
    for (auto& l : lv32)
      for (auto* p_ : l.v) if (p_) (void)hipFree(p_);
    for (auto& l : lv64)
      for (auto* p_ : l.v) if (p_) (void)hipFree(p_);
    lv32.clear();
    lv64.clear();
    for (void* p_ : {(void*)r, (void*)p, (void*)q, (void*)zs, (void*)rp32, (void*)zp32, (void*)partials, (void*)sc,
                     (void*)flags})
      if (p_) (void)hipFree(p_);
    if (h_sc) (void)hipHostFree(h_sc);
    if (h_flags) (void)hipHostFree(h_flags);
    r = p = q = zs = nullptr;
    rp32 = zp32 = nullptr;
    partials = sc = h_sc = nullptr;
    flags = h_flags = nullptr;
    n = 0;
    nr = 0;
    level_n.clear();
  }

  // Room for n rows of nr columns, these level sizes and `blocks` partials per
  // column.  The sizes are recorded when all of it is there: after a failed
  // allocation nothing is held, and the next call starts again.  Returns a HIP
  // error code, 0 for none.
  int ensure(long long n_, int nr_, const std::vector<int>& levels, int need64cycle, int blocks) {
    bool same = n > 0 && n >= n_ && nr == nr_ && max_blocks >= blocks && level_n.size() == levels.size() &&
                lv32.size() == levels.size() && (!need64cycle || lv64.size() == levels.size());
    for (size_t l = 0; same && l < levels.size(); ++l) same = level_n[l] >= levels[l];
    if (same) return 0;
    release();
    const hipError_t e = allocate(n_, nr_, levels, need64cycle, blocks);
    if (e != hipSuccess) {
      release();
      (void)hipGetLastError();  // reported here, not by the next launch
      return static_cast<int>(e);
    }
    n = n_;
    nr = nr_;
    level_n = levels;
    max_blocks = blocks;
    return 0;
  }

 private:
  hipError_t allocate(long long n_, int nr_, const std::vector<int>& levels, int need64cycle, int blocks) {
    const size_t nv = (size_t)n_ * nr_, m = (size_t)nr_;
    hipError_t e = hipSuccess;
    const auto dev = [&](auto*& p_, size_t count) {
      if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&p_), sizeof(*p_) * count);
    };
    const auto host = [&](auto*& p_, size_t count) {
      if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void**>(&p_), sizeof(*p_) * count, 0);
    };
    dev(r, nv);
    dev(p, nv);
    dev(q, nv);
    dev(zs, nv);
    dev(rp32, nv);
    dev(zp32, nv);
    dev(partials, m * (size_t)blocks);
    dev(sc, kMsCount * m);
    dev(flags, 2 + 2 * m);
    host(h_sc, kMsCount * m);
    host(h_flags, 2 + 2 * m);
    lv32.resize(levels.size());
    if (need64cycle) lv64.resize(levels.size());
    for (size_t l = 0; l < levels.size(); ++l) {
      const size_t nl = (size_t)std::max(levels[l], 1) * m;
      for (int k = 0; k < 5; ++k) {
        dev(lv32[l].v[k], nl);
        if (need64cycle) dev(lv64[l].v[k], nl);
      }
    }
    return e;
  }
};

}  // namespace wn
