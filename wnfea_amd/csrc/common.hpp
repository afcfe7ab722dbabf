// Shared helpers of the gfx950 solve-path library: status codes, launch
// helpers, wavefront (64-lane) reductions and the deterministic "last block
// finalises" grid reduction used by every fused dot product.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstddef>

namespace wn {

// Status convention of the C-ABI: 0 ok, <0 argument errors, >0 HIP errors.
enum Status : int {
  kOk = 0,
  kBadArg = -1,
  kBadSize = -2,
  kBadMode = -3,
  kNotReady = -4,
  kBadMesh = -5,
  kNoConverge = -6,
};

#define WN_HIP(expr)                                   \
  do {                                                 \
    hipError_t _e = (expr);                            \
    if (_e != hipSuccess) return static_cast<int>(_e); \
  } while (0)

// Device scalar slots used by the Krylov kernels.  Slots written together by
// one two-dot reduction are consecutive (kScTrue/kScTrueS, kScTrue2/kScTrue2S).
enum ScIdx : int {
  kScRho = 0,
  kScRhoPrev = 1,
  kScBeta = 2,
  kScAlpha = 3,
  kScGamma = 4,
  kScRR = 5,       // ||r||^2 of the (inner) recursion
  kScRR0 = 6,
  kScTrue = 7,     // ||f - K u||^2 (FP64 true residual) ...
  kScTrueS = 8,    // ... and ||S (f - K u)||^2
  kScF2 = 9,       // ||f||^2
  kScInnerN = 10,  // ||r_hat||^2 of the current inner right-hand side
  kScTol2 = 11,    // convergence threshold on kScRR
  kScTrue2 = 15,   // ||f - K u||^2 of the restart refinement loop ...
  kScTrue2S = 16,  // ... and its scaled companion
  kScTmp = 17,
  kScCount = 24,
};

constexpr int kWave = 64;

inline int ceil_div(long a, long b) { return static_cast<int>((a + b - 1) / b); }

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// Block-wide sum (blockDim.x a multiple of 64, at most 1024); result valid in
// every thread.  `smem` holds at least blockDim.x/64 values.
template <typename T>
__device__ __forceinline__ T block_sum(T v, T* smem) {
  v = wave_sum(v);
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  const int nw = blockDim.x / kWave;
  __syncthreads();
  if (lane == 0) smem[wid] = v;
  __syncthreads();
  T t = 0;
  for (int w = 0; w < nw; ++w) t += smem[w];  // fixed order: deterministic
  return t;
}

// Deterministic grid reductions, in two launches.  A reducing kernel stores
// one partial per block (thread 0 of block b writes partials[k*nb + b]); a
// one-block finalise kernel (dot_finalize, blas.hip) then sums the partials
// in index order and applies the solver bookkeeping.  No device-scope fences
// in the reducing kernel: on a multi-XCD GPU each such fence writes back the
// non-coherent L2, which costs far more than one extra small launch.
template <int K>
__device__ __forceinline__ void store_block_partials(const double (&vals)[K], double* partials) {
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < K; ++k) partials[(size_t)k * gridDim.x + blockIdx.x] = vals[k];
  }
}

// Bookkeeping applied by the finalise kernel to the reduced sums.
enum FinMode : int {
  kFinStore = 0,  // out[k] = sum_k
  kFinRho = 1,    // rho: sc[Rho] = sum; sc[Beta] = first ? 0 : rho / rho_prev; sc[RhoPrev] = rho
  kFinGamma = 2,  // gamma: sc[Gamma] = sum; sc[Alpha] = rho / gamma
  kFinRR = 3,     // ||r||^2: sc[RR] = sum; count the iteration; done flag when sc[RR] <= sc[Tol2]
  kFinRhoFlex = 4,  // rho and z.q_old: flexible (Polak-Ribiere) beta = -alpha (z.q_old) / rho_prev
};

// kFinRR carried by another kernel: the next iteration's first kernel launches
// one block more, which finalises ||r||^2 beside that kernel's own work
// instead of in a launch between the two.  The kernel's other blocks must not
// read flags[0], which that block may set: they look at flags[2], the done
// flag as the last update of x and r found it.  part null: nothing to do.
// Saves that launch, 2.5 to 4.7 us of an iteration: box of 19 683 DOF
// 1625 -> 1550 us a solve, 32-cell lattice 18.2 -> 17.75 ms, 144k-row FP64
// solid 8.84 -> 8.72 ms.
struct FinRR {
  const double* part = nullptr;  // nb <= kFinRRMax partials
  int nb = 0;
  double* sc = nullptr;
  int* flags = nullptr;
};
constexpr int kFinRRMax = 4096;

__device__ __forceinline__ void fin_rr(double* sc, int* flags, double rr) {
  sc[kScRR] = rr;
  if (flags) {
    flags[1] += 1;
    if (rr <= sc[kScTol2] || !(rr == rr)) flags[0] = 1;
  }
}

// thread t of `threads` of a finalising block: four independent accumulators
// keep several loads in flight
__device__ __forceinline__ double partial_sum4(const double* __restrict__ p, int nb, int t, int threads) {
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
  int i = t;
  for (; i + 3 * threads < nb; i += 4 * threads) {
    a0 += p[i];
    a1 += p[i + threads];
    a2 += p[i + 2 * threads];
    a3 += p[i + 3 * threads];
  }
  for (; i < nb; i += threads) a0 += p[i];
  return (a0 + a1) + (a2 + a3);
}

// the extra block's work, whatever its size: the sums of a finalise launch's
// 256 threads in the same order, so the same bits.  red: four doubles of LDS.
__device__ __forceinline__ void fin_rr_block(const FinRR& f, double* red) {
  if (f.flags[0]) return;
  const int lane = threadIdx.x & (kWave - 1);
  for (int w = threadIdx.x / kWave; w < 4; w += blockDim.x / kWave) {
    const double s = wave_sum(partial_sum4(f.part, f.nb, w * kWave + lane, 256));
    if (lane == 0) red[w] = s;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  double v = 0.0;
  for (int w = 0; w < 4; ++w) v += red[w];
  fin_rr(f.sc, f.flags, v);
}

}  // namespace wn
