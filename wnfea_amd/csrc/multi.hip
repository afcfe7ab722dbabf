// Multiple right-hand sides: block SpMM, the V-cycle and PCG on NR columns
// at once.
//
// Vectors of NR columns are stored interleaved, X[dof][NR], so the NR values
// a block column gathers are contiguous (one or a few 16-byte loads) and each
// matrix block is read once for all NR columns: the matrix stream, which is
// ~90 % of an SpMV's bytes, is amortised NR ways.  Columns are independent
// CG runs (per-column rho, alpha, beta, ||r||^2 on the device); a column that
// has converged is frozen (alpha = beta = 0) while the others continue, and
// the loop ends when all are done.  Same precision split as the single-column
// solver: FP64 Krylov vectors, SpMM and updates; the V-cycle in FP32 on S K S
// as z = S M(S r).
#include <cmath>
#include "multi_state.hpp"
#include "sell.hpp"
#include "solver.hpp"

namespace wn {

constexpr int kMrBlock = 256;

// Sliced-ELL block SpMM (layout of sell.hpp) on NR interleaved columns.
//
// Bound: L1 and instruction issue.  A block's BC x rows (96 bytes for FP32
// 3x3 and 8 columns) are contiguous, and loads of a line that is still on its
// way stall the L1 pipeline (40 % of the cycles of a kernel whose lanes load
// their block's x rows one after the other), so each line is asked for once:
// a wavefront takes 64 blocks at a time, one per lane, its lanes load the x
// of those blocks as one stream of 16-byte chunks (lane t of load i takes
// chunk 64 i + t; CH chunks per block) into LDS, and every lane reads its own
// block's rows from there.  A row's blocks are split over G >= max(8, L)
// lanes (lane group q takes blocks q, q + G, ...; L divides G), so a
// wavefront works on RW = 64 / G rows of one slice, its addresses advance by
// a constant per step, and no row waits for another wavefront.  The groups'
// sums meet in a reduce-scatter (at each level a lane keeps half of its
// columns), and one more exchange turns the lanes to the outputs' memory
// order: lane n has column n mod NR of row (n / NR) mod RW, so that the
// epilogue's loads (issued before the block loop) and stores of a row are
// contiguous.  Idx: 32-bit offsets into x where they suffice.
// Measured with 8 columns on 212 355 rows (24 blocks of 3x3 per row), FP32
// Chebyshev step / FP64 product / 6x6 level-1 step, us: all columns per lane
// with x from L1 and four wavefronts per slice 72 / 107 / 50; four columns
// per lane with x from L1 and the reduce-scatter 45 / 72 / 27; this kernel
// 44 / 58 / 30 (kernel trace of a solve of 12 load cases).  (Loading a step's x during the one before costs 22 registers
// and gains nothing; one scalar column per lane, three times the loads, takes
// 75 / 80 / 45.)
template <int BR, int BC, typename XT, int NR>
constexpr int spmm_waves() {  // wavefronts per workgroup: at most 48 KB of LDS for x
  return BC * NR * (int)sizeof(XT) > 208 ? 2 : 4;
}

template <int BR, int BC, typename VT, typename XT, int NR, typename Idx, class Op>
__global__ __launch_bounds__(64 * (spmm_waves<BR, BC, XT, NR>())) void sell_spmm_kernel(
    SellView<VT> A, const XT* __restrict__ x, Op op, int gsh, int xcd_remap, const int* flags, int guard) {
  if (guard_skip(flags, guard)) return;
  using AT = typename AccT<VT>::type;
  constexpr int BB = BR * BC, W = spmm_waves<BR, BC, XT, NR>();
  constexpr int V = 16 / (int)sizeof(VT), FULL = BB / V, REM = BB - FULL * V;
  constexpr int XV = 16 / (int)sizeof(XT), CH = BC * NR / XV;  // x values per chunk, chunks per block
  static_assert(NR % XV == 0 && (NR & (NR - 1)) == 0, "column split");
  using Chunk = XT __attribute__((ext_vector_type(XV)));
  __shared__ Chunk xs[W][64 * CH];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lsh = __ffs(A.lanes) - 1, rsh = 6 - lsh;  // log2 of L and of the rows per slice
  const int G = 1 << gsh, RW = 64 >> gsh;             // lsh <= gsh: a wavefront stays in one slice
  // this wavefront's row positions pos0 .. pos0 + RW, below end
  const int end = A.n_slices << rsh;
  const int pos0 = (slice_of_block((end + W * RW - 1) / (W * RW), xcd_remap) * W + wave) * RW;
  double dot = 0.0;
  if (pos0 < end) {
    // this lane's outputs: column ek, rows es, es + RS, ... of block row erow
    const int ek = lane % NR, el = (lane / NR) & (RW - 1), es = lane / NR >> (6 - gsh), RS = G / NR;
    const int erow = A.rinfo[pos0 + el].x;
    const long long eo = (long long)(erow < 0 ? 0 : erow) * BR * NR + ek;
    typename Op::Pre pre[BR];
    if (erow >= 0) {
#pragma unroll
      for (int r = 0; r < BR; ++r)
        if ((r & (RS - 1)) == es) op.load(eo + r * NR, (long long)erow * BR + r, pre[r]);
    }
    // this lane's blocks: q, q + G, ... of row position pos0 + rl, found in
    // step (q >> lsh) + t (G / L) of the slice at lane r0 + R (q mod L)
    const int rl = lane & (RW - 1), q = lane >> (6 - gsh);
    const int s = pos0 >> rsh, r0 = (pos0 & ((1 << rsh) - 1)) + rl;
    const int len = A.rinfo[pos0 + rl].y;
    const long long base = A.off[s];
    const int n_steps = (int)((A.off[s + 1] - base) >> 6);  // of the slice, L blocks of a row each
    const int steps = (n_steps + (1 << (gsh - lsh)) - 1) >> (gsh - lsh);
    const int sl = r0 + ((q & (A.lanes - 1)) << rsh);
    int step = q >> lsh;
    const int* __restrict__ colp = A.col + base;
    const VT* __restrict__ valp = A.val + base * BB;
    AT acc[BR][NR];
#pragma unroll
    for (int r = 0; r < BR; ++r)
#pragma unroll
      for (int k = 0; k < NR; ++k) acc[r][k] = AT(0);
    // a lane without a block in a step loads its row's first one again, unused
    const auto column = [&](int b, int st) { return load_col(colp + (b < len ? 64 * st + sl : sl)); };
    int b = q, cn = steps > 0 ? column(b, step) : 0;
    for (int t = 0; t < steps; ++t) {
      const bool have = b < len;
      // chunk 64 i + lane belongs to block (64 i + lane) / CH of the wavefront
      Chunk xc[CH];
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int ch = 64 * i + lane;
        const Idx c = (Idx)__shfl(cn, ch / CH, 64);
        xc[i] = *reinterpret_cast<const Chunk*>(reinterpret_cast<const char*>(x) +
                                                (c * (Idx)(BC * NR * sizeof(XT)) + (Idx)(ch % CH * 16)));
      }
      VT v[BB];
      {
        const unsigned st = have ? step : 0;
        const VT* __restrict__ region = valp;
        const unsigned o = st * (64 * BB);
#pragma unroll
        for (int g = 0; g < FULL; ++g) load_vec<VT, V>(region + (o + g * 64 * V + sl * V), v + g * V);
        if constexpr (REM > 0) load_vec<VT, REM>(region + (o + FULL * 64 * V + sl * REM), v + FULL * V);
      }
      b += G;
      step += 1 << (gsh - lsh);
      if (t + 1 < steps) cn = column(b, step);  // one step ahead of its x
#pragma unroll
      for (int i = 0; i < CH; ++i) xs[wave][64 * i + lane] = xc[i];
      // only this wavefront's part of xs is read: LDS operations of a
      // wavefront complete in order
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (have) {
#pragma unroll
        for (int k = 0; k < BC; ++k) {
          XT xv[NR];
#pragma unroll
          for (int i = 0; i < NR / XV; ++i) {
            const Chunk c = xs[wave][lane * CH + k * (NR / XV) + i];
#pragma unroll
            for (int e = 0; e < XV; ++e) xv[i * XV + e] = c[e];
          }
#pragma unroll
          for (int r = 0; r < BR; ++r)
#pragma unroll
            for (int c = 0; c < NR; ++c) acc[r][c] = fma(AT(v[r * BC + k]), AT(xv[c]), acc[r][c]);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    // reduce-scatter over the low bits of q (bit m keeps the half
    // NR >> (m + 1) of its columns), plain sums over the rest
#pragma unroll
    for (int r = 0; r < BR; ++r) {
#pragma unroll
      for (int m = 0; (NR >> m) > 1; ++m) {
        const int half = NR >> (m + 1);
        const bool hi = (q >> m) & 1;
#pragma unroll
        for (int c = 0; c < half; ++c) {
          const AT give = hi ? acc[r][c] : acc[r][c + half], keep = hi ? acc[r][c + half] : acc[r][c];
          acc[r][c] = keep + __shfl_xor(give, RW << m, 64);
        }
      }
      for (int off = NR; off < G; off *= 2) acc[r][0] += __shfl_xor(acc[r][0], off * RW, 64);
    }
    // to the outputs' order: column ek is in the groups whose low bits, read
    // backwards, are ek
    int qe = 0;
#pragma unroll
    for (int m = 0; (NR >> m) > 1; ++m) qe |= ((ek / (NR >> (m + 1))) & 1) << m;
    const int src = el + RW * (qe + NR * es);
#pragma unroll
    for (int r = 0; r < BR; ++r) {
      const AT a = __shfl(acc[r][0], src, 64);
      if (erow >= 0 && (r & (RS - 1)) == es) op.out(eo + r * NR, a, dot, pre[r]);
    }
  }
  if constexpr (Op::kDots > 0) {
#pragma unroll
    for (int off = 32; off >= NR; off >>= 1) dot += __shfl_xor(dot, off, 64);
    __shared__ double sm[W][NR];
    if (lane < NR) sm[wave][lane] = dot;
    __syncthreads();
    if (threadIdx.x < NR) {
      double t = 0.0;
#pragma unroll
      for (int w = 0; w < W; ++w) t += sm[w][threadIdx.x];
      op.partials[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = t;
    }
  }
}

// ---------------------------------------------------------------- epilogues
// One output: o = (i BR + r) NR + k of the interleaved columns, i_r = i BR + r.
template <typename YT, typename AT>
struct MOpStore {  // y = A x, or y += A x with add
  static constexpr int kDots = 0;
  YT* y;
  int add;
  double* partials = nullptr;
  struct Pre { AT y; };
  __device__ __forceinline__ void load(long long o, long long, Pre& p) const { p.y = add ? AT(y[o]) : AT(0); }
  __device__ __forceinline__ void out(long long o, AT a, double&, const Pre& p) const { y[o] = YT(p.y + a); }
};

// y = R x and the coarse level's first Chebyshev iterate x1 = d1 = c2 dinv y
// (the expression of the separate first-step kernel).
template <typename T, typename AT>
struct MOpRestrictFirst {
  static constexpr int kDots = 0;
  T* y;
  const T* dinv;
  T* x1;
  T* d1;
  T c2;
  double* partials = nullptr;
  struct Pre { T dinv; };
  __device__ __forceinline__ void load(long long, long long i_r, Pre& p) const { p.dinv = dinv[i_r]; }
  __device__ __forceinline__ void out(long long o, AT a, double&, const Pre& p) const {
    const T b = T(a), v = c2 * p.dinv * b;
    y[o] = b;
    d1[o] = v;
    x1[o] = v;
  }
};

template <typename T>
struct MOpSpmvDot {  // q = A p, gamma_k = p_k . q_k
  static constexpr int kDots = 1;
  T* y;
  const T* p;
  double* partials;
  struct Pre { T p; };
  __device__ __forceinline__ void load(long long o, long long, Pre& pr) const { pr.p = p[o]; }
  __device__ __forceinline__ void out(long long o, T a, double& d, const Pre& pr) const {
    y[o] = a;
    d += double(pr.p) * double(a);
  }
};

template <typename T>
struct MOpCheb {  // res = b - A x_in; d = c1 d + c2 dinv res; x_out = x_in + d
  static constexpr int kDots = 0;
  const T* b;
  const T* dinv;  // per DOF
  const T* x_in;
  T* x_out;
  T* d;
  T c1, c2;
  double* partials = nullptr;
  struct Pre { T b, dinv, x, d; };
  __device__ __forceinline__ void load(long long o, long long i_r, Pre& p) const {
    p.b = b[o];
    p.dinv = dinv[i_r];
    p.x = x_in[o];
    p.d = d[o];
  }
  __device__ __forceinline__ void out(long long o, T a, double&, const Pre& p) const {
    const T dn = c1 * p.d + c2 * p.dinv * (p.b - a);
    d[o] = dn;
    x_out[o] = p.x + dn;
  }
};

template <typename T>
struct MOpDefect {
  static constexpr int kDots = 0;
  const T* b;
  T* res;
  double* partials = nullptr;
  struct Pre { T b; };
  __device__ __forceinline__ void load(long long o, long long, Pre& p) const { p.b = b[o]; }
  __device__ __forceinline__ void out(long long o, T a, double&, const Pre& p) const { res[o] = p.b - a; }
};

// ---------------------------------------------------------------- launch
// log2 of the lanes per row, at least those of the layout: 8, or 16 where the
// matrix would leave the chip with few wavefronts (under about four per SIMD)
// and its rows hold two blocks per lane (8 columns; 12 285 rows of 23 3x3
// blocks: 4.75 -> 4.57 ms per 8 load cases; 4 441 rows of 60 6x6 blocks, the
// level below 70 785 rows: 36.4 -> 35.5 ms per 12; the 70 785 rows
// themselves: 36.4 -> 38.8 ms, so they keep 8).
static int spmm_group_shift(const SellMatrix& A) {
  int g = 3;
  if (((long long)A.n_rows << g) < 64LL * 4096 && A.nnzb >= 16LL * A.n_rows) ++g;
  while ((1 << g) < A.lanes) ++g;
  return g;
}

// workgroups of the SpMM (each writes one partial per column of a fused dot);
// xs: bytes per value of x
static int spmm_grid(const SellMatrix& A, int nr, int xs, int xcd) {
  const int waves = A.bc * nr * xs > 208 ? 2 : 4;  // spmm_waves
  const int rows = waves * (64 >> spmm_group_shift(A));
  const int n = ceil_div((long)A.n_slices * (64 / A.lanes), rows);
  return xcd ? 8 * ceil_div(n, 8) : n;
}

template <int BR, int BC, typename VT, typename XT, int NR, class Op>
static int launch_spmm(const SellMatrix& A, const XT* x, const Op& op, const SpmvTune& t, hipStream_t s) {
  const SellView<VT> v = A.view<VT>();
  if (A.n_slices == 0) return kOk;
  const int xcd = t.xcd_for<VT>(), g = spmm_group_shift(A);
  const dim3 grid(spmm_grid(A, NR, sizeof(XT), xcd)), block(64 * spmm_waves<BR, BC, XT, NR>());
  if ((long long)A.n_cols * BC * NR * (long long)sizeof(XT) < (1LL << 32))
    hipLaunchKernelGGL((sell_spmm_kernel<BR, BC, VT, XT, NR, unsigned, Op>), grid, block, 0, s, v, x, op, g, xcd,
                       t.flags, t.guard);
  else
    hipLaunchKernelGGL((sell_spmm_kernel<BR, BC, VT, XT, NR, size_t, Op>), grid, block, 0, s, v, x, op, g, xcd,
                       t.flags, t.guard);
  return static_cast<int>(hipGetLastError());
}

#define WN_MR_DISPATCH(A, CALL)                      \
  if ((A).br == 3 && (A).bc == 3) CALL(3, 3)         \
  else if ((A).br == 6 && (A).bc == 6) CALL(6, 6)    \
  else if ((A).br == 3 && (A).bc == 6) CALL(3, 6)    \
  else if ((A).br == 6 && (A).bc == 3) CALL(6, 3)    \
  else return kBadArg;

template <typename VT, typename T, int NR>
static int spmm_store(const SellMatrix& A, const T* x, T* y, int add, const SpmvTune& t, hipStream_t s) {
  using AT = typename AccT<VT>::type;
#define CALL(R, C)                                            \
  {                                                           \
    MOpStore<T, AT> op{y, add};                        \
    return launch_spmm<R, C, VT, T, NR>(A, x, op, t, s);      \
  }
  WN_MR_DISPATCH(A, CALL);
#undef CALL
}

template <typename VT, typename T, int NR>
static int spmm_restrict_first(const SellMatrix& A, const T* x, T* y, const T* dinv, T* x1, T* d1, double c2,
                               const SpmvTune& t, hipStream_t s) {
  using AT = typename AccT<VT>::type;
#define CALL(R, C)                                              \
  {                                                             \
    MOpRestrictFirst<T, AT> op{y, dinv, x1, d1, T(c2)};         \
    return launch_spmm<R, C, VT, T, NR>(A, x, op, t, s);        \
  }
  WN_MR_DISPATCH(A, CALL);  // 3-row blocks: a coarse space of the translations alone
#undef CALL
}

template <typename VT, typename T, int NR>
static int spmm_cheb(const SellMatrix& A, const T* x_in, T* x_out, const T* b, const T* dinv, T* d, double c1,
                     double c2, const SpmvTune& t, hipStream_t s) {
#define CALL(R, C)                                                     \
  {                                                                    \
    MOpCheb<T> op{b, dinv, x_in, x_out, d, T(c1), T(c2)};       \
    return launch_spmm<R, C, VT, T, NR>(A, x_in, op, t, s);            \
  }
  if (A.br == 3 && A.bc == 3) CALL(3, 3) else if (A.br == 6 && A.bc == 6) CALL(6, 6) else return kBadArg;
#undef CALL
}

template <typename VT, typename T, int NR>
static int spmm_defect(const SellMatrix& A, const T* x, const T* b, T* res, const SpmvTune& t, hipStream_t s) {
#define CALL(R, C)                                            \
  {                                                           \
    MOpDefect<T> op{b, res};                           \
    return launch_spmm<R, C, VT, T, NR>(A, x, op, t, s);      \
  }
  if (A.br == 3 && A.bc == 3) CALL(3, 3) else if (A.br == 6 && A.bc == 6) CALL(6, 6) else return kBadArg;
#undef CALL
}

// ---------------------------------------------------------------- multi-column vector kernels
template <typename T, int NR>
__global__ void mr_cheb_first_kernel(long long n, const T* __restrict__ b, const T* __restrict__ dinv,
                                     T* __restrict__ d, T* __restrict__ x, T c2, const int* skip) {
  if (skip && *skip) return;
  const long long total = n * NR;
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < total;
       t += (long long)gridDim.x * blockDim.x) {
    const T v = c2 * dinv[t / NR] * b[t];
    d[t] = v;
    x[t] = v;
  }
}

// X[i][k] = sum_j inv[i][j] B[j][k] on the coarsest level, products and sums
// in FP64 (v_mfma_f64_16x16x4f64: lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16], result r of lane l is D[4 r + l / 16][l % 16]).  A
// workgroup owns 16 rows; its 16 wavefronts take every 16th run of 32 columns
// of the inverse, each lane twice four consecutive entries of its row in one
// load, and meet in LDS in wavefront order.  Bound by the inverse's bytes, and
// on a small level by the chain of loads.  FP32 inverse, us, 8 columns: 256
// threads per row and 8 FP64 reductions 21.1 at 2 244 rows, 172 at 8 622, 265
// at 10 740; runs of 16 columns in single loads 175 and 229 at the last two;
// here 10.2, 89 and 131.  4 columns: 14.0, 116 and 176; 15.1 and 164 at the
// first two; here 9.7, 83 and 124.  Runs of 64 columns, or 8 wavefronts (which
// fit the chip in one round up to 16 384 rows), are up to 8 % slower.
typedef double mr_d4 __attribute__((ext_vector_type(4)));
constexpr int kMrCoarseWaves = 16;

template <typename T, int NR>
__global__ __launch_bounds__(64 * kMrCoarseWaves) void mr_coarse_kernel(int n, const T* __restrict__ inv,
                                                                        const T* __restrict__ b, T* __restrict__ x,
                                                                        const int* skip) {
  if (skip && *skip) return;
  constexpr int W = kMrCoarseWaves, U = 2, RUN = 16 * U;  // RUN: columns a wavefront takes at a time
  using V4 = T __attribute__((ext_vector_type(4), aligned(sizeof(T))));  // rows start at any multiple of T
  __shared__ double red[W][16][NR];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int i = blockIdx.x * 16 + lr;
  const T* __restrict__ row = inv + (size_t)min(i, n - 1) * n;
  const T* __restrict__ col = b + (lr < NR ? lr : 0);
  mr_d4 acc = {0.0, 0.0, 0.0, 0.0};
  int k0 = RUN * wave;
  for (; k0 + RUN <= n; k0 += RUN * W) {
    const int k = k0 + 4 * lk;
    V4 av[U];
    T bv[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) av[u] = *reinterpret_cast<const V4*>(row + k + 16 * u);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) bv[u][e] = col[(size_t)(k + 16 * u + e) * NR];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(double(av[u][e]), lr < NR ? double(bv[u][e]) : 0.0, acc, 0, 0, 0);
  }
  // the last, partial run, whose wavefront ends there: clamped, in bounds
  for (; k0 < n; k0 += 16) {
    const int k = k0 + 4 * lk;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = k + e < n;
      const int kk = min(k + e, n - 1);
      const double av = in ? double(row[kk]) : 0.0, bv = in && lr < NR ? double(col[(size_t)kk * NR]) : 0.0;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (lr < NR) red[wave][4 * r + lk][lr] = acc[r];
  __syncthreads();
  for (int t = threadIdx.x; t < 16 * NR; t += blockDim.x) {
    const int r = t / NR, k = t % NR, o = blockIdx.x * 16 + r;
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < W; ++w) v += red[w][r][k];
    if (o < n) x[(size_t)o * NR + k] = T(v);
  }
}

static int mr_grid(long long n) {
  long long g = (n + kMrBlock - 1) / kMrBlock;
  if (g > 2048) g = 2048;
  return static_cast<int>(g < 1 ? 1 : g);
}

static void multi_free(void* p) {
  auto* m = static_cast<MultiState*>(p);
  m->release();
  delete m;
}

static int multi_ensure(Solver& S, long long n, int nr, const Amg* g, int need64cycle, int n_blocks) {
  if (!S.multi) {
    S.multi = new MultiState();
    S.multi_free = multi_free;
  }
  std::vector<int> level_n;
  if (g)
    for (const auto& l : g->L) level_n.push_back(l->n);
  return static_cast<MultiState*>(S.multi)->ensure(n, nr, level_n, need64cycle, std::max(n_blocks + 8, 4096));
}

template <typename T> static std::vector<MrLevel<T>>& mr_levels(MultiState& M);
template <> std::vector<MrLevel<float>>& mr_levels<float>(MultiState& M) { return M.lv32; }
template <> [[maybe_unused]] std::vector<MrLevel<double>>& mr_levels<double>(MultiState& M) { return M.lv64; }

// The V-cycle of solver.hip on NR columns (same smoother, buffer plan and
// coarse solve).
// first_done: the kernel that wrote b wrote the level's first iterate too.
template <typename T>
static T* mr_first_iterate(int deg, T* x, T* tmp) {
  T* post = (deg % 2 == 0) ? x : tmp;
  return ((deg - 1) % 2 == 0) ? post : (post == x ? tmp : x);
}

template <typename VT, typename VTC, typename T, int NR>
static int vcycle_mr(Amg& g, MultiState& M, int l, const T* b, T* x, const int* skip, hipStream_t s,
                     bool first_done = false) {
  AmgLevel& L = *g.L[l];
  SpmvTune t = g.tune;
  t.flags = skip;
  t.guard = skip ? 1 : 0;
  const long long n = L.n;
  if (l == (int)g.L.size() - 1) {
    const T* inv = coarse_inv<T>(g);
    if (L.n != g.n_coarse || !inv) return kNotReady;
    hipLaunchKernelGGL((mr_coarse_kernel<T, NR>), dim3(std::max(ceil_div(L.n, 16), 1)), dim3(64 * kMrCoarseWaves), 0, s,
                       L.n, inv, b, x, skip);
    return static_cast<int>(hipGetLastError());
  }
  MrLevel<T>& V = mr_levels<T>(M)[l];
  T* tmp = V.v[2];
  T* d = V.v[3];
  T* res = V.v[4];
  const T* dinv = level_dinv<T>(L);
  if (!dinv || !L.has_PR) return kNotReady;
  const int deg = std::max(1, std::min(L.degree, 16));
  const ChebCoef c = cheb_coefs(L.lmax, L.ratio, deg);
  const SellMatrix& A = *L.A;
  int r;
  T* cur = mr_first_iterate(deg, x, tmp);
  T* oth = (cur == x) ? tmp : x;
  if (!first_done) {
    hipLaunchKernelGGL((mr_cheb_first_kernel<T, NR>), dim3(mr_grid(n * NR)), dim3(kMrBlock), 0, s, n, b, dinv, d, cur,
                       T(c.c2[0]), skip);
    if ((r = static_cast<int>(hipGetLastError()))) return r;
  }
  for (int k = 1; k < deg; ++k) {
    if ((r = spmm_cheb<VT, T, NR>(A, cur, oth, b, dinv, d, c.c1[k], c.c2[k], t, s))) return r;
    std::swap(cur, oth);
  }
  if ((r = spmm_defect<VT, T, NR>(A, cur, b, res, t, s))) return r;
  MrLevel<T>& N = mr_levels<T>(M)[l + 1];
  AmgLevel& NL = *g.L[l + 1];
  const T* dinv_n = level_dinv<T>(NL);
  const bool fuse_first = l + 1 < (int)g.L.size() - 1 && dinv_n;  // a smoothed level below
  if (fuse_first) {
    const int deg_n = std::max(1, std::min(NL.degree, 16));
    r = spmm_restrict_first<VT, T, NR>(L.R, res, N.v[0], dinv_n, mr_first_iterate(deg_n, N.v[1], N.v[2]), N.v[3],
                                       cheb_coefs(NL.lmax, NL.ratio, deg_n).c2[0], t, s);
  } else {
    r = spmm_store<VT, T, NR>(L.R, res, N.v[0], 0, t, s);
  }
  if (r) return r;
  if ((r = vcycle_mr<VTC, VTC, T, NR>(g, M, l + 1, N.v[0], N.v[1], skip, s, fuse_first))) return r;
  if ((r = spmm_store<VT, T, NR>(L.P, N.v[1], cur, 1, t, s))) return r;
  oth = (cur == x) ? tmp : x;
  for (int k = 0; k < deg; ++k) {
    if ((r = spmm_cheb<VT, T, NR>(A, cur, oth, b, dinv, d, c.c1[k], c.c2[k], t, s))) return r;
    std::swap(cur, oth);
  }
  return kOk;
}

// ---------------------------------------------------------------- PCG on NR columns
// The vector kernels walk the flat n*NR arrays (fully coalesced); with a
// grid stride that is a multiple of NR every thread stays on one column
// k = t mod NR, and the per-column sums meet in a shuffle over the lanes of
// equal k, then across the waves of the block (fixed order).
template <int NR>
__device__ __forceinline__ void store_column_partials(double v, double* partials) {
  static_assert(NR <= 64 && (NR & (NR - 1)) == 0, "NR must be a power of two <= 64");
#pragma unroll
  for (int off = 32; off >= NR; off >>= 1) v += __shfl_xor(v, off, 64);
  __shared__ double sm[kMrBlock / 64][NR];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane < NR) sm[wid][lane] = v;
  __syncthreads();
  if (threadIdx.x < NR) {
    double t = 0.0;
    for (int w = 0; w < kMrBlock / 64; ++w) t += sm[w][threadIdx.x];
    partials[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = t;
  }
}

// partial dots of r_k . (S z_k) (z in ZT, S per DOF)
template <typename ZT, int NR>
__global__ __launch_bounds__(kMrBlock) void mr_rho_kernel(long long n, const double* __restrict__ r,
                                                          const ZT* __restrict__ z, const double* __restrict__ scale,
                                                          double* partials, const int* skip) {
  if (skip && skip[0]) return;
  double acc = 0.0;
  const long long total = n * NR;
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < total;
       t += (long long)gridDim.x * blockDim.x)
    acc += r[t] * double(z[t]) * (scale ? scale[t / NR] : 1.0);
  store_column_partials<NR>(acc, partials);
}

// p_k = S z_k + beta_k p_k (beta 0 on the first iteration or for a done column)
template <typename ZT, int NR>
__global__ void mr_update_p_kernel(long long n, const ZT* __restrict__ z, const double* __restrict__ scale,
                                   double* __restrict__ p, const double* __restrict__ sc, const int* flags) {
  if (flags[0]) return;
  const bool first = flags[1] == 0;
  double beta[NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) beta[k] = first ? 0.0 : sc[kMsBeta * NR + k];
  const long long total = n * NR;
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < total;
       t += (long long)gridDim.x * blockDim.x) {
    const long long i = t / NR;
    const int k = (int)(t - i * NR);
    const double zi = (scale ? scale[i] : 1.0) * double(z[t]);
    p[t] = first ? zi : zi + beta[k] * p[t];
  }
}

// x_k += alpha_k p_k; r_k -= alpha_k q_k; partial ||r_k||^2; rp = S r (FP32)
// and, with fx1, the next cycle's first Chebyshev iterate fx1 = fd1 = fc2 dinv rp
template <int NR>
__global__ __launch_bounds__(kMrBlock) void mr_update_xr_kernel(long long n, double* __restrict__ x,
                                                                double* __restrict__ r, const double* __restrict__ p,
                                                                const double* __restrict__ q,
                                                                float* __restrict__ rp,
                                                                const double* __restrict__ scale, double* partials,
                                                                const double* __restrict__ sc, const int* flags,
                                                                const float* __restrict__ fdinv,
                                                                float* __restrict__ fx1, float* __restrict__ fd1,
                                                                float fc2) {
  if (flags[0]) return;
  const double alpha = sc[kMsAlpha * NR + (threadIdx.x & (NR - 1))];
  double acc = 0.0;
  const long long total = n * NR;
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < total;
       t += (long long)gridDim.x * blockDim.x) {
    x[t] += alpha * p[t];
    const double ri = r[t] - alpha * q[t];
    r[t] = ri;
    if (rp) {
      const float v = float((scale ? scale[t / NR] : 1.0) * ri);
      rp[t] = v;
      if (fx1) {
        const float f = fc2 * fdinv[t / NR] * v;
        fd1[t] = f;
        fx1[t] = f;
      }
    }
    acc += ri * ri;
  }
  store_column_partials<NR>(acc, partials);
}

enum MrFin { kMrRho = 0, kMrGamma = 1, kMrRR = 2, kMrStart = 3 };

// One block: column sums of the partials in a fixed order, then the per-column
// scalar updates of the CG recurrences.
template <int NR>
__global__ __launch_bounds__(1024) void mr_finalize_kernel(const double* __restrict__ partials, int nb, int mode,
                                                           double* sc, int* flags, double rtol2) {
  if (mode != kMrStart && flags[0]) return;
  // wavefront w: column w mod NR, every (16 / NR)-th run of 64 partials; the
  // columns' loads run side by side, eight in flight per lane (one column
  // after the other was eight serial memory latencies: 9.9 us, here 4.6 us)
  constexpr int S = 16 / NR, U = 8;
  __shared__ double red[NR][S];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  {
    const double* p = partials + (size_t)(wid % NR) * nb;
    double a = 0.0;
    for (int i0 = (wid / NR) * 64 + lane; i0 < nb; i0 += 64 * S * U) {
      double v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + 64 * S * u;
        v[u] = i < nb ? p[i] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) a += v[u];
    }
    a = wave_sum(a);
    if (lane == 0) red[wid % NR][wid / NR] = a;
  }
  __syncthreads();
  int* done = flags + 2;
  int* iters = flags + 2 + NR;
  const int k = threadIdx.x;
  if (k < NR) {
  double v = 0.0;
  for (int w = 0; w < S; ++w) v += red[k][w];
  switch (mode) {
    case kMrStart:  // v = ||b_k||^2
      sc[kMsRR * NR + k] = v;
      sc[kMsRR0 * NR + k] = v;
      sc[kMsTol2 * NR + k] = rtol2 * v;
      done[k] = (v == 0.0) ? 1 : 0;
      iters[k] = 0;
      break;
    case kMrRho: {
      const double prev = sc[kMsRhoPrev * NR + k];
      sc[kMsRho * NR + k] = v;
      sc[kMsBeta * NR + k] = (done[k] || flags[1] == 0 || prev == 0.0) ? 0.0 : v / prev;
      sc[kMsRhoPrev * NR + k] = v;
      break;
    }
    case kMrGamma:
      sc[kMsGamma * NR + k] = v;
      sc[kMsAlpha * NR + k] = (done[k] || v == 0.0) ? 0.0 : sc[kMsRho * NR + k] / v;
      break;
    case kMrRR:
      if (!done[k]) {
        sc[kMsRR * NR + k] = v;
        iters[k] += 1;
        if (v <= sc[kMsTol2 * NR + k] || !(v == v)) done[k] = 1;
      }
      break;
  }
  }
  __syncthreads();
  if ((mode == kMrRR || mode == kMrStart) && k == 0) {
    int all = 1;
    for (int c = 0; c < NR; ++c) all &= done[c];
    flags[1] = (mode == kMrRR) ? flags[1] + 1 : 0;
    flags[0] = all;
  }
}

template <int NR>
static int mr_fin(MultiState& M, int nb, int mode, double rtol2, hipStream_t s) {
  hipLaunchKernelGGL((mr_finalize_kernel<NR>), dim3(1), dim3(1024), 0, s, M.partials, nb, mode, M.sc, M.flags, rtol2);
  return static_cast<int>(hipGetLastError());
}

// ||b_k||^2 partials and r = b, x = 0, rp = S r (FP32)
template <int NR>
__global__ __launch_bounds__(kMrBlock) void mr_start_kernel(long long n, const double* __restrict__ b,
                                                            double* __restrict__ x, double* __restrict__ r,
                                                            float* __restrict__ rp, const double* __restrict__ scale,
                                                            double* partials) {
  double acc = 0.0;
  const long long total = n * NR;
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < total;
       t += (long long)gridDim.x * blockDim.x) {
    const double bi = b[t];
    x[t] = 0.0;
    r[t] = bi;
    if (rp) rp[t] = float((scale ? scale[t / NR] : 1.0) * bi);
    acc += bi * bi;
  }
  store_column_partials<NR>(acc, partials);
}

// q = A p with gamma partials (FP64)
template <int NR>
static int mr_spmm_dot(const SellMatrix& A, const double* p, double* q, double* partials, const SpmvTune& t,
                       hipStream_t s) {
#define CALL(R, C)                                                  \
  {                                                                 \
    MOpSpmvDot<double> op{q, p, partials};                   \
    return launch_spmm<R, C, double, double, NR>(A, p, op, t, s);   \
  }
  if (A.br == 3 && A.bc == 3) CALL(3, 3) else if (A.br == 6 && A.bc == 6) CALL(6, 6) else return kBadArg;
#undef CALL
}

// PCG on NR columns of A X = B from X = 0; preconditioner: AMG V-cycle in
// FP32 (vt 1) or FP64 (vt 0) on S A S, z = S M(S r).  B, X: FP64 [n][NR].
template <int NR>
static int pcg_multi_run(Solver& S, const SellMatrix& A, Amg* g, int vt, const double* scale, const double* B,
                         double* X, double rtol, int max_iter, int check_every, const SpmvTune& tune0, hipStream_t s,
                         int* iters, double* rel) {
  const long long n = (long long)A.n_rows * A.br;
  int r;
  if ((r = multi_ensure(S, n, NR, g, vt == 0, spmm_grid(A, NR, 8, 1)))) return r;
  MultiState& M = *static_cast<MultiState*>(S.multi);
  SpmvTune t = tune0;
  t.flags = M.flags;
  t.guard = 1;
  if (check_every <= 0) check_every = 8;
  const int gv = mr_grid(n * NR);
  hipLaunchKernelGGL((mr_start_kernel<NR>), dim3(gv), dim3(kMrBlock), 0, s, n, B, X, M.r, M.rp32, scale, M.partials);
  if ((r = static_cast<int>(hipGetLastError()))) return r;
  if ((r = mr_fin<NR>(M, gv, kMrStart, rtol * rtol, s))) return r;
  const int gs = spmm_grid(A, NR, 8, t.xcd_for<double>());
  // each cycle's first iterate on the finest level comes from the kernel that
  // writes the cycle's input: the x, r update, and one launch here
  const AmgLevel& L0 = *g->L[0];
  const bool first = g->L.size() > 1 && L0.dinv32;
  const int deg0 = std::max(1, std::min(L0.degree, 16));
  const float c20 = (float)cheb_coefs(L0.lmax, L0.ratio, deg0).c2[0];
  float* d0 = first ? M.lv32[0].v[3] : nullptr;
  float* x0 = first ? mr_first_iterate(deg0, M.zp32, M.lv32[0].v[2]) : nullptr;
  if (first) {
    hipLaunchKernelGGL((mr_cheb_first_kernel<float, NR>), dim3(gv), dim3(kMrBlock), 0, s, n, M.rp32, L0.dinv32, d0, x0,
                       c20, nullptr);
    if ((r = static_cast<int>(hipGetLastError()))) return r;
  }
  int done_all = 0;
  // chunks sized from each open column's residual reduction rate, as in the
  // single-column PCG (idle iterations after convergence are costly)
  int chunk = check_every, it_prev = 0;
  double rr_prev[NR] = {};
  for (int it = 0; it < max_iter && !done_all;) {
    chunk = std::max(1, std::min(chunk, max_iter - it));
    const int it0 = it;
    for (int c = 0; c < chunk; ++c, ++it) {
      if ((r = vcycle_mr<float, float, float, NR>(*g, M, 0, M.rp32, M.zp32, M.flags, s, first))) return r;
      hipLaunchKernelGGL((mr_rho_kernel<float, NR>), dim3(gv), dim3(kMrBlock), 0, s, n, M.r, M.zp32, scale,
                         M.partials, M.flags);
      if ((r = static_cast<int>(hipGetLastError()))) return r;
      if ((r = mr_fin<NR>(M, gv, kMrRho, 0.0, s))) return r;
      hipLaunchKernelGGL((mr_update_p_kernel<float, NR>), dim3(mr_grid(n * NR)), dim3(kMrBlock), 0, s, n, M.zp32,
                         scale, M.p, M.sc, M.flags);
      if ((r = static_cast<int>(hipGetLastError()))) return r;
      if ((r = mr_spmm_dot<NR>(A, M.p, M.q, M.partials, t, s))) return r;
      if ((r = mr_fin<NR>(M, gs, kMrGamma, 0.0, s))) return r;
      hipLaunchKernelGGL((mr_update_xr_kernel<NR>), dim3(gv), dim3(kMrBlock), 0, s, n, X, M.r, M.p, M.q, M.rp32,
                         scale, M.partials, M.sc, M.flags, L0.dinv32, x0, d0, c20);
      if ((r = static_cast<int>(hipGetLastError()))) return r;
      if ((r = mr_fin<NR>(M, gv, kMrRR, 0.0, s))) return r;
    }
    WN_HIP(hipMemcpyAsync(M.h_flags, M.flags, sizeof(int) * (2 + 2 * NR), hipMemcpyDeviceToHost, s));
    WN_HIP(hipMemcpyAsync(M.h_sc, M.sc, sizeof(double) * kMsCount * NR, hipMemcpyDeviceToHost, s));
    WN_HIP(hipStreamSynchronize(s));
    done_all = M.h_flags[0];
    if (done_all) break;
    double need_max = 0.0;
    bool known = true;
    for (int k = 0; k < NR; ++k) {
      if (M.h_flags[2 + k]) continue;
      const double rr = M.h_sc[kMsRR * NR + k], tol2 = M.h_sc[kMsTol2 * NR + k];
      const double prev = it_prev == 0 ? M.h_sc[kMsRR0 * NR + k] : rr_prev[k];
      rr_prev[k] = rr;
      if (!(rr > 0.0 && rr < prev && tol2 > 0.0 && tol2 < rr)) {
        known = false;
        continue;
      }
      need_max = std::max(need_max, std::log(tol2 / rr) / (std::log(rr / prev) / (it - it0)));
    }
    it_prev = it;
    chunk = (known && need_max < check_every) ? std::max(1, (int)need_max) : check_every;
  }
  WN_HIP(hipMemcpyAsync(M.h_sc, M.sc, sizeof(double) * kMsCount * NR, hipMemcpyDeviceToHost, s));
  WN_HIP(hipMemcpyAsync(M.h_flags, M.flags, sizeof(int) * (2 + 2 * NR), hipMemcpyDeviceToHost, s));
  WN_HIP(hipStreamSynchronize(s));
  for (int k = 0; k < NR; ++k) {
    if (iters) iters[k] = M.h_flags[2 + NR + k];
    const double rr0 = M.h_sc[kMsRR0 * NR + k];
    if (rel) rel[k] = rr0 > 0.0 ? std::sqrt(M.h_sc[kMsRR * NR + k] / rr0) : 0.0;
  }
  return kOk;
}

int pcg_multi(Solver& S, const SellMatrix& A, Amg* g, int vt, const double* scale, int nr, const double* B, double* X,
              double rtol, int max_iter, int check_every, const SpmvTune& t, hipStream_t s, int* iters, double* rel) {
  if (!g || vt != 1 || (g->store & 2) == 0) return kBadMode;
  switch (nr) {
    case 4: return pcg_multi_run<4>(S, A, g, vt, scale, B, X, rtol, max_iter, check_every, t, s, iters, rel);
    case 8: return pcg_multi_run<8>(S, A, g, vt, scale, B, X, rtol, max_iter, check_every, t, s, iters, rel);
    default: return kBadArg;
  }
}

// Y = A X on nr interleaved columns (prec 0 FP64, 1 FP32)
int bsr_spmm(const SellMatrix& A, int prec, int nr, const void* X, void* Y, const SpmvTune& t, hipStream_t s) {
  SpmvTune tt = t;
  tt.flags = nullptr;
  tt.guard = 0;
  if (prec == 0) {
    if (!A.d_v64) return kNotReady;
    if (nr == 4) return spmm_store<double, double, 4>(A, (const double*)X, (double*)Y, 0, tt, s);
    if (nr == 8) return spmm_store<double, double, 8>(A, (const double*)X, (double*)Y, 0, tt, s);
    return kBadArg;
  }
  if (prec == 1) {
    if (!A.d_v32) return kNotReady;
    if (nr == 4) return spmm_store<float, float, 4>(A, (const float*)X, (float*)Y, 0, tt, s);
    if (nr == 8) return spmm_store<float, float, 8>(A, (const float*)X, (float*)Y, 0, tt, s);
    return kBadArg;
  }
  return kBadMode;
}

}  // namespace wn
