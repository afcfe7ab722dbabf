// Assembly of the 3x3-block C3D10 matrix of an affine mesh without element
// matrices, in the sliced-ELL layout's own order.
//
// The shape gradients of an affine element are linear in the barycentric
// coordinates, so with g_k = grad L_k (k = 0..3) node a's gradient at vertex v
// is (4 delta_av - 1) g_a for a corner and 4 (delta_qv g_p + delta_pv g_q) for
// the midside of edge (p, q), and the integral of the product of two linear
// functions is V/20 (1 + delta_vw) over their vertex values.  Hence
//   M_ab = int grad N_a (x) grad N_b = V/20 (g_p (x) (c0 g_s + c1 g_t) + g_q (x) (c2 g_s + c3 g_t))
// with integers c depending on which of p, q, s, t coincide, and the block is
//   K_ab = lambda M + mu M^T + mu tr(M) I
// (B_a^T D B_b summed over the 4-point rule, which is exact here; the element
// stiffness of wnfea/elements/c3d10.py:219-249 and the summation of
// wnfea/solver/solid_solver.py:62-84).
//
// One record of 128 bytes per element (the four gradients, each padded to 32
// bytes with lambda V/20 and mu V/20 in the first two pads) is all a block
// needs of an element, 60 FP64 operations per contribution; element matrices
// are 7 200 bytes per element written and read again.  Off-diagonal blocks
// have one to six contributions and one lane each; diagonal blocks have up to
// a few dozen and sixteen lanes each.  Lanes follow the layout's slots, so
// values are stored as contiguous 1 KB chunks.  117 585 rows, 69 600 elements:
// element matrices and their gather 145 + 440 us, here records 9,
// off-diagonal blocks 187 (ten 16-byte gathers per contribution) and diagonal
// blocks 33 us.  Against blocks in higher precision the error is that of the
// element matrices to about a tenth (9.0e-15 of the norm against 8.0e-15).
#include "sell.hpp"
#include "wn.hpp"

namespace wn {

// Element records (affine_records in element.hip): four gradients of four doubles.
constexpr int kRec = 16;

// corner pair of local node i: (i, i) for a corner, its edge's ends for a midside node
__device__ __forceinline__ int pair_p(int i) { return i < 4 ? i : (0x210210 >> (4 * i - 16)) & 7; }
__device__ __forceinline__ int pair_q(int i) { return i < 4 ? i : (0x333021 >> (4 * i - 16)) & 7; }

struct Grad {
  double x, y, z, pad;
};
__device__ __forceinline__ Grad load_grad(const double* __restrict__ rec, int k) {
  const double2* r = reinterpret_cast<const double2*>(rec) + 2 * k;
  const double2 a = r[0], b = r[1];
  return Grad{a.x, a.y, b.x, b.y};
}

// acc += K_ab of one element.  The block is formed for the smaller of (a, b)
// first and transposed otherwise, with every product and sum of the two
// orders in the same rounding, so that K_ba is K_ab^T bit for bit.
__device__ __forceinline__ void add_block(const double* __restrict__ rec, int a, int b, double (&acc)[9]) {
#pragma clang fp contract(off)
  const bool swap = a > b;
  const int i = swap ? b : a, j = swap ? a : b;
  const int p = pair_p(i), q = pair_q(i), s = pair_p(j), t = pair_q(j);
  double c0, c1, c2, c3;
  if (j < 4) {  // two corners (i < j)
    c0 = -4.0;
    c1 = c2 = c3 = 0.0;
  } else if (i < 4) {  // corner and midside
    c0 = i == t ? 12.0 : -4.0;
    c1 = i == s ? 12.0 : -4.0;
    c2 = c3 = 0.0;
  } else {  // two midsides
    c0 = q == t ? 32.0 : 16.0;
    c1 = q == s ? 32.0 : 16.0;
    c2 = p == t ? 32.0 : 16.0;
    c3 = p == s ? 32.0 : 16.0;
  }
  const Grad gp = load_grad(rec, p), gq = load_grad(rec, q), gs = load_grad(rec, s), gt = load_grad(rec, t);
  const double lam = rec[3], mu = rec[7];
  const double u[3] = {c0 * gs.x + c1 * gt.x, c0 * gs.y + c1 * gt.y, c0 * gs.z + c1 * gt.z};
  const double w[3] = {c2 * gs.x + c3 * gt.x, c2 * gs.y + c3 * gt.y, c2 * gs.z + c3 * gt.z};
  const double A[3] = {gp.x, gp.y, gp.z}, B[3] = {gq.x, gq.y, gq.z};
  double m[3][3];
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) m[r][c] = A[r] * u[c] + B[r] * w[c];
  const double tr = mu * (m[0][0] + m[1][1] + m[2][2]);
  const double l1 = swap ? mu : lam, l2 = swap ? lam : mu;
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double v = l1 * m[r][c] + l2 * m[c][r];
      acc[3 * r + c] += r == c ? v + tr : v;
    }
}

// The Dirichlet rule per scalar entry (solid_solver.py:95-127): a fixed row or
// column DOF zeroes the entry, the diagonal entry of a fixed DOF is 1.
__device__ __forceinline__ double with_supports(double v, unsigned fi, unsigned fj, int r, int c, bool diagonal) {
  return ((fi >> r) & 1u) || ((fj >> c) & 1u) ? (diagonal && r == c ? 1.0 : 0.0) : v;
}

// Off-diagonal blocks: one workgroup per slice, one wavefront per step, one
// lane per slot; contributions in list order (element order).
constexpr int kAsmWaves = 4;

__global__ __launch_bounds__(64 * kAsmWaves) void assemble_affine_kernel(
    SellView<double> A, const int* __restrict__ rstart, const long long* __restrict__ cptr,
    const int* __restrict__ codes, const double* __restrict__ rec, const unsigned char* __restrict__ node_fix,
    double* __restrict__ v64) {
  const int s = slice_of_block(A.n_slices, 1);
  if (s >= A.n_slices) return;
  const int lane = threadIdx.x & 63, rps = 64 / A.lanes, q = lane / rps;
  const int pos = s * rps + lane % rps;
  const int2 ri = A.rinfo[pos];
  const int row = ri.x;
  const unsigned fi = node_fix && row >= 0 ? node_fix[row] : 0u;
  const long long base = A.off[s];
  const int steps = (int)((A.off[s + 1] - base) >> 6);
  for (int j = threadIdx.x >> 6; j < steps; j += kAsmWaves) {
    const int b = j * A.lanes + q;
    if (b >= ri.y) continue;
    const int col = A.col[base + 64LL * j + lane];
    if (col == row) continue;  // diagonal block: assemble_affine_diag_kernel
    const long long k = (long long)rstart[pos] + b;
    double acc[9] = {};
    for (long long i = cptr[k]; i < cptr[k + 1]; ++i) {
      const int code = codes[i], e = code / 100, ab = code - e * 100;
      add_block(rec + (size_t)e * kRec, ab / 10, ab % 10, acc);
    }
    const unsigned fj = node_fix ? node_fix[col] : 0u;
#pragma unroll
    for (int x = 0; x < 9; ++x) acc[x] = with_supports(acc[x], fi, fj, x / 3, x % 3, false);
    double* o = v64 + (base + 64LL * j) * 9;
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<double2*>(o + g * 128 + 2 * lane) = make_double2(acc[2 * g], acc[2 * g + 1]);
    o[4 * 128 + lane] = acc[8];
  }
}

// Diagonal blocks: sixteen lanes per row position, whose partial sums meet in
// a fixed order.
__global__ __launch_bounds__(256) void assemble_affine_diag_kernel(
    SellView<double> A, const int* __restrict__ rstart, const long long* __restrict__ cptr,
    const int* __restrict__ codes, const double* __restrict__ rec, const unsigned char* __restrict__ node_fix,
    double* __restrict__ v64) {
  const int rps = 64 / A.lanes, n_pos = A.n_slices * rps;
  const int pos = blockIdx.x * 16 + (int)(threadIdx.x >> 4), sub = threadIdx.x & 15;
  const int2 ri = pos < n_pos ? A.rinfo[pos] : make_int2(-1, 0);
  const int row = ri.x;
  const long long base = pos < n_pos ? A.off[pos / rps] : 0;
  const int r0 = pos % rps;
  int bd = -1;  // the diagonal block's number in its row
  for (int b = sub; b < ri.y; b += 16)
    if (A.col[base + 64LL * (b / A.lanes) + (b % A.lanes) * rps + r0] == row) bd = b;
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) bd = max(bd, __shfl_xor(bd, off, 64));
  double acc[6] = {};  // 00, 01, 02, 11, 12, 22
  if (bd >= 0) {
    const long long k = (long long)rstart[pos] + bd;
    const long long i1 = cptr[k + 1];
    for (long long i = cptr[k] + sub; i < i1; i += 16) {
      const int code = codes[i], e = code / 100, a = code % 10;
      const double* __restrict__ rc = rec + (size_t)e * kRec;
      const Grad g = load_grad(rc, pair_p(a)), h = load_grad(rc, pair_q(a));
      const double lm = rc[3] + rc[7], mu = rc[7];
      // corner: 12 g g^T; midside: 32 (g g^T + h h^T) + 16 (g h^T + h g^T)
      const double x[3] = {g.x, g.y, g.z}, y[3] = {h.x, h.y, h.z};
      double m[6];
      int n = 0;
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = r; c < 3; ++c, ++n)
          m[n] = a < 4 ? 12.0 * (x[r] * x[c])
                       : 32.0 * (x[r] * x[c] + y[r] * y[c]) + 16.0 * (x[r] * y[c] + y[r] * x[c]);
      const double tr = mu * (m[0] + m[3] + m[5]);
#pragma unroll
      for (n = 0; n < 6; ++n) acc[n] += lm * m[n] + (n == 0 || n == 3 || n == 5 ? tr : 0.0);
    }
  }
#pragma unroll
  for (int n = 0; n < 6; ++n)
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) acc[n] += __shfl_xor(acc[n], off, 64);
  if (bd < 0 || sub >= 9) return;
  const int r = sub / 3, c = sub % 3, lo = min(r, c), hi = max(r, c);
  const int n = lo == 0 ? hi : (lo == 1 ? 2 + hi : 5);
  double v = acc[0];
#pragma unroll
  for (int x = 1; x < 6; ++x) v = x == n ? acc[x] : v;
  const unsigned f = node_fix ? node_fix[row] : 0u;
  const long long slot = base + 64LL * (bd / A.lanes) + (bd % A.lanes) * rps + r0;
  v64[val_index<double>(slot, sub, 9)] = with_supports(v, f, f, r, c, true);
}

int assemble_affine(SellMatrix& A, const long long* cptr, const int* codes, const double* rec,
                    const unsigned char* node_fix, hipStream_t s) {
  if (A.br != 3 || A.bc != 3 || A.n_rows != A.n_cols) return kBadArg;
  int r = A.ensure_values(1, 0);
  if (r) return r;
  if (A.nnzb == 0) return kOk;
  const SellView<double> v = A.view<double>();
  hipLaunchKernelGGL(assemble_affine_kernel, dim3(8 * ceil_div(A.n_slices, 8)), dim3(64 * kAsmWaves), 0, s, v,
                     A.d_rstart, cptr, codes, rec, node_fix, A.d_v64);
  hipLaunchKernelGGL(assemble_affine_diag_kernel, dim3(ceil_div((long)A.n_slices * (64 / A.lanes), 16)), dim3(256), 0,
                     s, v, A.d_rstart, cptr, codes, rec, node_fix, A.d_v64);
  return static_cast<int>(hipGetLastError());
}

// ---------------------------------------------------------------- element matrices
// Deterministic assembly of B x B blocks from element matrices
// Ke[M][npe B][npe B].  Block k = (i, j) sums the entries of its contributions
// in list order (element order, then local pair order), each code =
// e npe^2 + a npe + b addressing Ke[e][B a + r][B b + c]; sym: of the symmetric
// part 0.5 (Ke + Ke^T).
//
// 3x3 blocks: one thread per block in standard order, its nine entries' loads
// in flight together.  Bound by the diagonal blocks' chains of dependent loads
// on small meshes (a code, then its element's entries, up to a few dozen
// times) and by the element matrices' lines on large ones.  The tiles of the
// 6x6 blocks below take such a chain for every entry of a thread, three here:
// curved I-beams of 2 784, 13 920, 52 200 and 104 400 elements 81, 181, 384
// and 794 us in tiles, 27, 100, 334 and 657 here.
// NPE: nodes per element where it is known at compile time, else 0 (npe).
template <int NPE>
__global__ __launch_bounds__(256) void assemble_block3_kernel(
    long long nnzb, int npe_, int sym, const int* __restrict__ rowidx, const int* __restrict__ colidx,
    const long long* __restrict__ cptr, const int* __restrict__ codes, const double* __restrict__ Ke,
    const unsigned char* __restrict__ node_fix, const long long* __restrict__ slot, double* __restrict__ v64,
    double* __restrict__ vstd) {
  const long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (k >= nnzb) return;
  const int npe = NPE ? NPE : npe_, D = 3 * npe, nn = npe * npe;
  double acc[9] = {};
  for (long long q = cptr[k]; q < cptr[k + 1]; ++q) {
    const int code = codes[q], e = code / nn, ab = code - e * nn, a = ab / npe, b = ab - a * npe;
    const double* kp = Ke + (size_t)e * D * D;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        double v = kp[(size_t)(3 * a + r) * D + 3 * b + c];
        if (sym) v = 0.5 * (v + kp[(size_t)(3 * b + c) * D + 3 * a + r]);
        acc[3 * r + c] += v;
      }
  }
  const int i = rowidx[k], j = colidx[k];
  const unsigned fi = node_fix ? node_fix[i] : 0u, fj = node_fix ? node_fix[j] : 0u;
  const long long sl = slot[k];
#pragma unroll
  for (int x = 0; x < 9; ++x) {
    const double v = with_supports(acc[x], fi, fj, x / 3, x % 3, i == j);
    v64[val_index<double>(sl, x, 9)] = v;
    if (vstd) vstd[k * 9 + x] = v;
  }
}

// 6x6 blocks: kTileSteps workgroups per slice take its steps in turn; a step's
// 64 blocks are summed one thread per entry (an element's rows of B are read by
// neighbouring threads) into LDS and stored in the layout's order, contiguous.
// Bound by the element matrices' and the values' bytes; one thread per block
// read every entry from another line and stored 16-byte pieces (104 544 beams:
// 384 us, here 68 us; 240 beams 42 and 19).
constexpr int kTileThreads = 256, kTileSteps = 4;  // workgroups per slice

__global__ __launch_bounds__(kTileThreads) void assemble_tile_kernel(
    SellView<double> A, const int* __restrict__ rstart, int npe, int sym, const long long* __restrict__ cptr,
    const int* __restrict__ codes, const double* __restrict__ Ke, const unsigned char* __restrict__ node_fix,
    double* __restrict__ v64, double* __restrict__ vstd) {
  constexpr int B = 6, BB = B * B, PAD = BB | 1, V = 2;  // V: entries per 16-byte chunk
  static_assert(BB % V == 0, "the layout's chunks hold all of a block");
  __shared__ double tile[64][PAD];
  __shared__ long long s_k[64], s_c0[64], s_c1[64];  // block number (-1: none), its contributions
  __shared__ unsigned s_fix[64];                     // row bits, column bits << 8, diagonal << 16
  const int s = slice_of_block(A.n_slices, 1);
  if (s >= A.n_slices) return;
  const int t = (int)threadIdx.x, rps = 64 / A.lanes;
  const long long base = A.off[s];
  const int steps = (int)((A.off[s + 1] - base) >> 6);
  const int D = npe * B, nn = npe * npe;
  for (int j = blockIdx.y; j < steps; j += kTileSteps) {
    if (t < 64) {
      const int pos = s * rps + t % rps, b = j * A.lanes + t / rps;
      const int2 ri = A.rinfo[pos];
      long long k = -1;
      if (b < ri.y) {
        k = (long long)rstart[pos] + b;
        const int col = A.col[base + 64LL * j + t];
        s_c0[t] = cptr[k];
        s_c1[t] = cptr[k + 1];
        s_fix[t] = (node_fix ? node_fix[ri.x] | (unsigned)node_fix[col] << 8 : 0u) | (unsigned)(col == ri.x) << 16;
      }
      s_k[t] = k;
    }
    __syncthreads();
    for (int it = t; it < 64 * BB; it += kTileThreads) {
      const int l = it / BB, e = it - l * BB, r = e / B, c = e - r * B;
      const long long k = s_k[l];
      if (k < 0) continue;
      double v = 0.0;
      for (long long q = s_c0[l]; q < s_c1[l]; ++q) {
        const int code = codes[q], el = code / nn, ab = code - el * nn, a = ab / npe, b = ab - a * npe;
        const double* kp = Ke + (size_t)el * D * D;
        double x = kp[(size_t)(B * a + r) * D + B * b + c];
        if (sym) x = 0.5 * (x + kp[(size_t)(B * b + c) * D + B * a + r]);
        v += x;
      }
      const unsigned f = s_fix[l];
      v = with_supports(v, f & 255u, (f >> 8) & 255u, r, c, f >> 16);
      tile[l][e] = v;
      if (vstd) vstd[k * BB + e] = v;
    }
    __syncthreads();
    double* o = v64 + (base + 64LL * j) * BB;
    for (int f = t; f < 64 * BB; f += kTileThreads) {
      const int l = f % (64 * V) / V, e = f / (64 * V) * V + f % V;
      if (s_k[l] >= 0) o[f] = tile[l][e];
    }
    __syncthreads();
  }
}

int assemble_elem(SellMatrix& A, int npe, int sym, const int* rowidx, const int* colidx, const long long* cptr,
                  const int* codes, const double* Ke, const unsigned char* node_fix, double* vals_std, hipStream_t s) {
  if (A.br != A.bc || npe <= 0 || npe > 27) return kBadArg;
  int r = A.ensure_values(1, 0);
  if (r) return r;
  if (A.nnzb == 0) return kOk;
  const dim3 grid3(ceil_div(A.nnzb, 256)), grid6(8 * ceil_div(A.n_slices, 8), kTileSteps);
  if (A.br == 3 && npe == 10 && !sym)
    hipLaunchKernelGGL(assemble_block3_kernel<10>, grid3, dim3(256), 0, s, A.nnzb, npe, 0, rowidx, colidx, cptr, codes,
                       Ke, node_fix, A.d_slot, A.d_v64, vals_std);
  else if (A.br == 3)
    hipLaunchKernelGGL(assemble_block3_kernel<0>, grid3, dim3(256), 0, s, A.nnzb, npe, sym, rowidx, colidx, cptr,
                       codes, Ke, node_fix, A.d_slot, A.d_v64, vals_std);
  else if (A.br == 6)
    hipLaunchKernelGGL(assemble_tile_kernel, grid6, dim3(kTileThreads), 0, s, A.view<double>(), A.d_rstart, npe, sym,
                       cptr, codes, Ke, node_fix, A.d_v64, vals_std);
  else
    return kBadArg;
  return static_cast<int>(hipGetLastError());
}

// ---------------------------------------------------------------- values in the layout's order
// v32 (and v64e, v16) = s_i * v64 * s_j per scalar entry (symmetric diagonal
// equilibration).  One workgroup per slice, one wavefront per step, one lane
// per slot: loads and stores of the values are contiguous, the row's scale is
// loaded once, the column's is a 24- or 48-byte gather.  Bound by the values'
// bytes; one thread per entry in standard block order read and wrote 16-byte
// pieces (117 585 rows, 2.9 M blocks: 246 us, here 65 us).
template <int B>
__global__ __launch_bounds__(64 * kAsmWaves) void equilibrate_kernel(SellView<double> A,
                                                                     const double* __restrict__ scale,
                                                                     float* __restrict__ v32,
                                                                     double* __restrict__ v64e,
                                                                     _Float16* __restrict__ v16) {
  constexpr int BB = B * B;
  const int s = slice_of_block(A.n_slices, 1);
  if (s >= A.n_slices) return;
  const int lane = threadIdx.x & 63, rps = 64 / A.lanes, q = lane / rps;
  const int2 ri = A.rinfo[s * rps + lane % rps];
  const long long base = A.off[s];
  const int steps = (int)((A.off[s + 1] - base) >> 6);
  double sr[B];
#pragma unroll
  for (int r = 0; r < B; ++r) sr[r] = ri.x >= 0 ? scale[(size_t)ri.x * B + r] : 0.0;
  for (int j = threadIdx.x >> 6; j < steps; j += kAsmWaves) {
    if (j * A.lanes + q >= ri.y) continue;
    const long long slot = base + 64LL * j + lane, region = (base + 64LL * j) * BB;
    const size_t c0 = (size_t)A.col[slot] * B;
    double v[BB], sc[B];
#pragma unroll
    for (int c = 0; c < B; ++c) sc[c] = scale[c0 + c];
    load_block<double, BB>(A.val + region, lane, v);
#pragma unroll
    for (int e = 0; e < BB; ++e) v[e] = sr[e / B] * v[e] * sc[e % B];
    store_block<float, BB>(v32 + region, lane, v);
    if (v64e) store_block<double, BB>(v64e + region, lane, v);
    if (v16) {
      float f[BB];
#pragma unroll
      for (int e = 0; e < BB; ++e) f[e] = float(v[e]);
      store_block<_Float16, BB>(v16 + region, lane, f);
    }
  }
}

// The values back in standard block order: a wavefront's blocks of one row are
// consecutive there, so it turns its step through LDS and stores runs of up to
// L BB values (117 585 rows: one thread per entry, reading 16-byte pieces, 180
// us; a lane storing its own block 123 us; here 82 us).
template <int BB>
__global__ __launch_bounds__(64 * kAsmWaves) void sell_to_std_kernel(SellView<double> A,
                                                                     const int* __restrict__ rstart,
                                                                     double* __restrict__ vs) {
  __shared__ double tile[kAsmWaves][64 * (BB | 1)];
  const int s = slice_of_block(A.n_slices, 1);
  if (s >= A.n_slices) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, rps = 64 / A.lanes;
  const int pos = s * rps + lane % rps;
  const int len = A.rinfo[pos].y, k0 = rstart[pos];
  const long long base = A.off[s];
  const int steps = (int)((A.off[s + 1] - base) >> 6), run = A.lanes * BB;
  for (int j = wave; j < steps; j += kAsmWaves) {
    double v[BB];
    load_block<double, BB>(A.val + (base + 64LL * j) * BB, lane, v);  // padding slots hold values too
#pragma unroll
    for (int e = 0; e < BB; ++e) tile[wave][lane * (BB | 1) + e] = v[e];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < BB; ++i) {
      const int f = 64 * i + lane, r = f / run, w = f - r * run;  // row of the slice, entry of its run
      const int first = j * A.lanes, n = min(A.lanes, __shfl(len, r, 64) - first);
      const long long k = (long long)__shfl(k0, r, 64) + first;
      if (w < n * BB) vs[k * BB + w] = tile[wave][(w / BB * rps + r) * (BB | 1) + w % BB];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

void launch_equilibrate_slots(const SellMatrix& A, const double* scale, double* v64e, hipStream_t s) {
  const dim3 grid(8 * ceil_div(A.n_slices, 8)), block(64 * kAsmWaves);
  if (A.br == 3)
    hipLaunchKernelGGL(equilibrate_kernel<3>, grid, block, 0, s, A.view<double>(), scale, A.d_v32, v64e, A.d_v16);
  else
    hipLaunchKernelGGL(equilibrate_kernel<6>, grid, block, 0, s, A.view<double>(), scale, A.d_v32, v64e, A.d_v16);
}

void launch_to_std_slots(const SellMatrix& A, double* vals_std, hipStream_t s) {
  const dim3 grid(8 * ceil_div(A.n_slices, 8)), block(64 * kAsmWaves);
  const SellView<double> v = A.view<double>();
  if (A.br * A.bc == 9)
    hipLaunchKernelGGL(sell_to_std_kernel<9>, grid, block, 0, s, v, A.d_rstart, vals_std);
  else if (A.br * A.bc == 18)
    hipLaunchKernelGGL(sell_to_std_kernel<18>, grid, block, 0, s, v, A.d_rstart, vals_std);
  else
    hipLaunchKernelGGL(sell_to_std_kernel<36>, grid, block, 0, s, v, A.d_rstart, vals_std);
}

}  // namespace wn
