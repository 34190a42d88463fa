// Standalone batched unit-triangular solve: X = (I + L)^-1 B or
// X = (I + L)^-T B per head, L = strict lower part of a [H][C][C] (C <= 64),
// B [H][C][N] -- the drop-in for the reference's UT-solve kernels
// (net/kernels/kda_ut_solve.py:525 kernel, :536 kernel_t) -- and the backward
// rule of their custom_vjp (:563 _backward): dB = the sibling solve of dX,
// dA = strict_lower(-dB X^T) (or strict_lower(-X dB^T) for the transposed
// solve).  fp32 arithmetic; a, b, x fp32 or bf16.
//
// One workgroup per (head, 64-column tile of B): L (zero-padded to 64 x 64)
// and the B tile go to LDS (all of a thread's loads in flight together),
// T = (I + L)^-1 is formed there (kda_tri.h), and X = T B (or T^T B) runs on
// the fp32 matrix cores.  Padding rows/columns beyond C and N are zero and
// never stored.  The backward rule of few heads is one launch of its own kernel (below).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kda_common.h"
#include "kda_internal.h"
#include "kda_tri.h"

namespace kda {
namespace {

constexpr int kN = 64;        // padded size
constexpr int kPC = kN + 1;   // LDS pitch
constexpr int kUtThreads = 256;

template <int DT>
__device__ __forceinline__ float ut_ld(const void* p, int64_t i) {
  if constexpr (DT == 0) return static_cast<const float*>(p)[i];
  else return bf16_to_f32(static_cast<const u16*>(p)[i]);
}

template <int DT>
__device__ __forceinline__ void ut_st(void* p, int64_t i, float v) {
  if constexpr (DT == 0) static_cast<float*>(p)[i] = v;
  else static_cast<u16*>(p)[i] = f32_to_bf16_bits(v);
}

__device__ __forceinline__ f4 mfma4(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// A 64 x 64 block of a row-major [rows][ld] array (element (r, col0 + i)), zero
// outside rows < nr and columns < nc (LOWER: and on and above the diagonal), in
// registers: every load of a thread is issued, at a clamped, valid address.
constexpr int kUtPer = kN * kN / kUtThreads;

template <int DT, bool LOWER>
__device__ __forceinline__ void ut_tile_read(float* v, const void* src, int64_t base, int ld, int col0, int nr,
                                             int nc) {
#pragma unroll
  for (int p = 0; p < kUtPer; ++p) {
    const int e = threadIdx.x + kUtThreads * p;
    const int r = e >> 6, i = e & 63;
    const bool ok = r < nr && i < nc && (!LOWER || i < r);
    const int64_t idx = ok ? base + static_cast<int64_t>(r) * ld + col0 + i : base;
    const float x = ut_ld<DT>(src, idx);
    v[p] = ok ? x : 0.f;
  }
}

__device__ __forceinline__ void ut_tile_store(float* dst, const float* v) {
#pragma unroll
  for (int p = 0; p < kUtPer; ++p) {
    const int e = threadIdx.x + kUtThreads * p;
    dst[(e >> 6) * kPC + (e & 63)] = v[p];
  }
}

// The same into LDS [64][kPC].
template <int DT, bool LOWER>
__device__ __forceinline__ void ut_tile_load(float* dst, const void* src, int64_t base, int ld, int col0, int nr,
                                             int nc) {
  float v[kUtPer];
  ut_tile_read<DT, LOWER>(v, src, base, ld, col0, nr, nc);
  ut_tile_store(dst, v);
}

// X = T B (or T^T B; the backward rule's dB with B = dX) on the fp32 matrix
// cores: wave w owns row tile w and the four column tiles.
template <int DT, bool TR>
__global__ __launch_bounds__(kUtThreads) void kda_ut_solve_kernel(UtArgs a) {
  __shared__ float sL[kN * kPC], sT[kN * kPC], sB[kN * kPC], tmp[768];
  const int t = threadIdx.x, w = t >> 6, l = t & 63, r = l & 15, gq = l >> 4;
  const int h = blockIdx.x / a.ntiles, tile = blockIdx.x - h * a.ntiles;
  const int j0 = kN * tile;
  const int C = a.C, N = a.N;
  const int64_t abase = static_cast<int64_t>(h) * C * C;
  const int64_t bbase = static_cast<int64_t>(h) * C * N;
  ut_tile_load<DT, true>(sL, a.a, abase, C, 0, C, C);
  ut_tile_load<DT, false>(sB, a.b, bbase, N, j0, C, N - j0);
  __syncthreads();
  invert_unit_lower64<kPC, kUtThreads>(sL, sT, tmp);
  f4 acc[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[q][e] = 0.f;
#pragma unroll 4
  for (int k = 0; k < kN / 4; ++k) {
    const int m = 4 * k + gq;
    const float at = TR ? sT[m * kPC + 16 * w + r] : sT[(16 * w + r) * kPC + m];   // (T or T^T)[c][m]
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = mfma4(at, sB[m * kPC + 16 * q + r], acc[q]);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = 16 * w + 4 * gq + e, col = j0 + 16 * q + r;
      if (c < C && col < N) ut_st<DT>(a.x, bbase + static_cast<int64_t>(c) * N + col, acc[q][e]);
    }
}

// dA[h] = strict_lower(-Y X^T) (TR = false: Y = db, X = forward solution) or
// strict_lower(-X Y^T) (TR = true); one workgroup per head, K = N in tiles of
// 64, on the fp32 matrix cores (wave w: row tile w, four column tiles).
template <int DT, bool TR>
__global__ __launch_bounds__(kUtThreads) void kda_ut_da_kernel(UtArgs a) {
  __shared__ float sY[kN * kPC], sX[kN * kPC];
  const int t = threadIdx.x, w = t >> 6, l = t & 63, r = l & 15, gq = l >> 4;
  const int h = blockIdx.x;
  const int C = a.C, N = a.N;
  const int64_t bbase = static_cast<int64_t>(h) * C * N;
  // P = sum_n R[c][n] Q[i][n] with R = Y, Q = X (TR: R = X, Q = Y)
  const void* Rp = TR ? a.xf : a.x;
  const void* Qp = TR ? a.x : a.xf;
  f4 acc[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[q][e] = 0.f;
  for (int n0 = 0; n0 < N; n0 += kN) {
    ut_tile_load<DT, false>(sY, Rp, bbase, N, n0, C, N - n0);
    ut_tile_load<DT, false>(sX, Qp, bbase, N, n0, C, N - n0);
    __syncthreads();
#pragma unroll 4
    for (int k = 0; k < kN / 4; ++k) {
      const int n = 4 * k + gq;
      const float ar = sY[(16 * w + r) * kPC + n];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = mfma4(ar, sX[(16 * q + r) * kPC + n], acc[q]);
    }
    __syncthreads();
  }
  const int64_t abase = static_cast<int64_t>(h) * C * C;
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = 16 * w + 4 * gq + e, col = 16 * q + r;
      if (c < C && col < C) ut_st<DT>(a.da, abase + static_cast<int64_t>(c) * C + col, (col < c) ? -acc[q][e] : 0.f);
    }
}

// The backward rule in one launch: one workgroup per (head, 16 rows of dB).  It
// forms its rows of dB for every column, in tiles of 64 (wave w: columns 16 w to
// 16 w + 15), and each wave takes them from its accumulators straight into its
// share of dA, a product over the columns; the four shares meet in LDS at the
// end.  TR as in the solve: T^T was applied, dA = strict_lower(-dB X^T), so the 16
// rows of dB are 16 rows of dA; else dA = strict_lower(-X dB^T) and they are 16 of
// its columns.
//
// Latency bounds it: the loads and the inverse once, then two barriers a tile, the
// next tile's loads behind the products.  Against the solve and a dA launch of one
// workgroup per head it splits dA over four times the workgroups and needs no
// second launch, which waits for the first and reads dB back; each workgroup
// repeats the head's inverse, as the solve's column tiles do.
// H 12, C 64, N 256, fp32: 8.4 + 11.0 us in two launches, 13.6 us in one.
template <int DT, bool TR>
__global__ __launch_bounds__(kUtThreads) void kda_ut_bwd_kernel(UtArgs a) {
  __shared__ float sm[4 * kN * kPC], tmp[768];
  float *sL = sm, *sT = sm + kN * kPC, *sB = sm + 2 * kN * kPC, *sX = sm + 3 * kN * kPC;
  const int t = threadIdx.x, w = t >> 6, l = t & 63, r = l & 15, gq = l >> 4;
  const int C = a.C, N = a.N, rtiles = (C + 15) / 16;
  const int h = blockIdx.x / rtiles, i = blockIdx.x - h * rtiles;
  const int64_t abase = static_cast<int64_t>(h) * C * C;
  const int64_t bbase = static_cast<int64_t>(h) * C * N;
  float vb[kUtPer], vx[kUtPer];
  {
    float vl[kUtPer];
    ut_tile_read<DT, true>(vl, a.a, abase, C, 0, C, C);
    ut_tile_read<DT, false>(vb, a.b, bbase, N, 0, C, N);
    ut_tile_read<DT, false>(vx, a.xf, bbase, N, 0, C, N);
    ut_tile_store(sL, vl);
  }
  ut_tile_store(sB, vb);
  ut_tile_store(sX, vx);
  __syncthreads();
  invert_unit_lower64<kPC, kUtThreads>(sL, sT, tmp);
  float at[kN / 4];   // (T^T or T)[16 i + r][4 k + gq], the same for every tile
#pragma unroll
  for (int k = 0; k < kN / 4; ++k) {
    const int m = 4 * k + gq;
    at[k] = TR ? sT[m * kPC + 16 * i + r] : sT[(16 * i + r) * kPC + m];
  }
  f4 acc[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[q][e] = 0.f;
  for (int n0 = 0; n0 < N; n0 += kN) {
    const bool more = n0 + kN < N;
    if (more) {
      ut_tile_read<DT, false>(vb, a.b, bbase, N, n0 + kN, C, N - n0 - kN);
      ut_tile_read<DT, false>(vx, a.xf, bbase, N, n0 + kN, C, N - n0 - kN);
    }
    // dB^T: lane (r, gq) gets dB[16 i + r][n0 + 16 w + 4 gq + e], which is also
    // what it supplies as B[k = gq][r] of the dA product's step e
    f4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kN / 4; ++k) d = mfma4(sB[(4 * k + gq) * kPC + 16 * w + r], at[k], d);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (TR ? q <= i : q >= i) {   // the other row tiles of X meet dA above the diagonal
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[q] = mfma4(sX[(16 * q + r) * kPC + 16 * w + 4 * gq + e], d[e], acc[q]);
      }
    const int c = 16 * i + r, col = n0 + 16 * w + 4 * gq;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c < C && col + e < N) ut_st<DT>(a.x, bbase + static_cast<int64_t>(c) * N + col + e, d[e]);
    __syncthreads();
    if (more) {
      ut_tile_store(sB, vb);
      ut_tile_store(sX, vx);
      __syncthreads();
    }
  }
  // the waves' shares of P[j][c] = sum_n X[j][n] dB[16 i + c][n], added in wave order;
  // sL and sT were last read before the loop's barriers
  constexpr int kPR = 17;
  float* red = sm;
  static_assert(4 * kN * kPR <= 2 * kN * kPC, "the shares fit sL and sT");
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) red[(w * kN + 16 * q + 4 * gq + e) * kPR + r] = acc[q][e];
  __syncthreads();
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int e = t + kUtThreads * p;
    const int j = TR ? e & 63 : e >> 4, c = TR ? e >> 6 : e & 15;
    float v = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) v += red[(s * kN + j) * kPR + c];
    const int row = TR ? 16 * i + c : j, col = TR ? j : 16 * i + c;
    if (row < C && col < C) ut_st<DT>(a.da, abase + static_cast<int64_t>(row) * C + col, col < row ? -v : 0.f);
  }
}

constexpr int kUtOneRound = 512;   // two workgroups (LDS) on each of 256 CUs

template <int DT>
hipError_t launch_ut_t(const UtArgs& a, bool transpose, bool with_da, hipStream_t s) {
  if (with_da) {
    // One launch while its workgroups (16 rows of a head each) run in one round, two
    // a CU, or, with at most 32 rows, form no more inverses than the solve's column
    // tiles would: past that each row tile's own inverse and reads of X and dX cost
    // more than the second launch.  us in two launches and in one, fp32: C 64 N 64,
    // 128 heads 12.8 and 10.6, 192 13.1 and 18.2, 1 024 34.0 and 69.2; C 64 N 1 024,
    // 128 heads 72.5 and 67.3, 192 84.8 and 105; C 32, 1 024 heads, N 64 28.5 and
    // 33.7, N 128 48.9 and 43.1, N 512 174 and 99; C 16 N 64, 1 024 heads 26.0 and 17.9.
    // Two launches also where an output shares memory with an input: workgroups of one
    // head read all of a, dX and X while others write, where the two launches
    // read a head's a and a column's dX before they write over them.
    const int rtiles = (a.C + 15) / 16;
    const bool one = static_cast<int64_t>(a.H) * rtiles <= kUtOneRound || (rtiles <= 2 && rtiles <= a.ntiles);
    const int64_t es = DT == 0 ? 4 : 2, na = es * a.H * a.C * a.C, nb = es * a.H * a.C * a.N;
    auto apart = [&](const void* in, int64_t n) { return !overlaps(a.x, nb, in, n) && !overlaps(a.da, na, in, n); };
    if (one && apart(a.a, na) && apart(a.b, nb) && apart(a.xf, nb)) {
      const dim3 grid(a.H * rtiles);
      if (transpose) hipLaunchKernelGGL((kda_ut_bwd_kernel<DT, true>), grid, dim3(kUtThreads), 0, s, a);
      else hipLaunchKernelGGL((kda_ut_bwd_kernel<DT, false>), grid, dim3(kUtThreads), 0, s, a);
      return hipGetLastError();
    }
  }
  const int grid = a.H * a.ntiles;
  if (transpose) hipLaunchKernelGGL((kda_ut_solve_kernel<DT, true>), dim3(grid), dim3(kUtThreads), 0, s, a);
  else hipLaunchKernelGGL((kda_ut_solve_kernel<DT, false>), dim3(grid), dim3(kUtThreads), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !with_da) return e;
  // the backward of the forward solve runs the transposed solve, and vice
  // versa; `transpose` here is the solve just run, so the dA form is its
  // opposite: forward solve's backward (transpose == true) uses -Y X^T
  if (transpose) hipLaunchKernelGGL((kda_ut_da_kernel<DT, false>), dim3(a.H), dim3(kUtThreads), 0, s, a);
  else hipLaunchKernelGGL((kda_ut_da_kernel<DT, true>), dim3(a.H), dim3(kUtThreads), 0, s, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_ut(const UtArgs& a, int dtype, bool transpose, bool with_da, hipStream_t s) {
  return dtype == 0 ? launch_ut_t<0>(a, transpose, with_da, s) : launch_ut_t<1>(a, transpose, with_da, s);
}

}  // namespace kda
