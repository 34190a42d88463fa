// Chunked KDA backward (dense [B, T, H, d] inputs).
//
// Gradients of o = chunk_fwd(q, k, v, g, beta, h0) and of the final state
// with respect to q, k, v, g (the log decay), beta and h0, following the
// reference's analytic adjoint per chunk (net/kernels/kda_cc_fused_bwd.py:30-55,
// code :139-228) scanned in reverse over the chunks
// (net/kernels/kda_cc_fused_persist.py:794-842, reference_bwd_scan).  Three
// launches, the two scans in one:
//   kda_bwd_prep_kernel   one workgroup per chunk-head: in-chunk log2 cumsum G,
//                         gamma*q, lambda*k, gamma_C, Aqk, T = (I+L)^-1, W, U;
//   forward state scan    one workgroup per (chain, 32 value columns): every
//                         chunk's incoming state S and its v~ = U - W S;
//   reverse scan          same grid, chunks in reverse: the state cotangent
//                         dS entering each chunk from the right, and
//                         dv~ = (lambda k) dS + Aqk^T do;
//                         dS <- gamma_C dS + (gamma q)^T do - W^T dv~; dh0;
//   kda_bwd_chunk_kernel  one workgroup per chunk-head: the rest of the adjoint
//                         (dY, dgq, dW, the two transposed solves, dL, dAqk, the
//                         score adjoints, the cumsum adjoint) and the outputs.
// Two precisions of the workspace, chosen by the input dtype:
//  * fp32 inputs: every workspace array fp32 row-major per chunk-head
//    ch = (b * NT + n) * H + h; scans fscan_block and rscan_block
//    (16 waves, operands split into bf16 hi/lo planes in LDS each chunk step).
//  * 16-bit inputs (bf16, fp16): the forward-side arrays gamma q, lambda k,
//    Aqk, T, W and the stored state S are fp16 (BwdWs<true>: the operand
//    width the forward's own kernels give them), and the
//    prep kernel writes the scans' operands directly as MFMA lane fragments
//    (FL, FA, FQ, FW, FWN, FLT); G, gamma_C, U, v~ and the cotangents dS', dv~
//    stay fp32.  Scans fscan16_block and rscan16_block in the column-owner
//    form: two compute waves (one 16-column tile each of the
//    32-column slice, the state slice in their accumulators) and four
//    producer waves that load two chunks ahead into registers, fill a
//    double-buffered LDS chunk, and store the compute waves' staged outputs
//    a step later; one barrier per chunk step.
// Products: fp16 operands on v_mfma_f32_16x16x32_f16 (exact products of the
// stored values); fp32 operands (cotangents, v~, U, S in the fp32 path) as
// hi/lo pairs of a 16-bit type, about 2^-16 of each product dropped (the
// 16-bit scans scale each column's cotangent by a power of two first, so the
// fp16 pair keeps ~22 bits whatever its range); the rest (prep scores, phase 4
// of the chunk kernel) on v_mfma_f32_16x16x4f32.  Decay factors of
// off-diagonal 16-row tiles are anchored at the row tile's first row
// (2^(G_c - G_a) * 2^(G_a - G_i), both <= 1; the chunk kernel also at the key
// tile's last row); diagonal tiles likewise when the tile's decay span allows
// (kDiagAnchorLog2), else per element.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kda_common.h"
#include "kda_internal.h"
#include "kda_tri.h"

namespace kda {
namespace {

constexpr int kC = 64;
constexpr int kThreads = 256;
// The per-chunk adjoint runs one workgroup per CU (its LDS) and is bound by
// latency: a wave per (row tile, two column tiles), so d = 128 has four waves
// per SIMD, each with half the gradients' partial sums of a two-wave form.
template <int D>
struct ChunkThreads {
  static constexpr int value = (D == 128) ? 1024 : 512;
};
// Scan workgroups: one per (chain, 32-column slice).  The scans are bound by
// the latency of their serial chunk steps (operand splits into LDS, three
// barriers and two short MFMA chains per step), so d = 128 runs 16 waves (four
// per SIMD: one state tile and half the operand splitting per wave), d = 64
// eight.
template <int D>
struct ScanThreads {
  static constexpr int value = (D == 128) ? 1024 : 512;
};
constexpr int kScanThreads = 512;   // threads of the 64-column transposed tiles of the scans
// The prep kernel likewise (the channel sums of a score tile pair split over
// the two halves of the workgroup).
constexpr int kPrepThreads = 512;

// The value, unknown to the compiler from here on (it recomputes what was
// derived from it instead of keeping the derived values in registers).
__device__ __forceinline__ int fresh_tid() {   // threadIdx.x, likewise
  int x = threadIdx.x;
  asm volatile("" : "+v"(x));
  return x;
}
__device__ __forceinline__ void opaque(int& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void opaque(float& x) { asm volatile("" : "+v"(x)); }

__device__ __forceinline__ float ex2(float x) { return __builtin_amdgcn_exp2f(x); }

constexpr int cmax(int a, int b) { return a > b ? a : b; }

// Token row of chunk row c (dense layout) and whether it exists.
struct ChunkRows {
  int64_t row0;   // b * T + n * 64
  int len;        // valid rows of this chunk
};

__device__ __forceinline__ ChunkRows chunk_rows(const BwdArgs& a, int u) {
  const int b = u / a.NT, n = u - b * a.NT;
  ChunkRows r;
  r.row0 = static_cast<int64_t>(b) * a.T + static_cast<int64_t>(n) * kC;
  r.len = min(kC, a.T - n * kC);
  return r;
}

// ROWS x COLS block of a row-major array (row stride src_ld elements, first
// column col0) into LDS rows, in two halves: the loads into registers (fetch; a
// thread's share, Tile::PER pieces of four elements) and the LDS writes (put).
// Apart, a scan kernel issues the next chunk's loads before the current chunk's
// arithmetic.
//
// Workspace arrays are fp32 (ET 0) or fp16 (ET 2, see BwdWs); an fp16 tile
// loads 8 bytes per piece and converts when it is written to LDS, so the wait
// for the load falls there, not at the fetch.
template <int ET>
struct WsPiece {
  typedef uint2 t;
};
template <>
struct WsPiece<0> {
  typedef float4 t;
};
template <int ET>
__device__ __forceinline__ float4 ws_unpack(const typename WsPiece<ET>::t& w) {
  if constexpr (ET == 0) {
    return w;
  } else {
    const f4 v = unpack4<ET>(w);
    return make_float4(v[0], v[1], v[2], v[3]);
  }
}
// element `off` of a workspace array of element type ET
template <int ET>
__device__ __forceinline__ const void* ws_at(const float* base, int64_t off) {
  if constexpr (ET == 0) return base + off;
  else return reinterpret_cast<const u16*>(base) + off;
}
template <int ET>
__device__ __forceinline__ void ws_st(float* base, int64_t off, float x) {
  static_assert(ET == 0 || ET == 2, "workspace arrays are fp32 or fp16");
  if constexpr (ET == 0) base[off] = x;
  else reinterpret_cast<u16*>(base)[off] = __builtin_bit_cast(u16, static_cast<_Float16>(x));
}
// four consecutive elements (off a multiple of 4)
template <int ET>
__device__ __forceinline__ void ws_st4(float* base, int64_t off, float4 x) {
  if constexpr (ET == 0) {
    *reinterpret_cast<float4*>(base + off) = x;
  } else {
    static_assert(ET == 2, "workspace arrays are fp32 or fp16");
    typedef _Float16 hv4 __attribute__((ext_vector_type(4)));
    const hv4 v = {static_cast<_Float16>(x.x), static_cast<_Float16>(x.y), static_cast<_Float16>(x.z),
                   static_cast<_Float16>(x.w)};
    *reinterpret_cast<uint2*>(reinterpret_cast<u16*>(base) + off) = __builtin_bit_cast(uint2, v);
  }
}

// four fp32 -> packed fp16 (round to nearest even)
__device__ __forceinline__ uint2 pack_f16x4(const f4& x) {
  const h4 v = {static_cast<_Float16>(x[0]), static_cast<_Float16>(x[1]), static_cast<_Float16>(x[2]),
                static_cast<_Float16>(x[3])};
  return __builtin_bit_cast(uint2, v);
}

// Element types of the backward's workspace.  fp32 inputs keep every array
// fp32.  16-bit inputs store six forward-side arrays in fp16 (gamma q,
// lambda k, Aqk, T, W and the chunk's incoming state S: the operand width the
// forward's own kernels use for them); G, gamma_C, U, v~ (U - W S cancels, so
// their rounding would reach the gradients amplified) and the cotangents dS,
// dv~ (whose scale is the caller's) stay fp32.
template <bool WS16>
struct BwdWs {
  static constexpr int F = WS16 ? 2 : 0;
};

template <int ROWS, int COLS, int NTH = kThreads, int ET = 0>
struct Tile {
  static constexpr int V = COLS / 4;
  static constexpr int N = ROWS * V;
  static constexpr int PER = (N + NTH - 1) / NTH;
  static_assert(COLS % 4 == 0, "four-element pieces");
  typedef typename WsPiece<ET>::t Piece;
  Piece r[PER];
  __device__ __forceinline__ void fetch(const void* src, int src_ld, int col0) {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int e = fresh_tid() + p * NTH;
      if (N % NTH == 0 || e < N) {
        const int row = e / V, c4 = e - row * V;
        const int64_t i = static_cast<int64_t>(row) * src_ld + col0 + 4 * c4;
        if constexpr (ET == 0) r[p] = *reinterpret_cast<const float4*>(static_cast<const float*>(src) + i);
        else r[p] = *reinterpret_cast<const uint2*>(static_cast<const u16*>(src) + i);
      }
    }
  }
  __device__ __forceinline__ float4 get(int p) const { return ws_unpack<ET>(r[p]); }
  template <int PITCH>
  __device__ __forceinline__ void put(float* dst) const {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int e = fresh_tid() + p * NTH;
      if (N % NTH == 0 || e < N) {
        const int row = e / V, c4 = e - row * V;
        const float4 x = get(p);
        float* d = dst + row * PITCH + 4 * c4;
        d[0] = x.x;
        d[1] = x.y;
        d[2] = x.z;
        d[3] = x.w;
      }
    }
  }
};

// Largest in-tile decay (log2 units, one channel) at which the chunk
// kernel's diagonal score-adjoint tiles run on the matrix cores anchored at
// the tile's first row: the key factors reach 2^kDiagAnchorLog2, which leaves
// 2^96 of fp32's range for the cotangent sums they multiply.
constexpr float kDiagAnchorLog2 = 32.f;

// Workgroup -> (chain, 32-column slice) of the scan kernels: the NS slices
// of a chain on one XCD (workgroup x runs on XCD x % 8), so the operands all
// of them read come from that XCD's L2.  Grid: ceil(chains / 8) * 8 * NS.
template <int NS>
__device__ __forceinline__ bool scan_slot(int x, int nchains, int& chain, int& split) {
  const int xcd = x & 7, kk = x >> 3;
  const int slot = kk / NS;
  split = kk - slot * NS;
  chain = slot * 8 + xcd;
  return chain < nchains;
}

// Columns [col0, col0 + COLS) of the 64 rows of a chunk of a token-major input
// tensor [*, H, D] (DT 0 fp32, 1 bf16, 2 fp16; rows past `len` read as zero),
// 8 elements per load: the loads (fetch) and the LDS writes (put) are apart, so
// a kernel can issue the loads of a later phase before this phase's arithmetic.
template <int DT, int D, int COLS, int NTH>
struct InTile {
  static constexpr int V = COLS / 8;
  static constexpr int N = kC * V;
  static constexpr int PER = (N + NTH - 1) / NTH;
  static_assert(COLS % 8 == 0, "8-element loads");
  uint4 w[DT == 0 ? 2 * PER : PER];
  __device__ __forceinline__ void fetch(const void* src, int64_t row0, int len, int H, int h, int col0) {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int e = fresh_tid() + p * NTH;
      const int r = e / V, c8 = e - r * V;
      const bool ok = (N % NTH == 0 || e < N) && r < len;
      const int64_t i = ((row0 + (ok ? r : 0)) * H + h) * D + col0 + 8 * c8;
      // the address is valid for every thread (row 0 when masked): load
      // unconditionally, then zero, so no load sits inside a branch
      const uint4 z = make_uint4(0, 0, 0, 0);
      if constexpr (DT == 0) {
        const uint4* q = reinterpret_cast<const uint4*>(static_cast<const float*>(src) + i);
        const uint4 v0 = q[0], v1 = q[1];
        w[2 * p] = ok ? v0 : z;
        w[2 * p + 1] = ok ? v1 : z;
      } else {
        const uint4 v = *reinterpret_cast<const uint4*>(static_cast<const u16*>(src) + i);
        w[p] = ok ? v : z;
      }
    }
  }
  // the elements as they are (LOG: as in put), rows of PITCH elements
  template <int PITCH, bool LOG = false>
  __device__ __forceinline__ void put_raw(typename InT<DT>::t* dst, int len = kC) const {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int e = fresh_tid() + p * NTH;
      if (N % NTH == 0 || e < N) {
        const int r = e / V, c8 = e - r * V;
        u32x4* o = reinterpret_cast<u32x4*>(dst + r * PITCH + 8 * c8);
        auto vec = [&](const uint4& x) {
          u32x4 y = {x.x, x.y, x.z, x.w};
          if constexpr (LOG) {
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = (r < len) ? __float_as_uint(logf(__uint_as_float(y[i]))) : 0u;
          }
          return y;
        };
        if constexpr (DT == 0) {
          o[0] = vec(w[2 * p]);
          o[1] = vec(w[2 * p + 1]);
        } else {
          o[0] = vec(w[p]);
        }
      }
    }
  }
  // LOG: the elements are decay factors alpha; their logarithm (0 in the rows from len on)
  template <int PITCH, bool LOG = false>
  __device__ __forceinline__ void put(float* dst, float mul, int len = kC) const {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int e = fresh_tid() + p * NTH;
      if (N % NTH == 0 || e < N) {
        const int r = e / V, c8 = e - r * V;
        float x[8];
        if constexpr (DT == 0) {
          const uint4 a = w[2 * p], b = w[2 * p + 1];
          x[0] = __uint_as_float(a.x); x[1] = __uint_as_float(a.y); x[2] = __uint_as_float(a.z); x[3] = __uint_as_float(a.w);
          x[4] = __uint_as_float(b.x); x[5] = __uint_as_float(b.y); x[6] = __uint_as_float(b.z); x[7] = __uint_as_float(b.w);
        } else {
          const f4 lo = unpack4<DT>(make_uint2(w[p].x, w[p].y)), hi = unpack4<DT>(make_uint2(w[p].z, w[p].w));
#pragma unroll
          for (int q = 0; q < 4; ++q) { x[q] = lo[q]; x[4 + q] = hi[q]; }
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          if constexpr (LOG) dst[r * PITCH + 8 * c8 + q] = (r < len) ? logf(x[q]) : 0.f;
          else dst[r * PITCH + 8 * c8 + q] = x[q] * mul;
        }
      }
    }
  }
};

// Gate type (beside the element types 0 fp32, 1 bf16, 2 fp16) of the cc_scan
// seam: g holds the decay factors alpha in fp32 (the log decay is their
// logarithm) and beta the [token-head][32] columns beta32 whose mean it is.
constexpr int kAlphaGates = 3;

// beta of one token-head (the seam's 32 columns summed in column order, as
// the forward does)
template <int DTG>
__device__ __forceinline__ float ld_beta(const void* p, int64_t th) {
  if constexpr (DTG == kAlphaGates) {
    const f4* b = reinterpret_cast<const f4*>(static_cast<const float*>(p) + th * 32);
    f4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = b[j];
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) s += v[j][e];
    return s * (1.0f / 32.0f);
  } else {
    return ld1<DTG>(p, th);
  }
}

// ---------------------------------------------------------------------------
// prep: G, gamma*q, lambda*k, gamma_C, Aqk, T, W, U of one chunk-head
// ---------------------------------------------------------------------------
__device__ __forceinline__ f4 mfma4(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Index of the stored Aqk^T A fragment (key tile it, K step kb over the query
// rows): (0,0) (0,1) (1,0) (1,1) (2,1) (3,1); (2,0) and (3,0) are zero and
// not stored.
__device__ __forceinline__ int fa_frag(int it, int kb) { return (it < 2) ? 2 * it + kb : it + 2; }

// The chunk's channels are taken in halves of 64 (d = 128) so the shared
// memory fits two workgroups per CU: the scores accumulate over the halves in
// registers, T = (I+L)^-1 is built once, and W, U are formed per half of
// their columns.
//
// Per half, thread (channel d = t % 64, rows 8 s .. 8 s + 7, s = t / 64) owns a
// column segment of q, k, g: it forms G there, and from G everything with a
// decay in it, once per element: the scores' operands q 2^(G - Ga), k 2^(G -
// Ga), k 2^(Ge - G) (Ga, Ge: G of the row tile's first and last row; into LDS,
// over the raw rows), gamma q, lambda k (stored as the scans' fragments) and
// gamma k (kept in registers for W).  The scores read their operands 16 bytes
// at a time, four channels per lane for four v_mfma_f32_16x16x4f32, and a tile
// pair costs one factor 2^(Ga_R - Ge_s) per channel.
// Bound by its phases' latencies beside its traffic (192 KiB per chunk-head at
// d = 128, 16-bit inputs: 155 us of 4 096 chunk-heads at the copy rate).  4 096
// chunk-heads, 16-bit inputs, traced medians: 273 us with each decay factor
// formed per operand and tile pair, element-wise LDS reads and the first half's
// k, g staged again for W; 214 now (within a training step of the layer 291 and
// 234); 3 072 of the seam's 229 (and an adapter pass) and 185; 256 in fp32 30 and 25.
template <int D, int DTQ, int DTG>
__global__ __launch_bounds__(kPrepThreads, 4) void kda_bwd_prep_kernel(BwdArgs a) {
  constexpr int EF = BwdWs<DTQ != 0>::F;   // gamma q, lambda k, Aqk, T, W
  constexpr bool ALPHA = DTG == kAlphaGates;
  constexpr int GT = ALPHA ? 0 : DTG;  // element type of g
  constexpr int HD = 64;              // channels per half
  constexpr int NHALF = D / HD;
  // [64][64] pitch: rows 4 banks apart and 16-byte aligned
  constexpr int P = HD + 4;
  __shared__ __attribute__((aligned(16))) float sQ[kC * P];   // q, then q 2^(G - Ga); T after the scores
  __shared__ __attribute__((aligned(16))) float sK[kC * P];   // k, then k 2^(G - Ga); (beta gamma k)^T for W
  __shared__ __attribute__((aligned(16))) float sG[kC * P];   // g, then k 2^(Ge - G); v for U
  __shared__ __attribute__((aligned(16))) float sL[kC * P];   // L; (beta v)^T for U
  __shared__ __attribute__((aligned(16))) float sGa[4 * HD], sGe[4 * HD];
  __shared__ float sTmp[768];         // segment sums; the triangular inversion's scratch
  __shared__ float sB[kC];
  __shared__ int sFar[NHALF];         // a diagonal tile of the half decays past the anchor's range
  constexpr int NTH = kPrepThreads;
  static_assert(NTH == 8 * HD && kC == 64, "eight 8-row segments per channel");
  const int t = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63, r16 = l & 15, gq = l >> 4;
  const int H = a.H;
  const int u = blockIdx.x / H, h = blockIdx.x - u * H;
  const ChunkRows cr = chunk_rows(a, u);
  const int64_t ch = static_cast<int64_t>(u) * H + h;
  float* const sT = sQ;
  const int d0 = t & (HD - 1), s8 = wv, tile = wv >> 1;   // this thread's column segment (in row tile `tile`)

  // scores: Aqk (c >= i) to the workspace, L = beta_c Akk (c > i) to LDS,
  // accumulated over the channel halves on the matrix cores, one 16 x 16 tile
  // pair per wave: waves 0..5 the off-diagonal pairs (row tile R > key tile
  // s), waves 6 and 7 two diagonal tiles each.  The decay of a pair is
  // 2^(G_c - Ga_R) 2^(Ga_R - Ge_s) 2^(Ge_s - G_i); the outer factors are <= 1
  // and in the operands, the middle one is <= 1 off the diagonal and, on it,
  // >= 1, up to the tile's decay (pairs whose product would exceed 1 are
  // masked).  A diagonal tile that decays by more than 2^-kDiagAnchorLog2 in a
  // channel of the half takes 2^(G_c - G_i) per element for that half instead
  // (lane (r, gq) forming its own four outputs, rows 4 gq + e, key r), before
  // the operands replace q, k, G.
  const int R_off = (wv < 1) ? 1 : (wv < 3) ? 2 : 3;
  const int sk_off = wv - R_off * (R_off - 1) / 2;
  const int NPAIR = (wv < 6) ? 1 : 2;   // wave-uniform
  auto pair_rs = [&](int pi, int& R, int& sk) {
    if (wv < 6) { R = R_off; sk = sk_off; }
    else { R = 2 * (wv - 6) + pi; sk = R; }
  };
  f4 accA[2], accL[2];
#pragma unroll
  for (int pi = 0; pi < 2; ++pi) accA[pi] = accL[pi] = f4{0.f, 0.f, 0.f, 0.f};
  float kg[NHALF][8];                 // gamma k of this thread's segment
  // the next half's q, k, g and beta, loaded during this half's scores
  InTile<DTQ, D, HD, NTH> nq, nk;
  InTile<GT, D, HD, NTH> ng;
  auto fetch_half = [&](int c0) {
    nq.fetch(a.q, cr.row0, cr.len, H, h, c0);
    nk.fetch(a.k, cr.row0, cr.len, H, h, c0);
    ng.fetch(a.g, cr.row0, cr.len, H, h, c0);
  };
  fetch_half(0);
  float nb = 0.f;
  if (t < NHALF) sFar[t] = 0;
  if (t < kC) nb = ld_beta<DTG>(a.beta, (cr.row0 + (t < cr.len ? t : 0)) * H + h);
#pragma unroll
  for (int hf = 0; hf < NHALF; ++hf) {
    const int c0 = HD * hf;
    if (hf > 0) __syncthreads();      // the previous half's reads are done
    nq.template put<P>(sQ, a.scale);
    nk.template put<P>(sK, 1.f);
    ng.template put<P, ALPHA>(sG, 1.f, cr.len);
    if (hf == 0 && t < kC) sB[t] = (t < cr.len) ? nb : 0.f;
    __syncthreads();
    // G of the segment (log2 units): its prefix, plus the sums of the segments above
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = sG[(8 * s8 + j) * P + d0];
    const float first = x[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) x[j] += x[j - 1];
    sTmp[s8 * HD + d0] = x[7];
    if ((s8 & 1) == 0) sGa[tile * HD + d0] = first;   // (g of the tile's first row, made G below)
    __syncthreads();
    float pre = 0.f, all = 0.f, mid = 0.f, end = 0.f;   // sums above the segment, of the chunk, up to the tile, through it
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      if (m == s8) pre = all;
      if (m == 2 * tile) mid = all;
      all += sTmp[m * HD + d0];
      if (m == 2 * tile + 1) end = all;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = (x[j] + pre) * kLog2e;
    const float ga = (mid + sGa[tile * HD + d0]) * kLog2e;
    const float ge = (s8 & 1) ? x[7] : end * kLog2e;
    const float gz = (s8 == 7) ? x[7] : all * kLog2e;
    if (__any(ga - ge > kDiagAnchorLog2) && l == 0) sFar[hf] = 1;
    __syncthreads();                  // (also: sGa's first rows are read)
    if ((s8 & 1) == 0) sGa[tile * HD + d0] = ga;
    else sGe[tile * HD + d0] = ge;
    unsigned far = 0;   // diagonal tiles of this wave done per element (bit pi)
    if (sFar[hf] != 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) sG[(8 * s8 + j) * P + d0] = x[j];
      __syncthreads();
      if (wv >= 6) {
#pragma unroll
        for (int pi = 0; pi < 2; ++pi) {
          const int a0 = 16 * (2 * (wv - 6) + pi), i = a0 + r16;
          if (!__any(sG[a0 * P + l] - sG[(a0 + 15) * P + l] > kDiagAnchorLog2)) continue;
          far |= 1u << pi;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int c = a0 + 4 * gq + e;
            if (r16 > 4 * gq + e) continue;   // above the diagonal (masked below)
            float sA = 0.f, sL4 = 0.f;
#pragma unroll 2
            for (int d4 = 0; d4 < HD; d4 += 4) {
              const f4 kI = *reinterpret_cast<const f4*>(&sK[i * P + d4]), gI = *reinterpret_cast<const f4*>(&sG[i * P + d4]);
              const f4 gC = *reinterpret_cast<const f4*>(&sG[c * P + d4]), qC = *reinterpret_cast<const f4*>(&sQ[c * P + d4]);
              const f4 kC4 = *reinterpret_cast<const f4*>(&sK[c * P + d4]);
#pragma unroll
              for (int y = 0; y < 4; ++y) {
                const float ki = kI[y] * ex2(gC[y] - gI[y]);
                sA = fmaf(qC[y], ki, sA);
                sL4 = fmaf(kC4[y], ki, sL4);
              }
            }
            accA[pi][e] += sA;
            accL[pi][e] += sL4;
          }
        }
      }
      __syncthreads();
    }
    {
      // the segment's operands over q, k, g in LDS; gamma q, lambda k stored
      const float fa = ex2(ga), fe = ex2(gz - ge);
      h4 vq[2], vl[2];
      f4 wq[2], wl[2];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int o = (8 * s8 + j) * P + d0;
        const float up = ex2(x[j] - ga), q = sQ[o] * up, k = sK[o], ku = k * up, kd = k * ex2(ge - x[j]);
        sQ[o] = q;
        sK[o] = ku;
        sG[o] = kd;
        kg[hf][j] = ku * fa;
        wq[j >> 2][j & 3] = q * fa;
        wl[j >> 2][j & 3] = kd * fe;
        vq[j >> 2][j & 3] = static_cast<_Float16>(wq[j >> 2][j & 3]);
        vl[j >> 2][j & 3] = static_cast<_Float16>(wl[j >> 2][j & 3]);
      }
      if constexpr (EF == 0) {
        // row-major
        const int64_t base = (ch * kC + 8 * s8) * D + c0 + d0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          a.QG[base + j * D] = wq[j >> 2][j & 3];
          a.KL[base + j * D] = wl[j >> 2][j & 3];
        }
      } else {
        // (gamma q)^T and (lambda k)^T fragments (the slot order of
        // kda_internal.h): channel tile dt, K step s8 / 4, half (s8 % 4) / 2,
        // row groups 2 (s8 % 2) and the next
        const int64_t f = ((ch * (D / 16) + (c0 + d0) / 16) * 2 + (s8 >> 2)) * 64 + (d0 & 15) + 32 * (s8 & 1);
        const int hh = 4 * ((s8 >> 1) & 1);
#pragma unroll
        for (int g2 = 0; g2 < 2; ++g2) {
          *reinterpret_cast<h4*>(static_cast<_Float16*>(a.FQ) + (f + 16 * g2) * 8 + hh) = vq[g2];
          *reinterpret_cast<h4*>(static_cast<_Float16*>(a.FLT) + (f + 16 * g2) * 8 + hh) = vl[g2];
        }
      }
      if (s8 == 7) a.GCV[ch * D + c0 + d0] = ex2(gz);
    }
    __syncthreads();
    if constexpr (EF != 0) {
      // lambda k fragments (rows as M): row tile tt, K step hi over the half's
      // channels, one lane fragment per thread
      static_assert(NTH == 512 && HD == 64, "one lambda k lane fragment per thread");
      const int hi = wv & 1, tt = wv >> 1, row = 16 * tt + r16;
      h8 v;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int dl = 32 * hi + 4 * gq + 16 * p;
        const f4 kd = *reinterpret_cast<const f4*>(&sG[row * P + dl]);
        const f4 ge4 = *reinterpret_cast<const f4*>(&sGe[tt * HD + dl]), gz4 = *reinterpret_cast<const f4*>(&sGe[3 * HD + dl]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * p + e] = static_cast<_Float16>(kd[e] * ex2(gz4[e] - ge4[e]));
      }
      *reinterpret_cast<h8*>(static_cast<_Float16*>(a.FL) + (((ch * 4 + tt) * (D / 32) + (c0 >> 5) + hi) * 64 + l) * 8) = v;
    }
    if (hf + 1 < NHALF) fetch_half(c0 + HD);
#pragma unroll
    for (int pi = 0; pi < 2; ++pi) {
      if (pi >= NPAIR) break;
      int R, sk;
      pair_rs(pi, R, sk);
      if (R == sk && (far >> pi & 1)) continue;
      const int ro = (16 * R + r16) * P + 4 * gq, ko = (16 * sk + r16) * P + 4 * gq;
#pragma unroll
      for (int j = 0; j < HD / 16; ++j) {
        const f4 qu = *reinterpret_cast<const f4*>(&sQ[ro + 16 * j]), ku = *reinterpret_cast<const f4*>(&sK[ro + 16 * j]);
        f4 kd = *reinterpret_cast<const f4*>(&sG[ko + 16 * j]);
        const f4 ga4 = *reinterpret_cast<const f4*>(&sGa[R * HD + 16 * j + 4 * gq]);
        const f4 ge4 = *reinterpret_cast<const f4*>(&sGe[sk * HD + 16 * j + 4 * gq]);
#pragma unroll
        for (int e = 0; e < 4; ++e) kd[e] *= ex2(ga4[e] - ge4[e]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          accA[pi] = mfma4(qu[e], kd[e], accA[pi]);
          accL[pi] = mfma4(ku[e], kd[e], accL[pi]);
        }
      }
    }
  }
  // the first W/U pass's v half, loaded until the scores are out of LDS
  InTile<DTQ, D, HD, NTH> iv;
  iv.fetch(a.v, cr.row0, cr.len, H, h, 0);
  const int64_t aq0 = ch * kC * kC;
#pragma unroll
  for (int pi = 0; pi < 2; ++pi) {
    if (pi >= NPAIR) break;
    int R, sk;
    pair_rs(pi, R, sk);
    const int a0 = 16 * R, i = 16 * sk + r16;
    f4 vA;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = a0 + 4 * gq + e;
      const bool diag = R == sk;
      vA[e] = (!diag || r16 <= 4 * gq + e) ? accA[pi][e] : 0.f;   // Aqk: i <= c
      if constexpr (EF == 0) ws_st<EF>(a.AQ, aq0 + c * kC + i, vA[e]);
      sL[c * P + i] = (!diag || r16 < 4 * gq + e) ? accL[pi][e] * sB[c] : 0.f;   // L: i < c
    }
    if constexpr (EF != 0)   // Aqk^T fragment (key tile sk, K step R / 2), half R % 2
      *reinterpret_cast<uint2*>(static_cast<u16*>(a.FA) + ((ch * 6 + fa_frag(sk, R >> 1)) * 64 + l) * 8 +
                                4 * (R & 1)) = pack_f16x4(vA);
  }
  if constexpr (EF == 0) {
    // blocks above the diagonal: zero
    for (int e = t; e < 6 * 256; e += NTH) {
      const int blk = e >> 8, rc = (e >> 4) & 15, ri = e & 15;
      const int R = (blk < 3) ? 0 : (blk < 5) ? 1 : 2;             // (0,1) (0,2) (0,3) (1,2) (1,3) (2,3)
      const int sk = (blk < 3) ? blk + 1 : (blk < 5) ? blk - 1 : 3;
      ws_st<EF>(a.AQ, aq0 + (16 * R + rc) * kC + 16 * sk + ri, 0.f);
    }
  } else {
    // the zero halves of the stored Aqk^T fragments: key tile 1 against row
    // tile 0, key tile 3 against row tile 2
    if (t < 128)
      *reinterpret_cast<uint2*>(static_cast<u16*>(a.FA) +
                                ((ch * 6 + (t < 64 ? fa_frag(1, 0) : fa_frag(3, 1))) * 64 + (t & 63)) * 8) =
          uint2{0u, 0u};
  }
  __syncthreads();

  // W = T (beta gamma k), U = T (beta v) on the matrix cores, per half of
  // their columns, the right sides transposed in LDS so both operands are
  // 16-byte reads of four K values; wave wv owns row tile wv / 2 and column
  // tiles (wv % 2) HD/32 + q of the half.  The first half's beta gamma k and v
  // go to LDS here, T = (I + L)^-1 goes into sQ's buffer.
  float bs[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) bs[j] = sB[8 * s8 + j];
  auto put_col = [&](float* dst, const float (&y)[8]) {   // beta times the segment, transposed
    float* o = dst + d0 * P + 8 * s8;
    *reinterpret_cast<f4*>(o) = f4{bs[0] * y[0], bs[1] * y[1], bs[2] * y[2], bs[3] * y[3]};
    *reinterpret_cast<f4*>(o + 4) = f4{bs[4] * y[4], bs[5] * y[5], bs[6] * y[6], bs[7] * y[7]};
  };
  put_col(sK, kg[0]);
  iv.template put<P>(sG, 1.f);
  if constexpr (NHALF > 1) iv.fetch(a.v, cr.row0, cr.len, H, h, HD);   // the next half's, during the inversion
  invert_unit_lower64<P, NTH>(sL, sT, sTmp);
  {
    static_assert(kC * kC == 8 * NTH, "eight entries of T per thread");
    const int c = t >> 3, i0 = 8 * (t & 7);
    const f4 lo = *reinterpret_cast<const f4*>(sT + c * P + i0), hi = *reinterpret_cast<const f4*>(sT + c * P + i0 + 4);
    const int64_t o = ch * kC * kC + c * kC + i0;
    ws_st4<EF>(a.TM, o, make_float4(lo[0], lo[1], lo[2], lo[3]));
    ws_st4<EF>(a.TM, o + 4, make_float4(hi[0], hi[1], hi[2], hi[3]));
  }
#pragma unroll
  for (int hf = 0; hf < NHALF; ++hf) {
    const int c0 = HD * hf;
    if (hf > 0) {
      __syncthreads();                // the previous half's products are done
      put_col(sK, kg[hf]);
    }
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = sG[(8 * s8 + j) * P + d0];
    put_col(sL, y);
    __syncthreads();
    if (hf + 1 < NHALF) iv.template put<P>(sG, 1.f);
    constexpr int NDT = HD / 32;
    const int mt = wv >> 1, dg = wv & 1;
    f4 accW[NDT], accU[NDT];
#pragma unroll
    for (int q = 0; q < NDT; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) accW[q][e] = accU[q][e] = 0.f;
    // T[c][i] is zero for i > c: row tile mt needs the K blocks up to its own
    for (int j = 0; j <= mt; ++j) {
      const f4 at = *reinterpret_cast<const f4*>(&sT[(16 * mt + r16) * P + 16 * j + 4 * gq]);
      f4 bk[NDT], bv[NDT];
#pragma unroll
      for (int q = 0; q < NDT; ++q) {
        const int o = (16 * (dg * NDT + q) + r16) * P + 16 * j + 4 * gq;
        bk[q] = *reinterpret_cast<const f4*>(&sK[o]);
        bv[q] = *reinterpret_cast<const f4*>(&sL[o]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int q = 0; q < NDT; ++q) {
          accW[q] = mfma4(at[e], bk[q][e], accW[q]);
          accU[q] = mfma4(at[e], bv[q][e], accU[q]);
        }
    }
    const int64_t wu0 = ch * kC * D + c0;
#pragma unroll
    for (int q = 0; q < NDT; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int o = (16 * mt + 4 * gq + e) * D + 16 * (dg * NDT + q) + r16;
        if constexpr (EF == 0) ws_st<EF>(a.WM, wu0 + o, accW[q][e]);
        a.UM[wu0 + o] = accU[q][e];
      }
    if constexpr (EF != 0) {
      // W^T fragments: channel tile of column tile q, K step mt / 2, half mt % 2;
      // W fragments (rows x channels) of K step c0 / 32 + dg: the D-layout tile
      // read as an A fragment is W^T, and its product with the identity lands
      // row r of W, channels 4 gq .. 4 gq + 3 of the tile, in lane (r, gq)
      static_assert(NDT == 2, "two column tiles per wave: one 32-channel K step");
      h4 ident;
#pragma unroll
      for (int i = 0; i < 4; ++i) ident[i] = static_cast<_Float16>((4 * gq + i == r16) ? 1.f : 0.f);
      h8 wn;
#pragma unroll
      for (int q = 0; q < NDT; ++q) {
        const int dt = (c0 >> 4) + dg * NDT + q;
        const uint2 w16 = pack_f16x4(accW[q]);
        *reinterpret_cast<uint2*>(static_cast<u16*>(a.FW) + (((ch * (D / 16) + dt) * 2 + (mt >> 1)) * 64 + l) * 8 +
                                  4 * (mt & 1)) = w16;
        const f4 tr = mma16(f4{0.f, 0.f, 0.f, 0.f}, __builtin_bit_cast(h4, w16), ident);
#pragma unroll
        for (int i = 0; i < 4; ++i) wn[4 * q + i] = static_cast<_Float16>(tr[i]);
      }
      *reinterpret_cast<h8*>(static_cast<_Float16*>(a.FWN) + (((ch * 4 + mt) * (D / 32) + (c0 >> 5) + dg) * 64 + l) * 8) = wn;
    }
  }
}

// ---------------------------------------------------------------------------
// The scans run their products on the bf16 matrix cores as hi/lo triples
// (v_mfma_f32_16x16x32_bf16): lane (r = l & 15, gq = l >> 4) supplies
// A[r][32 s + 8 gq .. + 7] and B[32 s + 8 gq .. + 7][r] of K block s and
// holds D rows 4 gq + i, column r.  Eight waves per workgroup; the 32-column
// state slice is (D/16) x 2 tiles in accumulators, D/64 tiles per wave; the
// [64][32] results of a chunk are 8 tiles, one per wave.  Operands sit in LDS
// as hi and lo bf16 planes with the K index contiguous, so each fragment is
// one 16-byte read.
// ---------------------------------------------------------------------------
constexpr int kPB = 48;   // fp32 pitch of the forward scan's [64][32] U slice

// x0, x1 -> packed bf16 pairs hi (round to nearest even) and lo = bf16(x - hi)
__device__ __forceinline__ void split2_bf16(float x0, float x1, unsigned& h, unsigned& l) {
  h = pack_bf16x2(x0, x1);
  l = pack_bf16x2(x0 - __uint_as_float(h << 16), x1 - __uint_as_float(h & 0xFFFF0000u));
}
// hi * hi + hi * lo + lo * hi of one 32-wide K block on the bf16 matrix cores
// (products exact, sums fp32; the dropped lo * lo term and the rounding of lo
// leave about 2^-16 of each product)
__device__ __forceinline__ f4 mma3_bf16(f4 acc, const b8& ah, const b8& al, const b8& bh, const b8& bl) {
  acc = mma32_bf16(acc, ah, bh);
  acc = mma32_bf16(acc, ah, bl);
  return mma32_bf16(acc, al, bh);
}

// A fetched fp32 tile into LDS as hi / lo bf16 planes (row pitch PB bf16).
template <int PB, int ROWS, int COLS, int NTH, int ET>
__device__ __forceinline__ void put_hl(const Tile<ROWS, COLS, NTH, ET>& tl, __bf16* h, __bf16* l) {
  typedef Tile<ROWS, COLS, NTH, ET> TT;
#pragma unroll
  for (int p = 0; p < TT::PER; ++p) {
    const int e = fresh_tid() + p * NTH;
    if (TT::N % NTH == 0 || e < TT::N) {
      const int row = e / TT::V, c4 = e - row * TT::V;
      const float4 x = tl.get(p);
      uint2 hh, ll;
      split2_bf16(x.x, x.y, hh.x, ll.x);
      split2_bf16(x.z, x.w, hh.y, ll.y);
      *reinterpret_cast<uint2*>(&h[row * PB + 4 * c4]) = hh;
      *reinterpret_cast<uint2*>(&l[row * PB + 4 * c4]) = ll;
    }
  }
}
template <int PB, int DT, int D, int COLS, int NTH>
__device__ __forceinline__ void put_hl(const InTile<DT, D, COLS, NTH>& tl, __bf16* h, __bf16* l) {
  typedef InTile<DT, D, COLS, NTH> TT;
#pragma unroll
  for (int p = 0; p < TT::PER; ++p) {
    const int e = fresh_tid() + p * NTH;
    if (TT::N % NTH == 0 || e < TT::N) {
      const int r = e / TT::V, c8 = e - r * TT::V;
      float x[8];
      if constexpr (DT == 0) {
        const uint4 a = tl.w[2 * p], b = tl.w[2 * p + 1];
        x[0] = __uint_as_float(a.x); x[1] = __uint_as_float(a.y); x[2] = __uint_as_float(a.z); x[3] = __uint_as_float(a.w);
        x[4] = __uint_as_float(b.x); x[5] = __uint_as_float(b.y); x[6] = __uint_as_float(b.z); x[7] = __uint_as_float(b.w);
      } else {
        const f4 lo = unpack4<DT>(make_uint2(tl.w[p].x, tl.w[p].y)), hi = unpack4<DT>(make_uint2(tl.w[p].z, tl.w[p].w));
#pragma unroll
        for (int q = 0; q < 4; ++q) { x[q] = lo[q]; x[4 + q] = hi[q]; }
      }
      uint4 hh, ll;
      split2_bf16(x[0], x[1], hh.x, ll.x);
      split2_bf16(x[2], x[3], hh.y, ll.y);
      split2_bf16(x[4], x[5], hh.z, ll.z);
      split2_bf16(x[6], x[7], hh.w, ll.w);
      *reinterpret_cast<uint4*>(&h[r * PB + 8 * c8]) = hh;
      *reinterpret_cast<uint4*>(&l[r * PB + 8 * c8]) = ll;
    }
  }
}

// A [64][COLS] tile (element type ET) fetched for a transposed store into
// hi / lo bf16 planes [COLS][64] (the source row index becomes the contiguous
// K index): thread t holds rows 2 rp and 2 rp + 1 (rp = t % 32) of the
// four-column groups t / 32 + (NTH / 32) j, so each transposed row is written
// as packed row pairs, consecutive lanes at consecutive words.
template <int COLS, int NTH, int ET = 0>
struct TTile {
  static constexpr int G = NTH / 32;
  static constexpr int PER = (COLS / 4) / G;
  static_assert(NTH % 32 == 0 && (COLS / 4) % G == 0, "transposed tile mapping");
  typedef typename WsPiece<ET>::t Piece;
  Piece r[PER][2];
  __device__ __forceinline__ void fetch(const void* src, int src_ld, int col0) {
    const int tf = fresh_tid(), rp = tf & 31, cg = tf >> 5;
#pragma unroll
    for (int j = 0; j < PER; ++j)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        const int64_t i = static_cast<int64_t>(2 * rp + y) * src_ld + col0 + 4 * (cg + G * j);
        if constexpr (ET == 0) r[j][y] = *reinterpret_cast<const float4*>(static_cast<const float*>(src) + i);
        else r[j][y] = *reinterpret_cast<const uint2*>(static_cast<const u16*>(src) + i);
      }
  }
  // columns HW hp .. HW hp + HW - 1 row-major into hi / lo planes of pitch PB
  // (a [rows][HW] pass of a product over the columns; PER == 1)
  template <int PB, int HW>
  __device__ __forceinline__ void put_rows_hl(int hp, __bf16* h, __bf16* l) const {
    static_assert(PER == 1 && HW % 4 == 0, "one column group per thread");
    const int tf = fresh_tid(), rp = tf & 31, cg = tf >> 5;
    if (cg / (HW / 4) != hp) return;
    const int c = 4 * (cg - hp * (HW / 4));
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const float4 x = ws_unpack<ET>(r[0][y]);
      uint2 hh, ll;
      split2_bf16(x.x, x.y, hh.x, ll.x);
      split2_bf16(x.z, x.w, hh.y, ll.y);
      *reinterpret_cast<uint2*>(&h[(2 * rp + y) * PB + c]) = hh;
      *reinterpret_cast<uint2*>(&l[(2 * rp + y) * PB + c]) = ll;
    }
  }
  template <int PB>
  __device__ __forceinline__ void put_hl(__bf16* h, __bf16* l) const {
    const int tf = fresh_tid(), rp = tf & 31, cg = tf >> 5;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int c4 = 4 * (cg + G * j);
      const float4 y0 = ws_unpack<ET>(r[j][0]), y1 = ws_unpack<ET>(r[j][1]);
      const float x0[4] = {y0.x, y0.y, y0.z, y0.w};
      const float x1[4] = {y1.x, y1.y, y1.z, y1.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        unsigned hh, ll;
        split2_bf16(x0[e], x1[e], hh, ll);
        *reinterpret_cast<unsigned*>(&h[(c4 + e) * PB + 2 * rp]) = hh;
        *reinterpret_cast<unsigned*>(&l[(c4 + e) * PB + 2 * rp]) = ll;
      }
    }
  }
};

// forward state scan of one (chain, 32-column slice): S_in and v~ per chunk.
// The products run as bf16 hi/lo triples (v_mfma_f32_16x16x32_bf16, lane
// (r, gq) holding K values 8 gq .. 8 gq + 7 of each 32-wide block): W and
// (lambda k)^T, the state slice S^T and v~^T are kept in LDS as hi and lo
// bf16 planes with the K index contiguous, so each fragment is one 16-byte
// read.  The state itself stays fp32 in the accumulators.  (fp32 inputs; with
// 16-bit ones fscan16_block and rscan16_block run.)
template <int D>
struct alignas(16) FscanLds {
  static constexpr int PW = D + 8;     // bf16 pitch of rows whose K index is a channel
  static constexpr int PK = kC + 8;    // bf16 pitch of rows whose K index is a chunk row
  __bf16 Wh[kC * PW], Wl[kC * PW];     // W [64][D]
  __bf16 Kh[D * PK], Kl[D * PK];       // (lambda k)^T [D][64]
  __bf16 Sh[32 * PW], Sl[32 * PW];     // S^T [32][D]
  __bf16 Vh[32 * PK], Vl[32 * PK];     // v~^T [32][64]
  float U[kC * kPB], GC[D];
};

template <int D>
__device__ __forceinline__ void fscan_block(const BwdArgs& a, int block, FscanLds<D>& L) {
  constexpr int NTH = ScanThreads<D>::value;
  constexpr int NS = D / 32;
  constexpr int NST = (D / 8) / (NTH / 64);   // state tiles per wave (D / 8 tiles of the 32-column slice)
  static_assert(NST >= 1, "at least one state tile per wave");
  constexpr int PW = FscanLds<D>::PW, PK = FscanLds<D>::PK;
  __bf16 *const sWh = L.Wh, *const sWl = L.Wl, *const sKh = L.Kh, *const sKl = L.Kl;
  __bf16 *const sSh = L.Sh, *const sSl = L.Sl, *const sVh = L.Vh, *const sVl = L.Vl;
  float *const sU = L.U, *const sGC = L.GC;
  const int t = threadIdx.x, wv = t >> 6, l = t & 63, r = l & 15, gq = l >> 4;
  const int H = a.H;
  int chain, split;
  if (!scan_slot<NS>(block, a.B * H, chain, split)) return;   // uniform per workgroup
  const int b = chain / H, h = chain - b * H;
  const int c0 = 32 * split;
  const int mt = wv >> 1, ct = wv & 1;                  // this wave's v~ tile (waves 0-7: 8 tiles)
  const bool vt_wave = wv < 8;
  int rt[NST], cs[NST];                                 // this wave's state tiles
#pragma unroll
  for (int q = 0; q < NST; ++q) { rt[q] = (wv * NST + q) >> 1; cs[q] = (wv * NST + q) & 1; }
  f4 S[NST];
#pragma unroll
  for (int q = 0; q < NST; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      S[q][i] = (a.h0 != nullptr)
                    ? a.h0[(static_cast<int64_t>(chain) * D + 16 * rt[q] + 4 * gq + i) * D + c0 + 16 * cs[q] + r]
                    : 0.f;
  // chunk n's W, lambda*k and U slice are loaded into registers during
  // chunk n-1's arithmetic
  typedef Tile<kC, D, NTH> TD;
  TD tW;
  Tile<kC, 32, NTH> tU;
  // lambda*k, fetched for its transposed store: thread t holds rows 2 rp and
  // 2 rp + 1 (rp = t % 32) of the column groups KCG j + t / 32, so each
  // transposed row is written as packed row pairs, consecutive lanes at
  // consecutive words
  constexpr int KCG = NTH / 32;                    // column groups per pass
  constexpr int KPER = (D / 4) / KCG;              // float4 column groups per thread
  static_assert((D / 4) % KCG == 0, "lambda*k column groups");
  float4 kq[KPER][2];
  const int rp = t & 31, cg = t >> 5;
  float pgc;   // gamma_C of the chunk, loaded with its operands (every thread; t < D stores it)
  auto fetch = [&](int n) {
    const int64_t ch = (static_cast<int64_t>(b) * a.NT + n) * H + h;
    pgc = a.GCV[ch * D + (t & (D - 1))];
    tW.fetch(a.WM + ch * kC * D, D, 0);
    const float* KLp = a.KL + ch * kC * D;
#pragma unroll
    for (int j = 0; j < KPER; ++j)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        const int i = (2 * rp + y) * D + 4 * (cg + KCG * j);
        kq[j][y] = *reinterpret_cast<const float4*>(KLp + i);
      }
    tU.fetch(a.UM + ch * kC * D, D, c0);
  };
  if (a.NT > 0) fetch(0);
  for (int n = 0; n < a.NT; ++n) {
    const int64_t ch = (static_cast<int64_t>(b) * a.NT + n) * H + h;
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      const int m0 = 16 * rt[q] + 4 * gq, col = 16 * cs[q] + r;
#pragma unroll
      for (int i = 0; i < 4; ++i) a.SI[ch * D * D + (m0 + i) * D + c0 + col] = S[q][i];
      uint2 hh, ll;
      split2_bf16(S[q][0], S[q][1], hh.x, ll.x);
      split2_bf16(S[q][2], S[q][3], hh.y, ll.y);
      *reinterpret_cast<uint2*>(&sSh[col * PW + m0]) = hh;
      *reinterpret_cast<uint2*>(&sSl[col * PW + m0]) = ll;
    }
    // W row-major and lambda*k transposed, as hi / lo planes
#pragma unroll
    for (int p = 0; p < TD::PER; ++p) {
      const int e = t + p * NTH;
      const int row = e / TD::V, c4 = e - row * TD::V;
      const float4 w = tW.get(p);
      uint2 hh, ll;
      split2_bf16(w.x, w.y, hh.x, ll.x);
      split2_bf16(w.z, w.w, hh.y, ll.y);
      *reinterpret_cast<uint2*>(&sWh[row * PW + 4 * c4]) = hh;
      *reinterpret_cast<uint2*>(&sWl[row * PW + 4 * c4]) = ll;
    }
#pragma unroll
    for (int j = 0; j < KPER; ++j) {
      const int ch4 = 4 * (cg + KCG * j);
      const float4 y0 = kq[j][0], y1 = kq[j][1];
      const float k0[4] = {y0.x, y0.y, y0.z, y0.w};
      const float k1[4] = {y1.x, y1.y, y1.z, y1.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        unsigned hh, ll;
        split2_bf16(k0[e], k1[e], hh, ll);     // rows 2 rp, 2 rp + 1 of channel ch4 + e
        *reinterpret_cast<unsigned*>(&sKh[(ch4 + e) * PK + 2 * rp]) = hh;
        *reinterpret_cast<unsigned*>(&sKl[(ch4 + e) * PK + 2 * rp]) = ll;
      }
    }
    tU.template put<kPB>(sU);
    if (t < D) sGC[t] = pgc;
    if (n + 1 < a.NT) fetch(n + 1);
    __syncthreads();
    // v~ = U - W S (two accumulation chains over the D / 32 K blocks)
    if (vt_wave) {
      f4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < D / 32; ++kb) {
        const int ka = (16 * mt + r) * PW + 32 * kb + 8 * gq, kbb = (16 * ct + r) * PW + 32 * kb + 8 * gq;
        f4& acc = (kb & 1) ? acc1 : acc0;
        const b8 ah = *reinterpret_cast<const b8*>(&sWh[ka]), al = *reinterpret_cast<const b8*>(&sWl[ka]);
        const b8 bh = *reinterpret_cast<const b8*>(&sSh[kbb]), bl = *reinterpret_cast<const b8*>(&sSl[kbb]);
        acc = mma3_bf16(acc, ah, al, bh, bl);
      }
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * mt + 4 * gq + i, col = 16 * ct + r;
        v[i] = sU[row * kPB + col] - (acc0[i] + acc1[i]);
        a.VT[ch * kC * D + row * D + c0 + col] = v[i];
      }
      uint2 hh, ll;
      split2_bf16(v[0], v[1], hh.x, ll.x);
      split2_bf16(v[2], v[3], hh.y, ll.y);
      *reinterpret_cast<uint2*>(&sVh[(16 * ct + r) * PK + 16 * mt + 4 * gq]) = hh;
      *reinterpret_cast<uint2*>(&sVl[(16 * ct + r) * PK + 16 * mt + 4 * gq]) = ll;
    }
    __syncthreads();
    // S <- gamma_C S + (lambda k)^T v~
#pragma unroll
    for (int q = 0; q < NST; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[q][i] *= sGC[16 * rt[q] + 4 * gq + i];
#pragma unroll
    for (int kb = 0; kb < kC / 32; ++kb)
#pragma unroll
      for (int q = 0; q < NST; ++q) {
        const int ka = (16 * rt[q] + r) * PK + 32 * kb + 8 * gq, kbb = (16 * cs[q] + r) * PK + 32 * kb + 8 * gq;
        S[q] = mma3_bf16(S[q], *reinterpret_cast<const b8*>(&sKh[ka]), *reinterpret_cast<const b8*>(&sKl[ka]),
                         *reinterpret_cast<const b8*>(&sVh[kbb]), *reinterpret_cast<const b8*>(&sVl[kbb]));
      }
    __syncthreads();
  }
}

// reverse scan of one (chain, 32-column slice): dS per chunk, dv~, dh0.
// The products run as bf16 hi/lo triples, as in the forward scan: lambda k
// and the state cotangent slice dS^T with the channel as the K index; Aqk^T,
// do^T, (gamma q)^T, W^T and (-dv~)^T with the chunk row as the K index
// (transposed stores of row pairs).  dS itself stays fp32 in the accumulators.
//
// A chunk step has three phases between workgroup barriers, and every
// operand has LDS of its own, so each is staged one phase or more before it
// is read, in the shadow of the products:
//   A  store dS, stage it as hi / lo planes; dS <- gamma_C dS + (gamma q)^T do
//      (everything it reads was staged during the previous chunk);
//   B  dv~ = (lambda k) dS + Aqk^T do on waves 0-7, then every wave stages
//      W^T of this chunk (read in C) and loads W of the next one;
//   C  dS <- dS - W^T dv~; every wave stages lambda k, Aqk^T, do^T,
//      (gamma q)^T and gamma_C of the next chunk (read in its A and B) and
//      loads the one after.
template <int D>
struct alignas(16) RscanLds {
  static constexpr int PW = D + 8;     // bf16 pitch of rows whose K index is a channel
  static constexpr int PK = kC + 8;    // bf16 pitch of rows whose K index is a chunk row
  __bf16 Lh[kC * PW], Ll[kC * PW];     // lambda k [64][D]
  __bf16 Ah[kC * PK], Al[kC * PK];     // Aqk^T [64][64]
  __bf16 Qh[D * PK], Ql[D * PK];       // (gamma q)^T [D][64]
  __bf16 Wh[D * PK], Wl[D * PK];       // W^T [D][64]
  __bf16 Sh[32 * PW], Sl[32 * PW];     // dS^T [32][D]
  __bf16 Oh[32 * PK], Ol[32 * PK];     // do^T [32][64]
  __bf16 Vh[32 * PK], Vl[32 * PK];     // (-dv~)^T [32][64]
  float GC[D];
};

template <int D, int DO>
__device__ __forceinline__ void rscan_block(const BwdArgs& a, int block, RscanLds<D>& L) {
  constexpr int NTH = ScanThreads<D>::value;
  constexpr int NS = D / 32;
  constexpr int NST = (D / 8) / (NTH / 64);
  static_assert(NST >= 1, "at least one state tile per wave");
  constexpr int PW = RscanLds<D>::PW, PK = RscanLds<D>::PK;
  __bf16 *const sLh = L.Lh, *const sLl = L.Ll, *const sAh = L.Ah, *const sAl = L.Al;
  __bf16 *const sQh = L.Qh, *const sQl = L.Ql, *const sWh = L.Wh, *const sWl = L.Wl;
  __bf16 *const sSh = L.Sh, *const sSl = L.Sl, *const sOh = L.Oh, *const sOl = L.Ol;
  __bf16 *const sVh = L.Vh, *const sVl = L.Vl;
  float* const sGC = L.GC;
  const int t = threadIdx.x, wv = t >> 6, l = t & 63, r = l & 15, gq = l >> 4;
  const int H = a.H;
  int chain, split;
  if (!scan_slot<NS>(block, a.B * H, chain, split)) return;   // uniform per workgroup
  const int b = chain / H, h = chain - b * H;
  const int c0 = 32 * split;
  const int mt = wv >> 1, ct = wv & 1;                  // this wave's dv~ tile (waves 0-7: 8 tiles)
  const bool vt_wave = wv < 8;
  const int mts = __builtin_amdgcn_readfirstlane(mt);
  int rt[NST], cs[NST];
#pragma unroll
  for (int q = 0; q < NST; ++q) { rt[q] = (wv * NST + q) >> 1; cs[q] = (wv * NST + q) & 1; }
  f4 dS[NST];
#pragma unroll
  for (int q = 0; q < NST; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      dS[q][i] = (a.dht != nullptr)
                     ? a.dht[(static_cast<int64_t>(chain) * D + 16 * rt[q] + 4 * gq + i) * D + c0 + 16 * cs[q] + r]
                     : 0.f;
  // Operands in registers between their loads and their staging, one set
  // each: a set is reloaded right after it is staged, so every load has a
  // whole chunk step to arrive.  The do slice is held as loaded (raw words),
  // so that no wait falls at its load.
  Tile<kC, D, NTH> tL;
  TTile<kC, kScanThreads> tA;   // threads t < kScanThreads
  TTile<D, NTH> tQ, tW;
  const bool a_thread = t < kScanThreads;
  float pgc;   // gamma_C of the chunk (every thread; t < D stages it)
  // do^T of the slice, spread over every thread: thread t holds rows 2 rp,
  // 2 rp + 1 of the DCPT columns c0 + DCPT cg .. (consecutive threads at
  // consecutive columns; rows past the chunk's end are loaded from row 0 and
  // zeroed where staged), as raw words
  constexpr int DCPT = (kC * 32) / 2 / NTH;   // columns per thread
  constexpr int DCG = 32 / DCPT;              // column groups
  static_assert(DCPT >= 1 && DCPT <= 2 && DCG * DCPT == 32 && 2 * DCG * 32 == 2 * NTH, "do slice mapping");
  uint32_t pdo[2][DCPT];
  const int dcg = t % DCG, drp = t / DCG;
  auto do_val = [&](uint32_t w) -> float {
    if constexpr (DO == 0) return __uint_as_float(w);
    else if constexpr (DO == 1) return __uint_as_float(w << 16);
    else return f16bits_to_f32(static_cast<u16>(w));
  };
  auto chead = [&](int n) { return (static_cast<int64_t>(b) * a.NT + n) * H + h; };
  auto fetch_a = [&](int n) {   // lambda k, Aqk, gamma q, gamma_C and do of chunk n
    const int u = b * a.NT + n;
    const int64_t ch = chead(n);
    tL.fetch(a.KL + ch * kC * D, D, 0);
    if (a_thread) tA.fetch(a.AQ + ch * kC * kC, kC, 0);
    tQ.fetch(a.QG + ch * kC * D, D, 0);
    pgc = a.GCV[ch * D + (t & (D - 1))];
    const ChunkRows crn = chunk_rows(a, u);
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int row = 2 * drp + y;
      const int64_t i = ((crn.row0 + (row < crn.len ? row : 0)) * H + h) * D + c0 + DCPT * dcg;
#pragma unroll
      for (int e = 0; e < DCPT; ++e) {
        if constexpr (DO == 0) pdo[y][e] = static_cast<const uint32_t*>(a.dout)[i + e];
        else pdo[y][e] = static_cast<const u16*>(a.dout)[i + e];
      }
    }
  };
  auto put_a = [&](int n) {     // ... staged for chunk n
    const ChunkRows crn = chunk_rows(a, b * a.NT + n);
    put_hl<PW>(tL, sLh, sLl);
    if (a_thread) tA.template put_hl<PK>(sAh, sAl);
    tQ.template put_hl<PK>(sQh, sQl);
    const bool ok0 = 2 * drp < crn.len, ok1 = 2 * drp + 1 < crn.len;
#pragma unroll
    for (int e = 0; e < DCPT; ++e) {
      unsigned hh, ll;
      split2_bf16(ok0 ? do_val(pdo[0][e]) : 0.f, ok1 ? do_val(pdo[1][e]) : 0.f, hh, ll);
      *reinterpret_cast<unsigned*>(&sOh[(DCPT * dcg + e) * PK + 2 * drp]) = hh;
      *reinterpret_cast<unsigned*>(&sOl[(DCPT * dcg + e) * PK + 2 * drp]) = ll;
    }
    if (t < D) sGC[t] = pgc;
  };
  if (a.NT > 0) {
    fetch_a(a.NT - 1);
    tW.fetch(a.WM + chead(a.NT - 1) * kC * D, D, 0);
    put_a(a.NT - 1);
    if (a.NT > 1) fetch_a(a.NT - 2);
    __syncthreads();
  }
  for (int n = a.NT - 1; n >= 0; --n) {
    const int64_t ch = chead(n);
    // ---- A: store and stage dS; dS <- gamma_C dS + (gamma q)^T do
#pragma unroll
    for (int q = 0; q < NST; ++q) {
      const int m0 = 16 * rt[q] + 4 * gq, col = 16 * cs[q] + r;
#pragma unroll
      for (int i = 0; i < 4; ++i) a.DS[ch * D * D + (m0 + i) * D + c0 + col] = dS[q][i];
      uint2 hh, ll;
      split2_bf16(dS[q][0], dS[q][1], hh.x, ll.x);
      split2_bf16(dS[q][2], dS[q][3], hh.y, ll.y);
      *reinterpret_cast<uint2*>(&sSh[col * PW + m0]) = hh;
      *reinterpret_cast<uint2*>(&sSl[col * PW + m0]) = ll;
    }
#pragma unroll
    for (int q = 0; q < NST; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) dS[q][i] *= sGC[16 * rt[q] + 4 * gq + i];
#pragma unroll
    for (int kb = 0; kb < kC / 32; ++kb)
#pragma unroll
      for (int q = 0; q < NST; ++q) {
        const int ka = (16 * rt[q] + r) * PK + 32 * kb + 8 * gq, kbb = (16 * cs[q] + r) * PK + 32 * kb + 8 * gq;
        dS[q] = mma3_bf16(dS[q], *reinterpret_cast<const b8*>(&sQh[ka]), *reinterpret_cast<const b8*>(&sQl[ka]),
                          *reinterpret_cast<const b8*>(&sOh[kbb]), *reinterpret_cast<const b8*>(&sOl[kbb]));
      }
    __syncthreads();
    // ---- B: dv~ = (lambda k) dS + Aqk^T do; Aqk[j][m] is zero for j < m,
    // so row tile mt starts at the K block holding row 16 mt
    if (vt_wave) {
      f4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < D / 32; ++kb) {
        const int ka = (16 * mt + r) * PW + 32 * kb + 8 * gq, kbb = (16 * ct + r) * PW + 32 * kb + 8 * gq;
        acc0 = mma3_bf16(acc0, *reinterpret_cast<const b8*>(&sLh[ka]), *reinterpret_cast<const b8*>(&sLl[ka]),
                         *reinterpret_cast<const b8*>(&sSh[kbb]), *reinterpret_cast<const b8*>(&sSl[kbb]));
      }
      for (int kb = mts >> 1; kb < kC / 32; ++kb) {
        const int ka = (16 * mt + r) * PK + 32 * kb + 8 * gq, kbb = (16 * ct + r) * PK + 32 * kb + 8 * gq;
        acc1 = mma3_bf16(acc1, *reinterpret_cast<const b8*>(&sAh[ka]), *reinterpret_cast<const b8*>(&sAl[ka]),
                         *reinterpret_cast<const b8*>(&sOh[kbb]), *reinterpret_cast<const b8*>(&sOl[kbb]));
      }
      float* DVT = a.DVT + ch * kC * D;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = acc0[i] + acc1[i];
        DVT[(16 * mt + 4 * gq + i) * D + c0 + 16 * ct + r] = v[i];
      }
      uint2 hh, ll;
      split2_bf16(-v[0], -v[1], hh.x, ll.x);
      split2_bf16(-v[2], -v[3], hh.y, ll.y);
      *reinterpret_cast<uint2*>(&sVh[(16 * ct + r) * PK + 16 * mt + 4 * gq]) = hh;
      *reinterpret_cast<uint2*>(&sVl[(16 * ct + r) * PK + 16 * mt + 4 * gq]) = ll;
    }
    tW.template put_hl<PK>(sWh, sWl);
    if (n > 0) tW.fetch(a.WM + chead(n - 1) * kC * D, D, 0);
    __syncthreads();
    // ---- C: dS <- dS - W^T dv~; the next chunk's lambda k, Aqk^T, do^T,
    // (gamma q)^T and gamma_C staged while the products run
#pragma unroll
    for (int kb = 0; kb < kC / 32; ++kb)
#pragma unroll
      for (int q = 0; q < NST; ++q) {
        const int ka = (16 * rt[q] + r) * PK + 32 * kb + 8 * gq, kbb = (16 * cs[q] + r) * PK + 32 * kb + 8 * gq;
        dS[q] = mma3_bf16(dS[q], *reinterpret_cast<const b8*>(&sWh[ka]), *reinterpret_cast<const b8*>(&sWl[ka]),
                          *reinterpret_cast<const b8*>(&sVh[kbb]), *reinterpret_cast<const b8*>(&sVl[kbb]));
      }
    if (n > 0) {
      put_a(n - 1);
      if (n > 1) fetch_a(n - 2);
    }
    __syncthreads();
  }
  if (a.dh0 != nullptr) {
#pragma unroll
    for (int q = 0; q < NST; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a.dh0[(static_cast<int64_t>(chain) * D + 16 * rt[q] + 4 * gq + i) * D + c0 + 16 * cs[q] + r] = dS[q][i];
  }
}

// ---------------------------------------------------------------------------
// Reverse scan for 16-bit inputs: one workgroup per (chain, 32-column slice),
// two compute waves (one 16-column value tile each) and four producer waves,
// as the forward's state kernel.  Each compute wave owns its tile's columns of
// dS for every channel, so a chunk step needs no exchange between waves:
//   dv~ = (lambda k) dS' + Aqk^T do,  dS <- gamma_C dS + (gamma q)^T do - W^T dv~
// with the forward-side operands (lambda k, Aqk^T, (gamma q)^T, W^T) as the
// prep kernel's fp16 A fragments, staged by the producers into one of two LDS
// buffers two chunks ahead, and the cotangent operands (dS', do, dv~) as B
// fragments formed in registers.  A cotangent's scale is the caller's, so
// each B column is scaled by a power of two that brings its largest element
// to [2^14, 2^15) and split into fp16 hi + lo (about 22 significant bits,
// fp16's range no limit); each product is two fp16 MFMAs per K step, and the
// column's scale is taken off the accumulator (every lane's D column is its
// own B column).  One barrier per chunk step.
// ---------------------------------------------------------------------------
constexpr int kRsProducers = 4;

template <int D>
struct RsLayout {
  static constexpr int NFL = 4 * (D / 32);         // lambda k fragments (row tile, K step over channels)
  static constexpr int NFA = 6;                    // Aqk^T fragments
  static constexpr int NFQ = 2 * (D / 16);         // (gamma q)^T fragments (channel tile, K step over rows)
  static constexpr int OFF_A = NFL;                // in 1 KiB fragments
  static constexpr int OFF_Q = OFF_A + NFA;
  static constexpr int OFF_W = OFF_Q + NFQ;
  static constexpr int NF = OFF_W + NFQ;           // fragments per chunk
  static constexpr int OFF_GC = NF * 1024;         // gamma_C, D floats
  static constexpr int OFF_DO = OFF_GC + 4 * D;    // do B fragments [K step][value tile][64][8] fp32
  static constexpr int BYTES = OFF_DO + 2 * 2 * 64 * 8 * 4;
  static constexpr int SROW = 36;                  // staging row stride in floats (rows 4 apart land 16 banks apart)
  static constexpr int STG = kC * SROW * 4;        // dv~ of the slice, fp32 [64][32], stored a step later
};

// One chunk's share of producer P: every kRsProducers-th fragment, two
// 16-byte pieces of the do rows, and (last producer) gamma_C.
template <int D, int P>
struct RsRegs {
  static constexpr int NFP = (RsLayout<D>::NF - P + kRsProducers - 1) / kRsProducers;
  u32x4 f[NFP];
  uint4 d[2];
  u32x4 g;
};

template <int D, int DO, int P>
__device__ __forceinline__ void rs_load(const BwdArgs& a, int b, int n, int h, int c0, int l, RsRegs<D, P>& R) {
  typedef RsLayout<D> LY;
  const int H = a.H;
  const int64_t ch = (static_cast<int64_t>(b) * a.NT + n) * H + h;
#pragma unroll
  for (int k = 0; k < RsRegs<D, P>::NFP; ++k) {
    const int f = P + kRsProducers * k;
    const _Float16* src;
    if (f < LY::OFF_A) src = static_cast<const _Float16*>(a.FL) + (ch * LY::NFL + f) * 512;
    else if (f < LY::OFF_Q) src = static_cast<const _Float16*>(a.FA) + (ch * LY::NFA + (f - LY::OFF_A)) * 512;
    else if (f < LY::OFF_W) src = static_cast<const _Float16*>(a.FQ) + (ch * LY::NFQ + (f - LY::OFF_Q)) * 512;
    else src = static_cast<const _Float16*>(a.FW) + (ch * LY::NFQ + (f - LY::OFF_W)) * 512;
    R.f[k] = *reinterpret_cast<const u32x4*>(src + l * 8);
  }
  // do rows of the slice: 64 rows x 32 columns = 512 pieces of four columns,
  // 128 per producer; rows past the chunk's end load row 0 (zeroed when written)
  const ChunkRows cr = chunk_rows(a, b * a.NT + n);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int pc = 128 * P + 64 * k + l, row = pc >> 3, c4 = pc & 7;
    const int64_t i = ((cr.row0 + (row < cr.len ? row : 0)) * H + h) * D + c0 + 4 * c4;
    if constexpr (DO == 0) R.d[k] = *reinterpret_cast<const uint4*>(static_cast<const float*>(a.dout) + i);
    else {
      const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const u16*>(a.dout) + i);
      R.d[k] = uint4{w.x, w.y, 0u, 0u};
    }
  }
  if constexpr (P == kRsProducers - 1) {
    R.g = u32x4{0, 0, 0, 0};
    if (l < D / 4) R.g = *reinterpret_cast<const u32x4*>(a.GCV + ch * D + 4 * l);
  }
}

template <int D, int DO, int P>
__device__ __forceinline__ void rs_write(unsigned char* dst, const BwdArgs& a, int b, int n, int l,
                                         const RsRegs<D, P>& R) {
  typedef RsLayout<D> LY;
#pragma unroll
  for (int k = 0; k < RsRegs<D, P>::NFP; ++k)
    *reinterpret_cast<u32x4*>(dst + (P + kRsProducers * k) * 1024 + l * 16) = R.f[k];
  const int len = chunk_rows(a, b * a.NT + n).len;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int pc = 128 * P + 64 * k + l, row = pc >> 3, c4 = pc & 7;
    float x[4];
    if constexpr (DO == 0) {
      x[0] = __uint_as_float(R.d[k].x); x[1] = __uint_as_float(R.d[k].y);
      x[2] = __uint_as_float(R.d[k].z); x[3] = __uint_as_float(R.d[k].w);
    } else {
      const f4 v = unpack4<1>(uint2{R.d[k].x, R.d[k].y});
      x[0] = v[0]; x[1] = v[1]; x[2] = v[2]; x[3] = v[3];
    }
    // B fragment (K step row / 32, value tile col / 16), lane (col % 16) +
    // 16 ((row % 16) / 4), element (row % 4) + 4 ((row % 32) / 16)
    const int kb = row >> 5, rr = row & 31;
    const int lane_hi = 16 * ((rr & 15) >> 2), e = (rr & 3) + 4 * (rr >> 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int col = 4 * c4 + i;
      float* p = reinterpret_cast<float*>(dst + LY::OFF_DO) +
                 ((kb * 2 + (col >> 4)) * 64 + (col & 15) + lane_hi) * 8 + e;
      *p = (row < len) ? x[i] : 0.f;
    }
  }
  if constexpr (P == kRsProducers - 1)
    if (l < D / 4) *reinterpret_cast<u32x4*>(dst + LY::OFF_GC + l * 16) = R.g;
}

// Producer P's share of chunk n's dv~ rows from the staging area (64 rows x
// 8 pieces of four columns, 16-byte stores).
template <int D, int P>
__device__ __forceinline__ void rs_store(const BwdArgs& a, const unsigned char* stg, int b, int n, int h, int c0,
                                         int l) {
  const int64_t ch = (static_cast<int64_t>(b) * a.NT + n) * a.H + h;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int pc = 128 * P + 64 * k + l, row = pc >> 3, c4 = pc & 7;
    const f4 v = *reinterpret_cast<const f4*>(stg + (row * RsLayout<D>::SROW + 4 * c4) * 4);
    *reinterpret_cast<f4*>(a.DVT + ch * kC * D + row * D + c0 + 4 * c4) = v;
  }
}

template <int D, int DO, int P>
__device__ __forceinline__ void rs_producer(const BwdArgs& a, unsigned char (*buf)[RsLayout<D>::BYTES],
                                            unsigned char (*stg)[RsLayout<D>::STG], int b, int h, int c0) {
  const int l = threadIdx.x & 63;
  const int NT = a.NT;
  RsRegs<D, P> R0, R1;
  // step s works on chunk NT - 1 - s
  rs_load<D, DO, P>(a, b, NT - 1, h, c0, l, R0);
  rs_load<D, DO, P>(a, b, max(NT - 2, 0), h, c0, l, R1);
  rs_write<D, DO, P>(buf[0], a, b, NT - 1, l, R0);
  lds_barrier();   // chunk of step 0 staged
  auto step = [&](int s, RsRegs<D, P>& Rn, RsRegs<D, P>& Rn1) {
    // store step s-1's dv~; Rn held step s's chunk (in LDS since the last
    // barrier): load step s+2's; write step s+1's from Rn1 (loaded a step
    // earlier) into the free buffer
    if (s > 0) rs_store<D, P>(a, stg[(s - 1) & 1], b, NT - s, h, c0, l);
    rs_load<D, DO, P>(a, b, max(NT - 3 - s, 0), h, c0, l, Rn);
    if (s + 1 < NT) rs_write<D, DO, P>(buf[(s + 1) & 1], a, b, NT - 2 - s, l, Rn1);
    lds_barrier();
  };
  int s = 0;
  for (; s + 1 < NT; s += 2) {
    step(s, R0, R1);
    step(s + 1, R1, R0);
  }
  if (s < NT) step(s, R0, R1);
  rs_store<D, P>(a, stg[(NT - 1) & 1], b, 0, h, c0, l);
  wait_vmem_all();
}

// A column's scale 2^e, e = 15 - exponent(largest |x|), so the largest
// scaled element lies in [2^14, 2^15); e is at most 126 (a column below
// 2^-111 is scaled less than that, which only costs it relative precision it
// cannot use), and at least 15 - 128 for finite x, so 2^e and 2^-e are normal
// floats: the scale and its inverse are exact multipliers.
struct RsScale {
  float up, down;
};
__device__ __forceinline__ RsScale rs_col_scale(float m) {
  const int e = min(15 - __builtin_amdgcn_frexp_expf(m), 126);
  return RsScale{__builtin_amdgcn_ldexpf(1.f, e), __builtin_amdgcn_ldexpf(1.f, -e)};
}
// eight B values, scaled, as fp16 hi + lo
__device__ __forceinline__ void rs_split(const float (&x)[8], float up, h8& hi, h8& lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float y = x[i] * up;
    hi[i] = static_cast<_Float16>(y);
    lo[i] = static_cast<_Float16>(y - static_cast<float>(hi[i]));
  }
}
// largest |x| of a column over the four lanes (gq) that hold it
__device__ __forceinline__ float rs_col_max(float m) {
  m = fmaxf(m, __shfl_xor(m, 16, 64));
  return fmaxf(m, __shfl_xor(m, 32, 64));
}

template <int D, int W>
__device__ __forceinline__ void rs_chain(const BwdArgs& a, unsigned char (*buf)[RsLayout<D>::BYTES],
                                         unsigned char (*stg)[RsLayout<D>::STG], int b, int h, int chain, int c0) {
  typedef RsLayout<D> LY;
  constexpr int NT_ = D / 16;   // channel tiles
  constexpr int NJ = D / 32;    // K steps over the channels
  const int l = threadIdx.x & 63, r = l & 15, gq = l >> 4;
  const int col = c0 + 16 * W + r;   // this lane's value column
  const int NT = a.NT;
  f4 dS[NT_];
  const int64_t sbase = static_cast<int64_t>(chain) * D * D + (4 * gq) * D + col;   // + (16 dt + i) D
#pragma unroll
  for (int dt = 0; dt < NT_; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) dS[dt][i] = (a.dht != nullptr) ? a.dht[sbase + (16 * dt + i) * D] : 0.f;
  lds_barrier();   // chunk of step 0 staged by the producers
  for (int s = 0; s < NT; ++s) {
    const int n = NT - 1 - s;
    const int64_t ch = (static_cast<int64_t>(b) * NT + n) * a.H + h;
    const unsigned char* cur = buf[s & 1];
    auto frag = [&](int f) { return *reinterpret_cast<const h8*>(cur + f * 1024 + l * 16); };
    // the dv~ products' A fragments and the do B values, read ahead of the
    // arithmetic that forms dS' and do's B fragments
    h8 AL[4][NJ], AA[6];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int j = 0; j < NJ; ++j) AL[ct][j] = frag(ct * NJ + j);
#pragma unroll
    for (int f = 0; f < 6; ++f) AA[f] = frag(LY::OFF_A + f);
    float dov[2][8];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const float* p = reinterpret_cast<const float*>(cur + LY::OFF_DO) + ((kb * 2 + W) * 64 + l) * 8;
      const f4 lo = *reinterpret_cast<const f4*>(p), hi4 = *reinterpret_cast<const f4*>(p + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) { dov[kb][i] = lo[i]; dov[kb][4 + i] = hi4[i]; }
    }
    // (the reads stay here, ahead of the arithmetic below)
    __builtin_amdgcn_sched_barrier(0);
    // dS' (the cotangent of the state this chunk leaves) to the workspace
    float* const dsp = a.DS + ch * D * D + (4 * gq) * D + col;
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) dsp[(16 * dt + i) * D] = dS[dt][i];
    // B fragments: dS' over the channels, do over the rows
    float m1 = 0.f;
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) m1 = fmaxf(m1, fabsf(dS[dt][i]));
    const RsScale e1 = rs_col_scale(rs_col_max(m1));
    h8 Sh[NJ], Sl[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const float x[8] = {dS[2 * j][0], dS[2 * j][1], dS[2 * j][2], dS[2 * j][3],
                          dS[2 * j + 1][0], dS[2 * j + 1][1], dS[2 * j + 1][2], dS[2 * j + 1][3]};
      rs_split(x, e1.up, Sh[j], Sl[j]);
    }
    float m2 = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 8; ++i) m2 = fmaxf(m2, fabsf(dov[kb][i]));
    const RsScale e2 = rs_col_scale(rs_col_max(m2));
    h8 Dh[2], Dl[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) rs_split(dov[kb], e2.up, Dh[kb], Dl[kb]);
    // dv~ = (lambda k) dS' + Aqk^T do, row tile ct
    f4 p1[4], p2[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      p1[ct] = f4{0.f, 0.f, 0.f, 0.f};
      p2[ct] = f4{0.f, 0.f, 0.f, 0.f};
    }
    // (consecutive MFMAs feed different accumulators)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) p1[ct] = mma32(p1[ct], AL[ct][j], Sh[j]);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) p1[ct] = mma32(p1[ct], AL[ct][j], Sl[j]);
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int hl = 0; hl < 2; ++hl)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          if (ct >= 2 && kb == 0) continue;   // query rows 0..31 hold no pair with keys 32..63
          p2[ct] = mma32(p2[ct], AA[fa_frag(ct, kb)], hl ? Dl[kb] : Dh[kb]);
        }
    // the dS update's (gamma q)^T fragments; (gamma q)^T do does not wait for dv~
    h8 AQ[NT_][2];
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) AQ[dt][kb] = frag(LY::OFF_Q + 2 * dt + kb);
    f4 pq[NT_];
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt) pq[dt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int hl = 0; hl < 2; ++hl)
#pragma unroll
        for (int dt = 0; dt < NT_; ++dt) pq[dt] = mma32(pq[dt], AQ[dt][kb], hl ? Dl[kb] : Dh[kb]);
    h8 AW[NT_][2];
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) AW[dt][kb] = frag(LY::OFF_W + 2 * dt + kb);
    f4 dvt[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dvt[ct][i] = fmaf(p1[ct][i], e1.down, p2[ct][i] * e2.down);
    float* const dvo = reinterpret_cast<float*>(stg[s & 1]);   // stored by the producers a step later
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) dvo[(16 * ct + 4 * gq + i) * LY::SROW + 16 * W + r] = dvt[ct][i];
    // dv~ as B fragments over the rows
    float m3 = 0.f;
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) m3 = fmaxf(m3, fabsf(dvt[ct][i]));
    const RsScale e3 = rs_col_scale(rs_col_max(m3));
    h8 Vh[2], Vl[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const float x[8] = {dvt[2 * kb][0], dvt[2 * kb][1], dvt[2 * kb][2], dvt[2 * kb][3],
                          dvt[2 * kb + 1][0], dvt[2 * kb + 1][1], dvt[2 * kb + 1][2], dvt[2 * kb + 1][3]};
      rs_split(x, e3.up, Vh[kb], Vl[kb]);
    }
    // dS <- gamma_C dS + (gamma q)^T do - W^T dv~, channel tile dt
    f4 pw[NT_];
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt) pw[dt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int hl = 0; hl < 2; ++hl)
#pragma unroll
        for (int dt = 0; dt < NT_; ++dt) pw[dt] = mma32(pw[dt], AW[dt][kb], hl ? Vl[kb] : Vh[kb]);
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt) {
      const f4 gc = *reinterpret_cast<const f4*>(cur + LY::OFF_GC + (16 * dt + 4 * gq) * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dS[dt][i] = fmaf(-pw[dt][i], e3.down, fmaf(pq[dt][i], e2.down, dS[dt][i] * gc[i]));
    }
    lds_barrier();   // this buffer is free, the next one staged
  }
  if (a.dh0 != nullptr) {
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) a.dh0[sbase + (16 * dt + i) * D] = dS[dt][i];
  }
}

template <int D>
struct alignas(16) Rscan16Lds {
  unsigned char buf[2][RsLayout<D>::BYTES];
  unsigned char stg[2][RsLayout<D>::STG];
};

template <int D, int DO>
__device__ __forceinline__ void rscan16_block(const BwdArgs& a, int block, Rscan16Lds<D>& L) {
  constexpr int NS = D / 32;
  auto& buf = L.buf;
  auto& stg = L.stg;
  int chain, split;
  if (!scan_slot<NS>(block, a.B * a.H, chain, split)) return;   // uniform per workgroup
  const int b = chain / a.H, h = chain - b * a.H;
  const int c0 = 32 * split;
  const int wave = threadIdx.x >> 6;
  switch (wave) {
    case 0: rs_chain<D, 0>(a, buf, stg, b, h, chain, c0); break;
    case 1: rs_chain<D, 1>(a, buf, stg, b, h, chain, c0); break;
    case 2: rs_producer<D, DO, 0>(a, buf, stg, b, h, c0); break;
    case 3: rs_producer<D, DO, 1>(a, buf, stg, b, h, c0); break;
    case 4: rs_producer<D, DO, 2>(a, buf, stg, b, h, c0); break;
    default: rs_producer<D, DO, 3>(a, buf, stg, b, h, c0); break;
  }
}

// ---------------------------------------------------------------------------
// Forward state scan for 16-bit inputs, in the form of the reverse scan above
// (and of the forward's state kernel): per (chain, 32-column slice) two
// compute waves own a 16-column tile of S each,
//   v~ = U - W S,  S <- gamma_C S + (lambda k)^T v~,
// with W and (lambda k)^T as the prep kernel's fp16 A fragments and S, v~
// handed to the matrix cores as fp16 (the forward kernels' operands); four
// producer waves stage W, (lambda k)^T, the slice's U tiles (fp32) and gamma_C
// two chunks ahead.  Each chunk's incoming S is stored fp16 row-major: the
// D-layout tile read as an A fragment is S^T, and its product with the
// identity puts four consecutive columns of one row of S in each lane.  The
// compute waves write S and v~ into a staging area and the producers store
// them with 16-byte stores a step later, so the compute waves issue no global
// memory operation inside the chunk loop.
// ---------------------------------------------------------------------------
constexpr int kFsProducers = 4;

template <int D>
struct FsLayout {
  static constexpr int NFW = 4 * (D / 32);         // W fragments (row tile, K step over channels)
  static constexpr int NFL = 2 * (D / 16);         // (lambda k)^T fragments (channel tile, K step over rows)
  static constexpr int NF = NFW + NFL;             // 1 KiB fragments
  static constexpr int OFF_U = NF * 1024;          // U tiles [row tile][value tile of the slice][64][4] fp32
  static constexpr int NU = 4 * 2;
  static constexpr int OFF_GC = OFF_U + NU * 1024; // gamma_C, D floats
  static constexpr int BYTES = OFF_GC + 4 * D;
  // the compute waves' outputs of a chunk, stored by the producers a step
  // later: S fp16 [D][32], v~ fp32 [64][32] of the slice
  static constexpr int STG_VT = D * 32 * 2;
  static constexpr int STG = STG_VT + kC * 32 * 4;
};

// Producer P's share of a chunk: every kFsProducers-th fragment, two four-
// column pieces of the slice's U rows (64 rows x 8 pieces, 128 per producer)
// and (last producer) gamma_C.
template <int D, int P>
struct FsRegs {
  static constexpr int NFP = (FsLayout<D>::NF - P + kFsProducers - 1) / kFsProducers;
  u32x4 f[NFP];
  f4 u[2];
  u32x4 g;
};

template <int D, int P>
__device__ __forceinline__ void fs_load(const BwdArgs& a, int b, int n, int h, int split, int l, FsRegs<D, P>& R) {
  typedef FsLayout<D> LY;
  const int64_t ch = (static_cast<int64_t>(b) * a.NT + n) * a.H + h;
#pragma unroll
  for (int k = 0; k < FsRegs<D, P>::NFP; ++k) {
    const int f = P + kFsProducers * k;
    const _Float16* src = (f < LY::NFW) ? static_cast<const _Float16*>(a.FWN) + (ch * LY::NFW + f) * 512
                                        : static_cast<const _Float16*>(a.FLT) + (ch * LY::NFL + (f - LY::NFW)) * 512;
    R.f[k] = *reinterpret_cast<const u32x4*>(src + l * 8);
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int pc = 128 * P + 64 * k + l, row = pc >> 3, c4 = pc & 7;
    R.u[k] = *reinterpret_cast<const f4*>(a.UM + ch * kC * D + row * D + 32 * split + 4 * c4);
  }
  if constexpr (P == kFsProducers - 1) {
    R.g = u32x4{0, 0, 0, 0};
    if (l < D / 4) R.g = *reinterpret_cast<const u32x4*>(a.GCV + ch * D + 4 * l);
  }
}

template <int D, int P>
__device__ __forceinline__ void fs_write(unsigned char* dst, int l, const FsRegs<D, P>& R) {
  typedef FsLayout<D> LY;
#pragma unroll
  for (int k = 0; k < FsRegs<D, P>::NFP; ++k)
    *reinterpret_cast<u32x4*>(dst + (P + kFsProducers * k) * 1024 + l * 16) = R.f[k];
  // U piece (row, four columns) into the D-layout tiles [row tile][value
  // tile]: lane (col % 16) + 16 ((row % 16) / 4), element row % 4
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int pc = 128 * P + 64 * k + l, row = pc >> 3, c4 = pc & 7;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int col = 4 * c4 + i;
      reinterpret_cast<float*>(dst + LY::OFF_U)[(((row >> 4) * 2 + (col >> 4)) * 64 + (col & 15) +
                                                 16 * ((row & 15) >> 2)) * 4 + (row & 3)] = R.u[k][i];
    }
  }
  if constexpr (P == kFsProducers - 1)
    if (l < D / 4) *reinterpret_cast<u32x4*>(dst + LY::OFF_GC + l * 16) = R.g;
}

// Producer P's share of chunk n's outputs from the staging area: 16-byte
// pieces of the S rows (D rows x 4) and of the v~ rows (64 rows x 8).
template <int D, int P>
__device__ __forceinline__ void fs_store(const BwdArgs& a, const unsigned char* stg, int b, int n, int h, int split,
                                         int l) {
  typedef FsLayout<D> LY;
  const int64_t ch = (static_cast<int64_t>(b) * a.NT + n) * a.H + h;
  constexpr int NSP = D * 4 / (64 * kFsProducers);   // S pieces per lane
#pragma unroll
  for (int k = 0; k < NSP; ++k) {
    const int pc = 64 * (NSP * P + k) + l, row = pc >> 2, c8 = pc & 3;
    const uint4 v = *reinterpret_cast<const uint4*>(stg + (row * 32 + 8 * c8) * 2);
    *reinterpret_cast<uint4*>(reinterpret_cast<u16*>(a.SI) + ch * D * D + row * D + 32 * split + 8 * c8) = v;
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int pc = 128 * P + 64 * k + l, row = pc >> 3, c4 = pc & 7;
    const f4 v = *reinterpret_cast<const f4*>(stg + LY::STG_VT + (row * 32 + 4 * c4) * 4);
    *reinterpret_cast<f4*>(a.VT + ch * kC * D + row * D + 32 * split + 4 * c4) = v;
  }
}

template <int D, int P>
__device__ __forceinline__ void fs_producer(const BwdArgs& a, unsigned char (*buf)[FsLayout<D>::BYTES],
                                            unsigned char (*stg)[FsLayout<D>::STG], int b, int h, int split) {
  const int l = threadIdx.x & 63;
  const int NT = a.NT;
  FsRegs<D, P> R0, R1;
  fs_load<D, P>(a, b, 0, h, split, l, R0);
  fs_load<D, P>(a, b, min(1, NT - 1), h, split, l, R1);
  fs_write<D, P>(buf[0], l, R0);
  lds_barrier();   // chunk 0 staged
  auto step = [&](int n, FsRegs<D, P>& Rn, FsRegs<D, P>& Rn1) {
    if (n > 0) fs_store<D, P>(a, stg[(n - 1) & 1], b, n - 1, h, split, l);
    fs_load<D, P>(a, b, min(n + 2, NT - 1), h, split, l, Rn);
    if (n + 1 < NT) fs_write<D, P>(buf[(n + 1) & 1], l, Rn1);
    lds_barrier();
  };
  int n = 0;
  for (; n + 1 < NT; n += 2) {
    step(n, R0, R1);
    step(n + 1, R1, R0);
  }
  if (n < NT) step(n, R0, R1);
  fs_store<D, P>(a, stg[(NT - 1) & 1], b, NT - 1, h, split, l);
  wait_vmem_all();
}

template <int D, int W>
__device__ __forceinline__ void fs_chain(const BwdArgs& a, unsigned char (*buf)[FsLayout<D>::BYTES],
                                         unsigned char (*stg)[FsLayout<D>::STG], int b, int h, int chain, int c0) {
  typedef FsLayout<D> LY;
  constexpr int NT_ = D / 16;
  constexpr int NJ = D / 32;
  const int l = threadIdx.x & 63, r = l & 15, gq = l >> 4;
  const int col = c0 + 16 * W + r;
  const int NT = a.NT;
  f4 S[NT_];
#pragma unroll
  for (int dt = 0; dt < NT_; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      S[dt][i] = (a.h0 != nullptr) ? a.h0[(static_cast<int64_t>(chain) * D + 16 * dt + 4 * gq + i) * D + col] : 0.f;
  h4 ident;
#pragma unroll
  for (int i = 0; i < 4; ++i) ident[i] = static_cast<_Float16>((4 * gq + i == r) ? 1.f : 0.f);
  lds_barrier();   // chunk 0 staged by the producers
  for (int n = 0; n < NT; ++n) {
    const int64_t ch = (static_cast<int64_t>(b) * NT + n) * a.H + h;
    const unsigned char* cur = buf[n & 1];
    auto frag = [&](int f) { return *reinterpret_cast<const h8*>(cur + f * 1024 + l * 16); };
    h8 AW[4][NJ];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int j = 0; j < NJ; ++j) AW[ct][j] = frag(ct * NJ + j);
    f4 Ut[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) Ut[ct] = *reinterpret_cast<const f4*>(cur + LY::OFF_U + (2 * ct + W) * 1024 + l * 16);
    __builtin_amdgcn_sched_barrier(0);
    // S as fp16: the B fragments over the channels, and the chunk's incoming
    // state to the workspace (row 16 dt + r, columns 4 gq .. 4 gq + 3 of the tile)
    h4 Sq[NT_];
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) Sq[dt][i] = static_cast<_Float16>(S[dt][i]);
    unsigned char* const so = stg[n & 1];
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt) {
      const f4 tr = mma16(f4{0.f, 0.f, 0.f, 0.f}, Sq[dt], ident);
      h4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = static_cast<_Float16>(tr[i]);
      *reinterpret_cast<h4*>(so + ((16 * dt + r) * 32 + 16 * W + 4 * gq) * 2) = v;
    }
    h8 Sb[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        Sb[j][i] = Sq[2 * j][i];
        Sb[j][4 + i] = Sq[2 * j + 1][i];
      }
    // v~ = U - W S, row tile ct
    f4 P[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) P[ct] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) P[ct] = mma32(P[ct], AW[ct][j], Sb[j]);
    h8 AL[NT_][2];
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) AL[dt][kb] = frag(LY::NFW + 2 * dt + kb);
    f4 vt[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) vt[ct] = Ut[ct] - P[ct];
    float* const vto = reinterpret_cast<float*>(so + LY::STG_VT);
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) vto[(16 * ct + 4 * gq + i) * 32 + 16 * W + r] = vt[ct][i];
    h8 Vb[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        Vb[kb][i] = static_cast<_Float16>(vt[2 * kb][i]);
        Vb[kb][4 + i] = static_cast<_Float16>(vt[2 * kb + 1][i]);
      }
    // S <- gamma_C S + (lambda k)^T v~, channel tile dt
#pragma unroll
    for (int dt = 0; dt < NT_; ++dt) {
      const f4 gc = *reinterpret_cast<const f4*>(cur + LY::OFF_GC + (16 * dt + 4 * gq) * 4);
      S[dt] = S[dt] * gc;
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int dt = 0; dt < NT_; ++dt) S[dt] = mma32(S[dt], AL[dt][kb], Vb[kb]);
    lds_barrier();   // this buffer is free, the next one staged
  }
}

template <int D>
struct alignas(16) Fscan16Lds {
  unsigned char buf[2][FsLayout<D>::BYTES];
  unsigned char stg[2][FsLayout<D>::STG];
};

template <int D>
__device__ __forceinline__ void fscan16_block(const BwdArgs& a, int block, Fscan16Lds<D>& L) {
  constexpr int NS = D / 32;
  auto& buf = L.buf;
  auto& stg = L.stg;
  int chain, split;
  if (!scan_slot<NS>(block, a.B * a.H, chain, split)) return;   // uniform per workgroup
  const int b = chain / a.H, h = chain - b * a.H;
  const int c0 = 32 * split;
  switch (threadIdx.x >> 6) {
    case 0: fs_chain<D, 0>(a, buf, stg, b, h, chain, c0); break;
    case 1: fs_chain<D, 1>(a, buf, stg, b, h, chain, c0); break;
    case 2: fs_producer<D, 0>(a, buf, stg, b, h, split); break;
    case 3: fs_producer<D, 1>(a, buf, stg, b, h, split); break;
    case 4: fs_producer<D, 2>(a, buf, stg, b, h, split); break;
    default: fs_producer<D, 3>(a, buf, stg, b, h, split); break;
  }
}

// ---------------------------------------------------------------------------
// Both scans in one launch: neither reads what the other writes (the forward
// scan gives S and v~ to the chunk kernel, the reverse scan dS' and dv~), and
// each is a serial chain on its own workgroups, so a call whose chains leave
// CUs idle runs them side by side.  The reverse scan's workgroups, the longer
// ones, come first: with more workgroups than CUs the forward ones fill in as
// CUs free up.  Whole backward against the two scans one after the other
// (d = 128, 16-bit inputs): 24 chains of 128 chunks 1 137 -> 974 us, 48 of 64
// 935 -> 896, 64 of 64 1 120 -> 1 117; fp32, 16 of 16 176 -> 138; d = 64, 16-bit
// inputs, 132 of 16 345 -> 315, 512 of 8 576 -> 569; the same bits.
// ---------------------------------------------------------------------------
static_assert(kRsProducers == kFsProducers, "one workgroup size");

template <int D, int DO>
__global__ __launch_bounds__(64 * (2 + kRsProducers), 1) void kda_bwd_scans16_kernel(BwdArgs a, int nblk) {
  constexpr size_t N = sizeof(Rscan16Lds<D>) > sizeof(Fscan16Lds<D>) ? sizeof(Rscan16Lds<D>) : sizeof(Fscan16Lds<D>);
  __shared__ __attribute__((aligned(16))) unsigned char sm[N];
  const int x = blockIdx.x;
  if (x < nblk) rscan16_block<D, DO>(a, x, *reinterpret_cast<Rscan16Lds<D>*>(sm));
  else fscan16_block<D>(a, x - nblk, *reinterpret_cast<Fscan16Lds<D>*>(sm));
}

template <int D, int DO>
__global__ __launch_bounds__(ScanThreads<D>::value) void kda_bwd_scans_kernel(BwdArgs a, int nblk) {
  constexpr size_t N = sizeof(RscanLds<D>) > sizeof(FscanLds<D>) ? sizeof(RscanLds<D>) : sizeof(FscanLds<D>);
  __shared__ __attribute__((aligned(16))) unsigned char sm[N];
  const int x = blockIdx.x;
  if (x < nblk) rscan_block<D, DO>(a, x, *reinterpret_cast<RscanLds<D>*>(sm));
  else fscan_block<D>(a, x - nblk, *reinterpret_cast<FscanLds<D>*>(sm));
}

// The forward scan alone, in LDS of its own size: at d = 64 two workgroups of it
// fit a CU, where a workgroup of the joined launch reserves the reverse scan's
// 99 KiB and has a CU to itself.  That only tells where a chain is one chunk, so
// that no next chunk's loads are in flight beside the step, and with workgroups
// for many rounds (fp32, d = 64, one chunk a chain, whole backward joined and
// apart: 512 chains 98 and 98 us, 1 024 196 and 195, 2 048 392 and 378, 4 096 758
// and 732; 2 048 chains of 16 tokens 349 and 335).  Longer chains are faster
// joined (132 chains of 16 chunks 392 and 444) or the same, as are 16-bit inputs.
template <int D>
__global__ __launch_bounds__(ScanThreads<D>::value) void kda_bwd_fscan_kernel(BwdArgs a) {
  __shared__ FscanLds<D> L;
  fscan_block<D>(a, blockIdx.x, L);
}
constexpr int kForwardApart = 2048;   // forward scan workgroups

// A 16 x 16 accumulator tile (lane (r, gq): rows 4 gq + i, column r) into
// row-major hi / lo bf16 planes of pitch PB at (row0, col0): lanes r and r ^ 1
// swap one value of each row pair, so each lane writes packed column pairs
// (columns r & ~1, r | 1) of rows 4 gq + (r & 1) and 4 gq + 2 + (r & 1).
template <int PB>
__device__ __forceinline__ void acc_put_hl(const f4& v, int row0, int col0, __bf16* h, __bf16* l) {
  const int lane = threadIdx.x & 63, r = lane & 15, gq = lane >> 4;
  const bool odd = (r & 1) != 0;
  const float x0 = __shfl_xor(odd ? v[0] : v[1], 1, 64);
  const float x1 = __shfl_xor(odd ? v[2] : v[3], 1, 64);
  const int o = (row0 + 4 * gq + (odd ? 1 : 0)) * PB + col0 + (r & ~1);
  unsigned hh, ll;
  split2_bf16(odd ? x0 : v[0], odd ? v[1] : x0, hh, ll);
  *reinterpret_cast<unsigned*>(&h[o]) = hh;
  *reinterpret_cast<unsigned*>(&l[o]) = ll;
  split2_bf16(odd ? x1 : v[2], odd ? v[3] : x1, hh, ll);
  *reinterpret_cast<unsigned*>(&h[o + 2 * PB]) = hh;
  *reinterpret_cast<unsigned*>(&l[o + 2 * PB]) = ll;
}

// W of a chunk-head from its fp16 A fragments (rows x channels, the slot
// order of kda_internal.h) into hi / lo bf16 planes [64][PB] with the channel
// contiguous: each lane fragment is row 16 ct + r, channels 32 j + 4 gq .. + 3
// and 32 j + 16 + 4 gq .. + 3.
template <int D, int NTH>
struct WnTile {
  static constexpr int N = 4 * (D / 32) * 64;     // lane fragments
  static constexpr int PER = (N + NTH - 1) / NTH;
  static_assert(N % NTH == 0, "whole lane fragments per thread");
  uint4 w[PER];
  __device__ __forceinline__ void fetch(const void* src) {
#pragma unroll
    for (int p = 0; p < PER; ++p)
      w[p] = *reinterpret_cast<const uint4*>(static_cast<const u16*>(src) + (fresh_tid() + p * NTH) * 8);
  }
  template <int PB>
  __device__ __forceinline__ void put_hl(__bf16* h, __bf16* l) const {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int e = fresh_tid() + p * NTH, f = e >> 6, ln = e & 63;
      const int ct = f / (D / 32), j = f - ct * (D / 32);
      const int row = 16 * ct + (ln & 15), ch0 = 32 * j + 4 * (ln >> 4);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const f4 v = unpack4<2>(hf ? uint2{w[p].z, w[p].w} : uint2{w[p].x, w[p].y});
        uint2 hh, ll;
        split2_bf16(v[0], v[1], hh.x, ll.x);
        split2_bf16(v[2], v[3], hh.y, ll.y);
        *reinterpret_cast<uint2*>(&h[row * PB + ch0 + 16 * hf]) = hh;
        *reinterpret_cast<uint2*>(&l[row * PB + ch0 + 16 * hf]) = ll;
      }
    }
  }
};

// Four consecutive rows of one column of an LDS tile of element type DT: fp32
// in four registers, 16-bit elements packed in two.
template <int DT>
struct Col4 {
  typedef typename InT<DT>::t E;
  uint32_t w[DT == 0 ? 4 : 2];
  __device__ __forceinline__ void load(const E* p, int pitch) {
    if constexpr (DT == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = __float_as_uint(p[i * pitch]);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) w[i] = p[2 * i * pitch] | (static_cast<uint32_t>(p[(2 * i + 1) * pitch]) << 16);
    }
  }
  __device__ __forceinline__ float get(int i) const {
    if constexpr (DT == 0) return __uint_as_float(w[i]);
    else {
      const uint32_t x = w[i >> 1];
      const u16 b = static_cast<u16>((i & 1) ? (x >> 16) : (x & 0xFFFFu));
      return (DT == 1) ? bf16_to_f32(b) : f16bits_to_f32(b);
    }
  }
  __device__ __forceinline__ void opaque_() {
#pragma unroll
    for (int i = 0; i < (DT == 0 ? 4 : 2); ++i) asm volatile("" : "+v"(w[i]));
  }
};

// ---------------------------------------------------------------------------
// per chunk-head adjoint: one workgroup per chunk-head (ChunkThreads), four
// phases separated by workgroup barriers, every phase in the same thread
// mapping so the partial dq, dk, dG stay in registers and each output is
// stored once:
//   1  dY = v~ dS'^T, dgq = do S^T, dW = dv~ S^T, dAqk = do v~^T (two
//      passes over the value channels); the epilogue forms dq's and dk's
//      terms and dG's first terms
//   2  Yw = T^T (-dW), Yu = T^T dv~; dv, dbeta's first terms, dk and dG
//   3  dL = -(Yw W^T + Yu U^T)
//   4  the score adjoints of the wave's row tile (row side) and key tile
//      (column side); dg's reverse cumsum; dq, dk, dg, dbeta stored
// Bound by the phases' latencies at one workgroup per CU (LDS) beside the 447
// KiB it moves per chunk-head (d = 128, 16-bit inputs: 360 us of a 4 096
// chunk-head call at the copy rate).  d = 128, 4 096 chunk-heads, 16-bit
// inputs, traced medians: 657 us with two waves per SIMD, a decay factor formed
// per operand and tile pair and the operands read element by element from LDS in
// phase 4, and two-byte column reads of q, k, v, g from memory; 559 us now
// (within a training step of the layer 691 and 588); 3 072 of the seam's 511 and
// 472, 256 in fp32 48 and 42.
// ---------------------------------------------------------------------------
template <int D, int DTQ, int DTG, int DO>
__global__ __launch_bounds__(ChunkThreads<D>::value) void kda_bwd_chunk_kernel(BwdArgs a) {
  constexpr int NTH = ChunkThreads<D>::value;
  constexpr bool ALPHA = DTG == kAlphaGates;
  constexpr int GT = ALPHA ? 0 : DTG;  // element type of g
  constexpr int NG = NTH / 256;      // waves per row tile (groups of column tiles)
  constexpr int HW = 64;             // value columns per pass of phase 1
  constexpr int NH = D / HW;
  // LDS of the largest phase: phase 1's bf16 planes, phase 2's planes plus
  // the dk, dG hand-off and the row tiles' sums of g, phase 3's planes,
  // phase 4's score cotangent and key / query fragments
  constexpr int ACC0 = (2 * kC + 4 * D) * (kC + 8) / 2;   // floats of phase 2's bf16 planes
  constexpr int GS0 = ACC0 + 2 * kC * D;                  // [4][D] row tiles' sums of g (phase 1's epilogue)
  constexpr int NCT = D / 16;        // column tiles
  constexpr int NPT = 10;            // 16 x 16 tiles (row tile R >= key tile s), at R (R + 1) / 2 + s
  constexpr int FG = 68, FT = 4 * FG;   // row fragments: floats per lane group (padded) and per tile
  constexpr int P4 = 2 * NPT * (FT + 256) + 3 * kC * D + 16 * D + D + NG * kC;   // floats of phase 4
  constexpr int SMEM_FLOATS = cmax(cmax(cmax((6 * kC + 4 * D) * (HW + 8) / 2, GS0 + 4 * D), 8 * kC * (D + 8) / 2), P4);
  __shared__ __attribute__((aligned(16))) float sm[SMEM_FLOATS];
  const int H = a.H;
  const int u = blockIdx.x / H, h = blockIdx.x - u * H;
  const ChunkRows cr = chunk_rows(a, u);
  const int64_t ch = static_cast<int64_t>(u) * H + h;
  auto in_idx = [&](int c, int d) { return ((cr.row0 + c) * H + h) * D + d; };
  // Every phase works in one mapping: wave wv owns row tile mt = wv / NG and
  // the NDT column tiles dt = (wv % NG) NDT + q of every [64][D] array (lane
  // (r, gq) holds rows 16 mt + 4 gq + i, column 16 dt + r), so the gradients
  // of q, k and G accumulate in registers from phase 1 to phase 4 and each
  // is stored once.  Phases 1-3 run on the matrix cores as bf16 hi / lo
  // triples.  Pad rows (c >= len) are never stored (their dG is zero: every
  // term carries a factor q_c or k_c).
  // Output types: fp32, or the primal's 16 bits, rounded here (each rounding
  // pass over fp32 gradients in memory was 37 us a tensor at 2^25 elements)
  const int qot = DTQ == 0 ? 0 : ALPHA ? 1 : a.qkv_out;
  const int got = (DTQ == 0 || GT == 0) ? 0 : a.g_out;
  // rows c0 .. c0 + 3 (those below len) of column d, the lane's column of 16
  // consecutive ones; 16-bit: lanes r and r ^ 1 swap one value of each row
  // pair, so each lane stores packed column pairs of two rows
  auto put_rows = [&](void* dst, int ot, int c0, int d, const float (&x)[4]) {
    if (ot == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (c0 + i < cr.len) static_cast<float*>(dst)[in_idx(c0 + i, d)] = x[i];
    } else {
      const bool odd = (d & 1) != 0;
      const float x0 = __shfl_xor(odd ? x[0] : x[1], 1, 64), x1 = __shfl_xor(odd ? x[2] : x[3], 1, 64);
      const float lo[2] = {odd ? x0 : x[0], odd ? x1 : x[2]}, hi[2] = {odd ? x[1] : x0, odd ? x[3] : x1};
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int c = c0 + 2 * j + (odd ? 1 : 0);
        uint32_t w;
        if (ot == 1) w = pack_bf16x2(lo[j], hi[j]);
        else {
          typedef _Float16 h2 __attribute__((ext_vector_type(2)));
          w = __builtin_bit_cast(uint32_t, h2{static_cast<_Float16>(lo[j]), static_cast<_Float16>(hi[j])});
        }
        if (c < cr.len) *reinterpret_cast<uint32_t*>(static_cast<u16*>(dst) + in_idx(c, d & ~1)) = w;
      }
    }
  };
  constexpr int NDT = NCT / NG;        // column tiles per wave of a [64][D] product
  float pq[NDT][4], pk[NDT][4], pG[NDT][4];   // partial dq, dk, dG at this thread's positions
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave-uniform, as mt and dg_
  const int mt = wv / NG, dg_ = wv % NG;
  // thread and lane indices are taken afresh in each phase (fresh_tid), so
  // the addresses of one phase do not occupy registers in the others

  float dbrD[4], dzp[NDT];             // dbeta partials (rows 16 mt + 4 gq + i), dz partials
#pragma unroll
  for (int i = 0; i < 4; ++i) dbrD[i] = 0.f;
#pragma unroll
  for (int q = 0; q < NDT; ++q) dzp[q] = 0.f;
  // G, k and q (times the scale; zero on pad rows) at this thread's positions
  // (rows 16 mt + 4 gq + i, columns 16 (dg_ NDT + q) + r16), read once in
  // phase 1's epilogue (G formed there from g): phase 2 shares the positions
  // and phase 4 takes its LDS copies of G, k, q from them
  // (q, k held as loaded: 16-bit inputs packed two to a register)
  float gH[NDT][4], gLast[NDT];
  float bH[4];                         // beta of rows 16 mt + 4 gq + i
  Col4<DTQ> kH[NDT], qH[NDT], vH[NDT];
  constexpr int EF = BwdWs<DTQ != 0>::F;    // S_in, T, W

  // Phase 1's dk and dG terms reach phase 2 (same thread, same positions)
  // through LDS past phase 2's buffers, not through dk and dg in memory.
  float* const sAcc = sm + ACC0;   // [2][64][D]: dk, dG
  static_assert(ACC0 + 2 * kC * D <= SMEM_FLOATS, "phase 1 -> 2 accumulators");

  // ---- phase 1: dY = v~ dS'^T, dgq = do S^T, dW = -dv~ S^T, dAqk = do v~^T
  // (K = dv in passes of HW)
  // The operands go to LDS as hi / lo bf16 planes (K contiguous) and each
  // product runs as three bf16 MFMAs per 32-wide K block (hi hi + hi lo +
  // lo hi, about 2^-16 of each product dropped); dW accumulates +dv~ S^T and
  // is negated where phase 2 takes it.
  f4 dW[NDT];
  // dAqk = tril(do v~^T), NKT 16 x 16 tiles per wave (row tile mt, key tiles
  // kt0 + q), from phase 1's do and v~ planes: K = the value channels
  // of each pass; key tiles above the row tile are skipped (masked in phase 3)
  constexpr int NKT = 4 / NG;
  f4 dAa[NKT];
  const int kt0 = __builtin_amdgcn_readfirstlane(NKT * dg_);
#pragma unroll
  for (int q = 0; q < NKT; ++q) dAa[q] = f4{0.f, 0.f, 0.f, 0.f};
  constexpr int TTH = 512;   // threads that hold T for its transposed store
  TTile<kC, TTH, EF> tT;     // phase 2's T, loaded during phase 1's epilogue
  // dv~ in row pairs: phase 1's passes take their columns of it, phase 2 the
  // whole tile as dv~^T (one read of dv~ serves both)
  TTile<D, NTH> tY;
  static_assert(TTile<D, NTH>::PER == 1, "one block of columns");
  // sum_n S[d][n] dS'[d][n] of the rows d this thread loads (a share of the
  // columns each; 16 neighbouring threads share a row)
  constexpr int NDG = Tile<D, HW, NTH>::PER;
  float dgc[NDG];
#pragma unroll
  for (int p = 0; p < NDG; ++p) dgc[p] = 0.f;
  {
    const int t = fresh_tid(), l = t & 63, r16 = l & 15, gq = l >> 4;
    f4 dY[NDT], dgq[NDT];
#pragma unroll
    for (int q = 0; q < NDT; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) dY[q][i] = dgq[q][i] = dW[q][i] = 0.f;
    constexpr int PB = HW + 8;         // bf16 pitch: rows of 32-wide K blocks start 16-byte aligned
    static_assert((6 * kC + 4 * D) * PB / 2 <= SMEM_FLOATS, "phase 1 LDS");
    __bf16* const sVh = reinterpret_cast<__bf16*>(sm);
    __bf16* const sVl = sVh + kC * PB;
    __bf16* const sOh = sVl + kC * PB;
    __bf16* const sOl = sOh + kC * PB;
    __bf16* const sUh = sOl + kC * PB;   // dv~
    __bf16* const sUl = sUh + kC * PB;
    __bf16* const sSh = sUl + kC * PB;
    __bf16* const sSl = sSh + D * PB;
    __bf16* const sDh = sSl + D * PB;    // dS'
    __bf16* const sDl = sDh + D * PB;
    // a pass's operands are loaded during the previous pass's products
    Tile<kC, HW, NTH> pV;
    Tile<D, HW, NTH, EF> pS;
    Tile<D, HW, NTH> pDS;
    InTile<DO, D, HW, NTH> pDo;
    auto fetch_pass = [&](int hp) {
      const int n0 = HW * hp;
      pV.fetch(a.VT + ch * kC * D, D, n0);
      if (hp == 0) tY.fetch(a.DVT + ch * kC * D, D, 0);
      pS.fetch(ws_at<EF>(a.SI, ch * D * D), D, n0);
      pDS.fetch(a.DS + ch * D * D, D, n0);
      pDo.fetch(a.dout, cr.row0, cr.len, H, h, n0);
    };
    InTile<GT, D, D, NTH> ig;
    InTile<DTQ, D, D, NTH> iq, ik, iv;
    auto fetch_in = [&]() {
      ig.fetch(a.g, cr.row0, cr.len, H, h, 0);
      iq.fetch(a.q, cr.row0, cr.len, H, h, 0);
      ik.fetch(a.k, cr.row0, cr.len, H, h, 0);
      iv.fetch(a.v, cr.row0, cr.len, H, h, 0);
    };
    fetch_pass(0);
#pragma unroll
    for (int hp = 0; hp < NH; ++hp) {
      put_hl<PB>(pV, sVh, sVl);
      tY.template put_rows_hl<PB, HW>(hp, sUh, sUl);
      put_hl<PB>(pS, sSh, sSl);
      put_hl<PB>(pDS, sDh, sDl);
      put_hl<PB>(pDo, sOh, sOl);
#pragma unroll
      for (int p = 0; p < NDG; ++p) {
        const float4 x = pS.get(p), y = pDS.get(p);
        dgc[p] += (x.x * y.x + x.y * y.y) + (x.z * y.z + x.w * y.w);
        opaque(dgc[p]);
      }
      __syncthreads();
      if (hp + 1 < NH) fetch_pass(hp + 1);
      else if constexpr (DTQ != 0) fetch_in();   // the epilogue's g, q, k, v (fp32 inputs: after the products)
#pragma unroll
      for (int kb = 0; kb < HW / 32; ++kb) {
        const int ka = (16 * mt + r16) * PB + 32 * kb + 8 * gq;
        // (operands in two groups, which bounds the fragments in registers)
        {
          const b8 vh = *reinterpret_cast<const b8*>(&sVh[ka]), vl = *reinterpret_cast<const b8*>(&sVl[ka]);
#pragma unroll
          for (int q = 0; q < NDT; ++q) {
            const int kbb = (16 * (dg_ * NDT + q) + r16) * PB + 32 * kb + 8 * gq;
            dY[q] = mma3_bf16(dY[q], vh, vl, *reinterpret_cast<const b8*>(&sDh[kbb]),
                              *reinterpret_cast<const b8*>(&sDl[kbb]));
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        const b8 oh = *reinterpret_cast<const b8*>(&sOh[ka]), ol = *reinterpret_cast<const b8*>(&sOl[ka]);
        {
          const b8 uh = *reinterpret_cast<const b8*>(&sUh[ka]), ul = *reinterpret_cast<const b8*>(&sUl[ka]);
#pragma unroll
          for (int q = 0; q < NDT; ++q) {
            const int kbb = (16 * (dg_ * NDT + q) + r16) * PB + 32 * kb + 8 * gq;
            const b8 sh = *reinterpret_cast<const b8*>(&sSh[kbb]), sl = *reinterpret_cast<const b8*>(&sSl[kbb]);
            dgq[q] = mma3_bf16(dgq[q], oh, ol, sh, sl);
            dW[q] = mma3_bf16(dW[q], uh, ul, sh, sl);
          }
        }
#pragma unroll
        for (int q = 0; q < NKT; ++q) {
          if (kt0 + q > mt) continue;
          const int kv = (16 * (kt0 + q) + r16) * PB + 32 * kb + 8 * gq;
          dAa[q] = mma3_bf16(dAa[q], oh, ol, *reinterpret_cast<const b8*>(&sVh[kv]),
                             *reinterpret_cast<const b8*>(&sVl[kv]));
        }
      }
      __syncthreads();
    }
    // g, q, k and v of the chunk-head through LDS (over phase 1's planes) to
    // this thread's positions: whole rows are read from memory and the lanes'
    // column reads fall on distinct banks (pad rows are zero)
    constexpr int PG = D + (GT == 0 ? 4 : 8), PQ = D + (DTQ == 0 ? 4 : 8);
    typedef typename InT<DTQ>::t EQ;
    typedef typename InT<GT>::t EG;
    EG* const sGr = reinterpret_cast<EG*>(sm);
    EQ* const sQr = reinterpret_cast<EQ*>(sm + (sizeof(EG) * kC * PG) / 4);
    EQ* const sKr = sQr + kC * PQ;
    EQ* const sVr = sKr + kC * PQ;
    static_assert(sizeof(EG) * kC * PG + 3 * sizeof(EQ) * kC * PQ <= 4 * GS0, "g, q, k, v end below the sums of g");
    if constexpr (DTQ == 0) fetch_in();
    ig.template put_raw<PG, ALPHA>(sGr, cr.len);
    iq.template put_raw<PQ>(sQr);
    ik.template put_raw<PQ>(sKr);
    iv.template put_raw<PQ>(sVr);
    float* const sBt = sm + GS0 - kC;
    static_assert(sizeof(EG) * kC * PG + 3 * sizeof(EQ) * kC * PQ <= 4 * (GS0 - kC), "beta past g, q, k, v");
    if (t < kC) {
      const float x = ld_beta<DTG>(a.beta, (cr.row0 + (t < cr.len ? t : 0)) * H + h);
      sBt[t] = (t < cr.len) ? x : 0.f;
    }
    __syncthreads();
    // G_c = log2(e) sum_{c' <= c} g_c' at this thread's positions, from g:
    // the prefix over the lane's four rows, plus the lane groups above it in
    // the row tile (shuffles), plus the row tiles above (their sums through
    // LDS, past phase 2's buffers).
    if (t < TTH) tT.fetch(ws_at<EF>(a.TM, ch * kC * kC), kC, 0);
    float* const sGs = sm + GS0;
    const int c0 = 16 * mt + 4 * gq;
#pragma unroll
    for (int i = 0; i < 4; ++i) bH[i] = sBt[c0 + i];
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
      const int d = 16 * (dg_ * NDT + q) + r16;
      Col4<GT> gR;
      gR.load(sGr + c0 * PG + d, PG);
#pragma unroll
      for (int i = 0; i < 4; ++i) gH[q][i] = gR.get(i);
      qH[q].load(sQr + c0 * PQ + d, PQ);
      kH[q].load(sKr + c0 * PQ + d, PQ);
      vH[q].load(sVr + c0 * PQ + d, PQ);
    }
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
#pragma unroll
      for (int i = 1; i < 4; ++i) gH[q][i] += gH[q][i - 1];
      const float tot = gH[q][3];
      const float t1 = __shfl_up(tot, 16), t2 = __shfl_up(tot, 32), t3 = __shfl_up(tot, 48);
      const float ex = (gq >= 1 ? t1 : 0.f) + (gq >= 2 ? t2 : 0.f) + (gq >= 3 ? t3 : 0.f);
#pragma unroll
      for (int i = 0; i < 4; ++i) gH[q][i] += ex;
      if (gq == 3) sGs[mt * D + 16 * (dg_ * NDT + q) + r16] = gH[q][3];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
      const int d = 16 * (dg_ * NDT + q) + r16;
      float pre = 0.f, run = 0.f;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (m == mt) pre = run;
        run += sGs[m * D + d];
      }
      gLast[q] = run * kLog2e;
#pragma unroll
      for (int i = 0; i < 4; ++i) gH[q][i] = (gH[q][i] + pre) * kLog2e;
    }
    // dq = dgq gamma; dG = dgq q gamma - dY k lambda; dk = dY lambda
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
      const int d = 16 * (dg_ * NDT + q) + r16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 16 * mt + 4 * gq + i;
        const float gam = ex2(gH[q][i]), lam = ex2(gLast[q] - gH[q][i]);
        const float dz = dY[q][i] * kH[q].get(i) * lam;
        dzp[q] += dz;
        pq[q][i] = dgq[q][i] * gam * a.scale;
        sAcc[c * D + d] = dY[q][i] * lam;
        sAcc[(kC + c) * D + d] = dgq[q][i] * (qH[q].get(i) * a.scale) * gam - dz;
      }
    }
  }
  // A value carried to a later phase is formed where it is, not sunk into its
  // use there with everything it depends on, and what each phase derives from
  // G, q, k is not kept for the next (registers).
  auto carry = [&](float (&x)[NDT][4]) {
#pragma unroll
    for (int q = 0; q < NDT; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) opaque(x[q][i]);
  };
  auto phase_end = [&]() {
    carry(pq);
    carry(gH);
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
      kH[q].opaque_();
      qH[q].opaque_();
    }
  };
  phase_end();

  // ---- phase 2: Yw = T^T dW, Yu = T^T dv~ (K = the chunk's 64 rows), as
  // bf16 hi / lo triples: T^T, (-dW)^T and dv~^T in LDS with the chunk row
  // contiguous; T[c][m] is zero for c < m, so row tile mt starts at the
  // K block holding row 16 mt.
  f4 Yw[NDT], Yu[NDT];
  // W from its row-major array (fp32 inputs) or its fp16 A fragments (16-bit)
  typename std::conditional<EF == 0, Tile<kC, D, NTH>, WnTile<D, NTH>>::type tW3;
  Tile<kC, D, NTH> tU3;
  {
    const int t = fresh_tid(), l = t & 63, r16 = l & 15, gq = l >> 4;
    constexpr int PB = kC + 8;
    static_assert((2 * kC + 4 * D) * PB / 2 <= ACC0, "phase 2 planes end below sAcc");
    __bf16* const sTh = reinterpret_cast<__bf16*>(sm);   // T^T [64][64]
    __bf16* const sTl = sTh + kC * PB;
    __bf16* const sXh = sTl + kC * PB;                   // (-dW)^T [D][64]
    __bf16* const sXl = sXh + D * PB;
    __bf16* const sYh = sXl + D * PB;                    // dv~^T [D][64]
    __bf16* const sYl = sYh + D * PB;
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
      const int o = (16 * (dg_ * NDT + q) + r16) * PB + 16 * mt + 4 * gq;
      uint2 hh, ll;
      split2_bf16(-dW[q][0], -dW[q][1], hh.x, ll.x);
      split2_bf16(-dW[q][2], -dW[q][3], hh.y, ll.y);
      *reinterpret_cast<uint2*>(&sXh[o]) = hh;
      *reinterpret_cast<uint2*>(&sXl[o]) = ll;
    }
    if (t < TTH) tT.template put_hl<PB>(sTh, sTl);
    tY.template put_hl<PB>(sYh, sYl);
    __syncthreads();
    // phase 3's W and U, during the products
    if constexpr (EF == 0) tW3.fetch(a.WM + ch * kC * D, D, 0);
    else tW3.fetch(static_cast<const u16*>(a.FWN) + ch * kC * D);
    tU3.fetch(a.UM + ch * kC * D, D, 0);
#pragma unroll
    for (int q = 0; q < NDT; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) Yw[q][i] = Yu[q][i] = 0.f;
    for (int kb = mt >> 1; kb < kC / 32; ++kb) {
      const int ka = (16 * mt + r16) * PB + 32 * kb + 8 * gq;
      const b8 th = *reinterpret_cast<const b8*>(&sTh[ka]), tl = *reinterpret_cast<const b8*>(&sTl[ka]);
#pragma unroll
      for (int q = 0; q < NDT; ++q) {
        const int kbb = (16 * (dg_ * NDT + q) + r16) * PB + 32 * kb + 8 * gq;
        Yw[q] = mma3_bf16(Yw[q], th, tl, *reinterpret_cast<const b8*>(&sXh[kbb]),
                          *reinterpret_cast<const b8*>(&sXl[kbb]));
        Yu[q] = mma3_bf16(Yu[q], th, tl, *reinterpret_cast<const b8*>(&sYh[kbb]),
                          *reinterpret_cast<const b8*>(&sYl[kbb]));
      }
    }
    __syncthreads();
    // dG += Yw k beta gamma; dk += Yw gamma beta; dv = Yu beta; dbeta += Yw gamma k + Yu v
    int cb = 16 * mt + 4 * gq;   // (addresses formed here, not held from the loads)
    opaque(cb);
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
      const int d = 16 * (dg_ * NDT + q) + r16;
      float gv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = cb + i;
        const float bc = bH[i], gam = ex2(gH[q][i]), kv = kH[q].get(i);
        dbrD[i] += Yw[q][i] * gam * kv + Yu[q][i] * vH[q].get(i);
        pG[q][i] = sAcc[(kC + c) * D + d] + Yw[q][i] * kv * bc * gam;
        pk[q][i] = sAcc[c * D + d] + Yw[q][i] * gam * bc;
        gv[i] = Yu[q][i] * bc;
      }
      put_rows(a.dv, qot, cb, d, gv);
    }
    __syncthreads();   // sAcc read before phase 3's operands overwrite it
    carry(pk);
    carry(pG);
#pragma unroll
    for (int i = 0; i < 4; ++i) opaque(dbrD[i]);
    phase_end();
  }

  // ---- phase 3: dL = strict(-(Yw W^T + Yu U^T)) [64][64] (dAqk came from
  // phase 1), NKT 16 x 16 tiles per wave: row tile mt, key tiles kt0 + q,
  // as bf16 hi / lo triples (operands row-major with the channel, the K index,
  // contiguous); key tiles above the row tile are masked to zero and skipped.
  // Phase 4's LDS, written at the end of phase 3.  Every fragment is 16 bytes
  // per lane: lane (r, gq) holds K values 4 gq .. 4 gq + 3, one per K step of
  // four v_mfma_f32_16x16x4f32 (the K order inside a tile is free as long as
  // both operands share it).
  float* const sFA = sm;                 // [NPT][FT]  dAqk tiles, rows as M (row r, keys 4 gq ..)
  float* const sFL = sFA + NPT * FT;     //            dL
  float* const sTA = sFL + NPT * FT;     // [NPT][64][4] their transposes, keys as M (key r, rows 4 gq ..)
  float* const sTL = sTA + NPT * 256;
  float* const sKD = sTL + NPT * 256;    // [4][NCT][64][4] k_i 2^(Ge - G_i)
  float* const sQU = sKD + kC * D;       // q_c 2^(G_c - Ga)
  float* const sKU = sQU + kC * D;       // beta_c k_c 2^(G_c - Ga)
  float* const sGa = sKU + kC * D;       // [4][D] G of each row tile's first and last row
  float* const sGe = sGa + 4 * D;
  float* const sDz = sGe + 4 * D;        // [4][D] dz sums of each row tile
  float* const sTile = sDz + 4 * D;      // [4][D] dG sums of each row tile
  float* const sBase = sTile + 4 * D;    // [D] per-column base of dg
  float* const sDb = sBase + D;          // [64][NG] dbeta's sums over each wave's columns
  const int tm0 = mt * (mt + 1) / 2;   // tile (mt, 0)
  {
    const int t = fresh_tid(), l = t & 63, r16 = l & 15, gq = l >> 4;
    constexpr int PB = D + 8;            // bf16 pitch: 16-byte aligned K blocks, rows 4 banks apart
    static_assert(8 * kC * PB / 2 <= SMEM_FLOATS, "phase 3 LDS");
    __bf16* const sAh = reinterpret_cast<__bf16*>(sm);   // Yw
    __bf16* const sAl = sAh + kC * PB;
    __bf16* const sBh = sAl + kC * PB;                   // Yu
    __bf16* const sBl = sBh + kC * PB;
    __bf16* const sWh = sBl + kC * PB;
    __bf16* const sWl = sWh + kC * PB;
    __bf16* const sUh = sWl + kC * PB;
    __bf16* const sUl = sUh + kC * PB;
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
      acc_put_hl<PB>(Yw[q], 16 * mt, 16 * (dg_ * NDT + q), sAh, sAl);
      acc_put_hl<PB>(Yu[q], 16 * mt, 16 * (dg_ * NDT + q), sBh, sBl);
    }
    if constexpr (EF == 0) put_hl<PB>(tW3, sWh, sWl);
    else tW3.template put_hl<PB>(sWh, sWl);
    put_hl<PB>(tU3, sUh, sUl);
    __syncthreads();
    f4 dLa[NKT];
#pragma unroll
    for (int q = 0; q < NKT; ++q) dLa[q] = f4{0.f, 0.f, 0.f, 0.f};
    if (kt0 <= mt) {
#pragma unroll 2
      for (int kb = 0; kb < D / 32; ++kb) {
        const int ka = (16 * mt + r16) * PB + 32 * kb + 8 * gq;
        const b8 ywh = *reinterpret_cast<const b8*>(&sAh[ka]), ywl = *reinterpret_cast<const b8*>(&sAl[ka]);
        const b8 yuh = *reinterpret_cast<const b8*>(&sBh[ka]), yul = *reinterpret_cast<const b8*>(&sBl[ka]);
#pragma unroll
        for (int q = 0; q < NKT; ++q) {
          if (kt0 + q > mt) continue;
          const int kbb = (16 * (kt0 + q) + r16) * PB + 32 * kb + 8 * gq;
          dLa[q] = mma3_bf16(dLa[q], ywh, ywl, *reinterpret_cast<const b8*>(&sWh[kbb]),
                             *reinterpret_cast<const b8*>(&sWl[kbb]));
          dLa[q] = mma3_bf16(dLa[q], yuh, yul, *reinterpret_cast<const b8*>(&sUh[kbb]),
                             *reinterpret_cast<const b8*>(&sUl[kbb]));
        }
      }
    }
    __syncthreads();   // every read of the planes done before phase 4's operands overwrite them
#pragma unroll
    for (int q = 0; q < NKT; ++q) {
      if (kt0 + q > mt) continue;
      const int ti = tm0 + kt0 + q;
      const bool diag = kt0 + q == mt;
      f4 vA, vL;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        vA[i] = (!diag || r16 <= 4 * gq + i) ? dAa[q][i] : 0.f;
        vL[i] = (!diag || r16 < 4 * gq + i) ? -dLa[q][i] : 0.f;
        const int o = ti * FT + (r16 >> 2) * FG + (4 * gq + i) * 4 + (r16 & 3);
        sFA[o] = vA[i];
        sFL[o] = vL[i];
      }
      *reinterpret_cast<f4*>(&sTA[ti * 256 + 4 * l]) = vA;
      *reinterpret_cast<f4*>(&sTL[ti * 256 + 4 * l]) = vL;
    }
  }

  // ---- phase 4: score adjoints.  With dA, dL masked:
  //   row side  rA[c] = sum_i dA[c][i] k_i 2^(G_c - G_i),  rK likewise with dL;
  //   col side  cS[i] = sum_c (dA[c][i] q_c + dL[c][i] beta_c k_c) 2^(G_c - G_i);
  //   dq += rA; dk += rK beta + cS; dG += rA q + rK k beta - cS k; dbeta_c += sum_d rK k_c
  // (q carries the scale).  The decay of a pair in row tile R, key tile s <= R
  // is 2^(G_c - Ga_R) 2^(Ga_R - Ge_s) 2^(Ge_s - G_i), Ga and Ge the G of a row
  // tile's first and last row: the outer factors (<= 1) belong to one row or
  // one key each, so they are formed once per element and shared through LDS
  // by every tile pair, and the middle one, constant over the pair for a
  // channel, is applied to the pair's accumulator column (it is <= 1 off the
  // diagonal, and up to the tile's decay on it; a diagonal tile that decays by
  // more than 2^-kDiagAnchorLog2 in one of the wave's columns takes
  // 2^-|G_c - G_i| per element instead).  Wave (mt, half) forms, for each of
  // its column tiles, the row side of row tile mt (key tiles s <= mt) and the
  // column side of key tile mt (row tiles R >= mt): five tile pairs for every
  // wave, and the results land on the positions whose partial sums it holds.
  // The fp32 matrix cores' floor is half of it (80 v_mfma_f32_16x16x4f32 per
  // wave at d = 128, 10 k of 21 k cycles for the SIMD's four waves); both
  // operands are one 16-byte read for four of them.
  {
    const int t = fresh_tid(), l = t & 63, r16 = l & 15, gq = l >> 4;
    float ga[NDT], ge[NDT];   // Ga, Ge of row tile mt
    unsigned far = 0;         // column tiles q whose diagonal tile goes per element (wave-uniform)
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
      const int ct = dg_ * NDT + q, d = 16 * ct + r16;
      ga[q] = __shfl(gH[q][0], r16, 64);
      ge[q] = __shfl(gH[q][3], 48 + r16, 64);
      if (__any(ga[q] - ge[q] > kDiagAnchorLog2)) far |= 1u << q;
      f4 kd, qu, ku;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float kk = kH[q].get(i), up = ex2(gH[q][i] - ga[q]);
        kd[i] = kk * ex2(ge[q] - gH[q][i]);
        qu[i] = qH[q].get(i) * a.scale * up;
        ku[i] = kk * bH[i] * up;
      }
      const int o = ((mt * NCT + ct) * 64 + l) * 4;
      *reinterpret_cast<f4*>(&sKD[o]) = kd;
      *reinterpret_cast<f4*>(&sQU[o]) = qu;
      *reinterpret_cast<f4*>(&sKU[o]) = ku;
      float dz = dzp[q];
      dz += __shfl_xor(dz, 16, 64);
      dz += __shfl_xor(dz, 32, 64);
      if (gq == 0) {
        sGa[mt * D + d] = ga[q];
        sGe[mt * D + d] = ge[q];
        sDz[mt * D + d] = dz;
      }
    }
    __syncthreads();
    // dg[c] = base + sum_{c' >= c} dG[c']: the G_{C-1} terms and the dz terms
#pragma unroll
    for (int p = 0; p < NDG; ++p) {
      float x = dgc[p];
#pragma unroll
      for (int off = 8; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
      const int d = (t + p * NTH) >> 4;
      if ((t & 15) == 0)
        sBase[d] = x * ex2(sGe[3 * D + d]) + ((sDz[d] + sDz[D + d]) + (sDz[2 * D + d] + sDz[3 * D + d]));
    }
    phase_end();
    float sfx[NDT][4], abv[NDT];
    // one column tile at a time, which keeps everything in registers
#pragma unroll
    for (int q0 = 0; q0 < NDT; ++q0) {
      __builtin_amdgcn_sched_barrier(0);
      f4 rA[NDT], rK[NDT], cS[NDT];
#pragma unroll
      for (int q = q0; q < q0 + 1; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) rA[q][i] = rK[q][i] = cS[q][i] = 0.f;
      // row side
      for (int s = 0; s <= mt; ++s) {
        const f4 fa = *reinterpret_cast<const f4*>(&sFA[(tm0 + s) * FT + gq * FG + r16 * 4]);
        const f4 fl = *reinterpret_cast<const f4*>(&sFL[(tm0 + s) * FT + gq * FG + r16 * 4]);
#pragma unroll
        for (int q = q0; q < q0 + 1; ++q) {
          if (s == mt && (far >> q & 1)) continue;
          const int ct = dg_ * NDT + q;
          const f4 kd = *reinterpret_cast<const f4*>(&sKD[((s * NCT + ct) * 64 + l) * 4]);
          const float m = ex2(ga[q] - sGe[s * D + 16 * ct + r16]);
          f4 x = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            x = mfma4(fa[k], kd[k], x);
            y = mfma4(fl[k], kd[k], y);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            rA[q][i] = fmaf(m, x[i], rA[q][i]);
            rK[q][i] = fmaf(m, y[i], rK[q][i]);
          }
        }
      }
      // column side
      for (int R = mt; R < 4; ++R) {
        const int ti = R * (R + 1) / 2 + mt;
        const f4 ta = *reinterpret_cast<const f4*>(&sTA[ti * 256 + 4 * l]);
        const f4 tl = *reinterpret_cast<const f4*>(&sTL[ti * 256 + 4 * l]);
#pragma unroll
        for (int q = q0; q < q0 + 1; ++q) {
          if (R == mt && (far >> q & 1)) continue;
          const int ct = dg_ * NDT + q, o = ((R * NCT + ct) * 64 + l) * 4;
          const f4 qu = *reinterpret_cast<const f4*>(&sQU[o]), ku = *reinterpret_cast<const f4*>(&sKU[o]);
          const float m = ex2(sGa[R * D + 16 * ct + r16] - ge[q]);
          f4 x = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            x = mfma4(ta[k], qu[k], x);
            y = mfma4(tl[k], ku[k], y);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) cS[q][i] = fmaf(m, x[i] + y[i], cS[q][i]);
        }
      }
#pragma unroll
      for (int q = q0; q < q0 + 1; ++q) {
        const int d = 16 * (dg_ * NDT + q) + r16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float up = ex2(gH[q][i] - ga[q]);
          rA[q][i] *= up;
          rK[q][i] *= up;
          cS[q][i] *= ex2(ge[q] - gH[q][i]);
        }
        if (far >> q & 1) {
          // With G non-increasing (g <= 0), the pair (c, y) of the row side
          // (y <= c) decays by 2^(G_c - G_y) and the pair (y, c) of the column
          // side (y >= c) by 2^(G_y - G_c): both are 2^-|G_c - G_y|, and the
          // masked cotangents zero the side a given y does not belong to.  Row
          // y's G, k, q, beta come from the lane of its column that holds them.
#pragma unroll
          for (int yy = 0; yy < 4; ++yy) {
            const float qs = qH[q].get(yy) * a.scale, kk = kH[q].get(yy);
#pragma unroll 1
            for (int y4 = 0; y4 < 4; ++y4) {
              const int src = 16 * y4 + r16, y = 4 * y4 + yy;
              const float gy = __shfl(gH[q][yy], src, 64), ky = __shfl(kk, src, 64);
              const float qy = __shfl(qs, src, 64), by = __shfl(bH[yy], src, 64);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int c = 4 * gq + e;
                const float ev = ex2(-fabsf(gH[q][e] - gy)), kr = ky * ev;
                const int of = (tm0 + mt) * FT + y4 * FG + c * 4 + yy;
                const int ot = (tm0 + mt) * 256 + (y4 * 16 + c) * 4 + yy;
                rA[q][e] = fmaf(sFA[of], kr, rA[q][e]);
                rK[q][e] = fmaf(sFL[of], kr, rK[q][e]);
                cS[q][e] = fmaf(sTA[ot], qy * ev, cS[q][e]);
                cS[q][e] = fmaf(sTL[ot], by * kr, cS[q][e]);
              }
            }
          }
        }
        float gn[4], oq[4], ok[4];   // this tile's dG (zero on pad rows), dq, dk
        int cb = 16 * mt + 4 * gq;   // (addresses formed here, not held from the loads)
        opaque(cb);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int c = cb + e;
          const float kc = kH[q].get(e), qc = qH[q].get(e) * a.scale, bc = bH[e];
          dbrD[e] = fmaf(rK[q][e], kc, dbrD[e]);
          gn[e] = (c < cr.len) ? pG[q][e] + rA[q][e] * qc + rK[q][e] * kc * bc - cS[q][e] * kc : 0.f;
          oq[e] = pq[q][e] + rA[q][e] * a.scale;
          ok[e] = pk[q][e] + rK[q][e] * bc + cS[q][e];
        }
        put_rows(a.dq, qot, cb, d, oq);
        put_rows(a.dk, qot, cb, d, ok);
        // reverse cumsum down the column: within the lane's four rows, then
        // over the row groups gq' > gq of the tile (lanes 16 gq' + r16); the
        // tiles below come after the barrier
        sfx[q][3] = gn[3];
        sfx[q][2] = gn[2] + sfx[q][3];
        sfx[q][1] = gn[1] + sfx[q][2];
        sfx[q][0] = gn[0] + sfx[q][1];
        const float x1 = __shfl_down(sfx[q][0], 16, 64), x2 = __shfl_down(sfx[q][0], 32, 64);
        const float x3 = __shfl_down(sfx[q][0], 48, 64);
        abv[q] = (gq < 3 ? x1 : 0.f) + (gq < 2 ? x2 : 0.f) + (gq < 1 ? x3 : 0.f);
        if (gq == 0) sTile[mt * D + d] = sfx[q][0] + abv[q];   // the tile's column sum
      }
    }
    // dbeta: phase 2's and this phase's terms, summed over the wave's columns
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = dbrD[e];
#pragma unroll
      for (int off = 8; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
      if (r16 == 0) sDb[(16 * mt + 4 * gq + e) * NG + dg_] = v;
    }
    float al[NDT][4];   // the seam's alpha at this thread's positions
    if constexpr (ALPHA) {
      int cb = 16 * mt + 4 * gq;
      opaque(cb);
#pragma unroll
      for (int q = 0; q < NDT; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          al[q][e] = static_cast<const float*>(a.g)[in_idx(cb + e < cr.len ? cb + e : 0, 16 * (dg_ * NDT + q) + r16)];
    }
    __syncthreads();   // every tile's column sums and dbeta's row sums written
#pragma unroll
    for (int q = 0; q < NDT; ++q) {
      const int d = 16 * (dg_ * NDT + q) + r16;
      float carry = 0.f;   // the tiles below, the furthest first
      for (int R = 3; R > mt; --R) carry += sTile[R * D + d];
      const float base = sBase[d] + carry + abv[q];
      int cb = 16 * mt + 4 * gq;
      opaque(cb);
      float gn[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        gn[e] = base + sfx[q][e];
        if constexpr (ALPHA) gn[e] /= al[q][e];   // dalpha = d(log alpha) / alpha
      }
      put_rows(a.dg, got, cb, d, gn);
    }
    if constexpr (ALPHA) {   // each of the 32 columns gets a 32nd
      constexpr int V = 8;   // 16-byte pieces per row
      if (t < kC * V && t / V < cr.len) {
        const int row = t / V;
        float x = sDb[row * NG];
#pragma unroll
        for (int j = 1; j < NG; ++j) x += sDb[row * NG + j];
        x *= 1.0f / 32.0f;
        *reinterpret_cast<f4*>(static_cast<float*>(a.dbeta) + ((cr.row0 + row) * H + h) * 32 + 4 * (t % V)) = f4{x, x, x, x};
      }
    } else if (t < kC && t < cr.len) {
      float x = sDb[t * NG];
#pragma unroll
      for (int j = 1; j < NG; ++j) x += sDb[t * NG + j];
      const int64_t o = (cr.row0 + t) * H + h;
      if (got == 0) static_cast<float*>(a.dbeta)[o] = x;
      else if (got == 1) static_cast<u16*>(a.dbeta)[o] = cvt_bf16(x);
      else static_cast<_Float16*>(a.dbeta)[o] = static_cast<_Float16>(x);
    }
  }
}

template <int D, int DTQ, int DTG, int DO>
hipError_t launch_bwd_t(const BwdArgs& a, hipStream_t s) {
  const int chunk_heads = a.B * a.NT * a.H;
  const int chains = a.B * a.H;
  hipLaunchKernelGGL((kda_bwd_prep_kernel<D, DTQ, DTG>), dim3(chunk_heads), dim3(kPrepThreads), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int scan_grid = (chains + 7) / 8 * 8 * (D / 32);   // workgroups of either scan
  auto scans = [&](int grid, int nblk) {   // the first nblk workgroups run the reverse scan
    if constexpr (DTQ != 0)
      hipLaunchKernelGGL((kda_bwd_scans16_kernel<D, DO>), dim3(grid), dim3(64 * (2 + kRsProducers)), 0, s, a, nblk);
    else
      hipLaunchKernelGGL((kda_bwd_scans_kernel<D, DO>), dim3(grid), dim3(ScanThreads<D>::value), 0, s, a, nblk);
    return hipGetLastError();
  };
  const int64_t state_bytes = static_cast<int64_t>(chains) * D * D * 4;
  auto forward = [&]() {   // the forward scan alone
    if constexpr (D == 64 && DTQ == 0) {
      hipLaunchKernelGGL(kda_bwd_fscan_kernel<D>, dim3(scan_grid), dim3(ScanThreads<D>::value), 0, s, a);
      return hipGetLastError();
    } else {
      return scans(scan_grid, 0);
    }
  };
  // apart: see kda_bwd_fscan_kernel; and with dh0 over h0 the forward scan reads h0 first
  if ((D == 64 && DTQ == 0 && a.NT == 1 && scan_grid >= kForwardApart) ||
      overlaps(a.dh0, state_bytes, a.h0, state_bytes)) {
    e = forward();
    if (e == hipSuccess) e = scans(scan_grid, scan_grid);
  } else {
    e = scans(2 * scan_grid, scan_grid);
  }
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((kda_bwd_chunk_kernel<D, DTQ, DTG, DO>), dim3(chunk_heads), dim3(ChunkThreads<D>::value), 0, s, a);
  return hipGetLastError();
}

template <int D, int DO>
hipError_t launch_bwd_dt(const BwdArgs& a, int in_dtype, hipStream_t s) {
  switch (in_dtype) {
    case 0: return launch_bwd_t<D, 0, 0, DO>(a, s);
    case 1: return launch_bwd_t<D, 1, 1, DO>(a, s);
    case 2: return launch_bwd_t<D, 2, 2, DO>(a, s);
    default: return launch_bwd_t<D, 1, 0, DO>(a, s);
  }
}

__global__ __launch_bounds__(kThreads) void kda_copy_or_zero_kernel(float* dst, const float* src, int64_t n) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * kThreads)
    dst[i] = (src != nullptr) ? src[i] : 0.f;
}

}  // namespace

hipError_t launch_copy_or_zero(float* dst, const float* src, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int64_t blocks = (n + kThreads - 1) / kThreads;
  const int grid = static_cast<int>(blocks < 4096 ? blocks : 4096);
  hipLaunchKernelGGL(kda_copy_or_zero_kernel, dim3(grid), dim3(kThreads), 0, s, dst, src, n);
  return hipGetLastError();
}

hipError_t launch_bwd(const BwdArgs& a, int d, int in_dtype, int do_dtype, hipStream_t s) {
  if (in_dtype == kInAlphaGates)   // do is fp32
    return d == 128 ? launch_bwd_t<128, 1, kAlphaGates, 0>(a, s) : launch_bwd_t<64, 1, kAlphaGates, 0>(a, s);
  if (d == 128) return do_dtype == 0 ? launch_bwd_dt<128, 0>(a, in_dtype, s) : launch_bwd_dt<128, 1>(a, in_dtype, s);
  return do_dtype == 0 ? launch_bwd_dt<64, 0>(a, in_dtype, s) : launch_bwd_dt<64, 1>(a, in_dtype, s);
}

}  // namespace kda
