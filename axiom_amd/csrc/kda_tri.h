// (I + L)^-1 of a strictly lower-triangular 64 x 64 fp32 matrix in LDS, by one
// workgroup: the four diagonal 16 x 16 blocks by forward substitution (one
// column per thread of the first wave, in registers; the other waves zero the
// blocks above the diagonal meanwhile), then the off-diagonal blocks by the
// blocked recurrence T_Rs = -T_RR sum_{j=s}^{R-1} L_Rj T_js on the fp32 matrix
// cores (exact fp32 products).  A block column needs only its own blocks and
// the diagonal ones, so wave s runs down column s without waiting for the
// others.  Used by the backward's prep kernel and the standalone solve.
#pragma once

#include <hip/hip_runtime.h>

namespace kda {

// sL, sT: [64][PC] (PC >= 64); tmp: >= 768 floats of LDS.  L's diagonal and
// upper part are not read.  All NTH >= 192 threads of the workgroup call it
// with sL written (a barrier before); it ends with a barrier, so sT is
// readable by every thread on return.
template <int PC, int NTH>
__device__ __forceinline__ void invert_unit_lower64(const float* sL, float* sT, float* tmp) {
  static_assert(NTH >= 192 && NTH % 64 == 0, "three block columns and the zeroing threads");
  const int t = threadIdx.x;
  if (t < 64) {
    // column j of the block's inverse: x_i = [i == j] - sum_{m<i} L_im x_m
    // (x_m = 0 for m < j, so the sums may run over all m < i)
    const int R = t >> 4, j = t & 15, a0 = 16 * R;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float acc = 0.f;
#pragma unroll
      for (int m = 0; m < i; ++m) acc = fmaf(sL[(a0 + i) * PC + a0 + m], x[m], acc);
      x[i] = (i < j) ? 0.f : ((i == j) ? 1.f : -acc);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) sT[(a0 + i) * PC + a0 + j] = x[i];
  } else {
    for (int e = t - 64; e < 6 * 256; e += NTH - 64) {
      const int blk = e >> 8, rc = (e >> 4) & 15, ri = e & 15;
      const int R = (blk < 3) ? 0 : (blk < 5) ? 1 : 2;             // (0,1) (0,2) (0,3) (1,2) (1,3) (2,3)
      const int sk = (blk < 3) ? blk + 1 : (blk < 5) ? blk - 1 : 3;
      sT[(16 * R + rc) * PC + 16 * sk + ri] = 0.f;
    }
  }
  __syncthreads();
  // Off-diagonal blocks of column sb, top to bottom: X = sum_{j=sb}^{R-1} L_Rj
  // T_js, through the wave's 16 x 16 of tmp into the B layout, then T_Rs =
  // -T_RR X.  Lane (r = l & 15, gq = l >> 4) supplies A[r][4k + gq] and
  // B[4k + gq][r] and holds rows 4 gq + e, column r of the result.
  const int sb = t >> 6, l = t & 63, r = l & 15, gq = l >> 4;
  if (sb < 3) {
    float* X = tmp + 256 * sb;
    typedef float f4_ __attribute__((ext_vector_type(4)));
    auto settle = [] {   // the wave's LDS writes, ordered before its reads
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };
    for (int R = sb + 1; R < 4; ++R) {
      f4_ acc = {0.f, 0.f, 0.f, 0.f};
      for (int j = sb; j < R; ++j) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(sL[(16 * R + r) * PC + 16 * j + 4 * k + gq],
                                                     sT[(16 * j + 4 * k + gq) * PC + 16 * sb + r], acc, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) X[(4 * gq + e) * 16 + r] = acc[e];
      settle();
      f4_ out = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; ++k)
        out = __builtin_amdgcn_mfma_f32_16x16x4f32(sT[(16 * R + r) * PC + 16 * R + 4 * k + gq],
                                                   X[(4 * k + gq) * 16 + r], out, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) sT[(16 * R + 4 * gq + e) * PC + 16 * sb + r] = -out[e];
      settle();
    }
  }
  __syncthreads();
}

}  // namespace kda
