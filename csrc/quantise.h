// e4m3 rows with one scale each: what the scaled matrix instruction multiplies with FP8 and MXFP4 weights.  Shared by the kernel that quantises a
// row (csrc/mfma_scaled.hip) and the one that updates the residual first (csrc/engine_kernels.hip): the same bytes and scales.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace quantise {

// of a row whose largest magnitude is `amax`: x ~= byte * scale (1 for an all-zero row)
__device__ inline float scale_of(float amax) { return amax > 0.f ? amax * (1.f / 448.f) : 1.f; }

// Columns i .. i + 7 (i a multiple of 8) of a row of bytes.  PERMUTE: inside every group of 64 columns the bytes are in the order of the packed FP8
// weight fragments (kv_pack_weight_fp8), byte 16 q + j holding k = 8 q + j for j < 8 and k = 32 + 8 q + (j - 8) for j >= 8, so that a 16-byte
// chunk of the row is exactly what lane quarter q of a weight fragment multiplies; else in order (the FP4 operand is in k order).
template <bool PERMUTE>
__device__ inline void store8(unsigned char* row, int i, const float (&x)[8], float inv) {
  float f[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) f[j] = x[j] * inv;
  unsigned int lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], hi, true);
  const int w = i & 63;  // k = 32 half + 8 q + j of the group
  *reinterpret_cast<uint2*>(row + (PERMUTE ? (i & ~63) + 16 * ((w & 31) >> 3) + 8 * (w >> 5) : i)) = make_uint2(lo, hi);
}

}  // namespace quantise
