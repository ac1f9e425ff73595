// Reductions over the lanes of a wave without LDS: lanes 1, 2, 4 and 8 apart by DPP moves, 16 and 32 apart by the swaps of rows and halves.  A shuffle through
// LDS (ds_bpermute) is some 100 cycles until its answer is there, six of them in a row 0.3 us of a launch that has two or three such sums and takes 3 to 5 in all; these
// take 60 cycles together.  The same pairs in the same order as a butterfly of shuffles: the same bits.  Where each lane brings one product, shuffles let the
// compiler fuse a lane's own with the rounded one that it got; the swaps would not, so such sums have a form of their own.
#pragma once
#include <hip/hip_runtime.h>

namespace lanes {

// the value of the lane M away (lane ^ M), M up to 8
template <int M>
__device__ inline unsigned int across(unsigned int v) {
  static_assert(M == 1 || M == 2 || M == 4 || M == 8, "inside a row of 16 lanes");
  const int x = (int)v;
  if constexpr (M == 1) return (unsigned int)__builtin_amdgcn_update_dpp(x, x, 0xB1, 0xf, 0xf, false);   // quad_perm 1 0 3 2
  if constexpr (M == 2) return (unsigned int)__builtin_amdgcn_update_dpp(x, x, 0x4E, 0xf, 0xf, false);   // quad_perm 2 3 0 1
  if constexpr (M == 8) return (unsigned int)__builtin_amdgcn_update_dpp(x, x, 0x128, 0xf, 0xf, false);  // row_ror 8
  const int up = __builtin_amdgcn_update_dpp(x, x, 0x104, 0xf, 0x5, false);                              // row_shl 4: the quads that have one above them
  return (unsigned int)__builtin_amdgcn_update_dpp(up, x, 0x114, 0xf, 0xa, false);                       // row_shr 4: the others
}

// op(v, the value of the lane M away), op the same either way round
template <int M, class Op>
__device__ inline float meet(float v, Op op) {
  const unsigned int u = __float_as_uint(v);
  if constexpr (M == 16) {
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return op(__uint_as_float(a[0]), __uint_as_float(a[1]));
  } else if constexpr (M == 32) {
    const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return op(__uint_as_float(a[0]), __uint_as_float(a[1]));
  } else {
    return op(v, __uint_as_float(across<M>(u)));
  }
}

// over the lanes FROM, FROM / 2 ... TO apart (powers of two)
template <int FROM, int TO, class Op>
__device__ inline float meet_down(float v, Op op) {
  v = meet<FROM>(v, op);
  if constexpr (FROM > TO) v = meet_down<FROM / 2, TO>(v, op);
  return v;
}
// over the lanes FROM, 2 FROM ... below END apart
template <int FROM, int END, class Op>
__device__ inline float meet_up(float v, Op op) {
  if constexpr (FROM < END) {
    v = meet<FROM>(v, op);
    v = meet_up<2 * FROM, END>(v, op);
  }
  return v;
}

struct Sum { __device__ float operator()(float a, float b) const { return a + b; } };
struct Max { __device__ float operator()(float a, float b) const { return fmaxf(a, b); } };

// of all 64 lanes, in all of them
__device__ inline float sum(float v) { return meet_down<32, 1>(v, Sum{}); }
__device__ inline float max(float v) { return meet_down<32, 1>(v, Max{}); }

// of all 64 lanes' a b: a lane's own product meets that of 32 lanes away unrounded (so the halves of the wave may differ in the last bit)
__device__ inline float sum_of_products(float a, float b) {
  const unsigned int u = __float_as_uint(a * b);
  const auto halves = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return meet_down<16, 1>(__builtin_fmaf(a, b, __uint_as_float(halves[0] ^ halves[1] ^ u)), Sum{});
}

// the larger value and, of equal ones, the smaller index, in all lanes
template <int M>
__device__ inline void best_of(float& v, int& i) {
  const unsigned int u = __float_as_uint(v);
  float ov[2];
  int oi[2];
  if constexpr (M == 16) {
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false), b = __builtin_amdgcn_permlane16_swap((unsigned int)i, (unsigned int)i, false, false);
    ov[0] = __uint_as_float(a[0]); ov[1] = __uint_as_float(a[1]); oi[0] = (int)b[0]; oi[1] = (int)b[1];
  } else if constexpr (M == 32) {
    const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false), b = __builtin_amdgcn_permlane32_swap((unsigned int)i, (unsigned int)i, false, false);
    ov[0] = __uint_as_float(a[0]); ov[1] = __uint_as_float(a[1]); oi[0] = (int)b[0]; oi[1] = (int)b[1];
  } else {
    ov[0] = v; oi[0] = i;
    ov[1] = __uint_as_float(across<M>(u)); oi[1] = (int)across<M>((unsigned int)i);
  }
  const bool other = ov[1] > ov[0] || (ov[1] == ov[0] && oi[1] < oi[0]);
  v = other ? ov[1] : ov[0];
  i = other ? oi[1] : oi[0];
}
__device__ inline void best(float& v, int& i) {
  best_of<32>(v, i); best_of<16>(v, i); best_of<8>(v, i); best_of<4>(v, i); best_of<2>(v, i); best_of<1>(v, i);
}

}  // namespace lanes
