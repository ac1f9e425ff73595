// Products by panels of 256 features on gfx950, for one matrix of many outputs and for a mixture of experts with many rows.
//  * A workgroup is a panel x up to 256 rows; each of its 8 waves owns 32 features and all rows.  Weights (in fragments, fragments.h) go
//    straight to registers, no byte twice, 3 to 6 stages of 64 columns ahead (96 KiB of them in flight per CU: through LDS there was room for
//    48), the rows to LDS by LDS-DMA, as far ahead, in a ring; all waves read all rows from there.
//  * The barrier of a stage stands before its last batch, where the first read of the next stage is issued, not at its top: what is fetched has a
//    stage longer to come (2048 x 28672 x 4096: 390 -> 373 us).
//  * Work follows the rows that exist, in steps of 32: 2 x NF products per 64 columns and feature tile, NF = rows / 16 rounded up to an even
//    number, one loop for each NF.  All waves have the same share, whatever the number.
//  * LDS-DMA and loads are buffer instructions: the offset of a stage is scalar, and the compiler counts them exactly in front of a use (beside
//    the FLAT form it waits for everything in flight).
//  * Stores are 16 bytes a lane, gathered from the two feature tiles (and, gated, two row tiles) by lane swaps.
// Four waves of 64 features each, which read the LDS half as often, are slower (464 against 395 us): with one wave per SIMD nothing multiplies
// while it issues memory operations.
//
// Experts (the (token, choice) pairs that chose one, up to 256 a tile, y[pair] = W[expert] x[row of the pair]) are bound by the matrices: every one is
// read once (1.2 GB for 64 of 2304 x 4096) for some 100 to 300 rows, so bytes and matrix work take about as long.  Every sum goes through the columns
// from the first to the last, so that a row's outputs do not depend on the tile and panel it falls into, and are those of the tiled kernel.  (Workgroups
// that start at columns of their own, past the caches' reuse, ask other memory channels at a time and take 3 to 5 % less, but round otherwise.)
// Measured, gate / up and down of 64 experts of 2304 x 4096 chosen by 187 rows each: 874 us; by tiles of 256 x 256 through LDS, all 256 rows multiplied,
// 1055; 300 rows 1306 and 2004, 64 rows 685 and 749.

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include <utility>

#include "experts.h"
#include "fragments.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 frag_ab;
typedef __attribute__((ext_vector_type(4))) float frag_cd;
typedef __attribute__((ext_vector_type(4))) unsigned int raw16;
typedef __attribute__((address_space(3))) void lds_void;
typedef __amdgpu_buffer_rsrc_t rsrc_t;

enum Mode { PLAIN = 0, GATED = 1, SQUARED = 2 };

constexpr int ROWS = 256, FEATURES = 256;  // of a tile
constexpr int RING_BYTES = 144 * 1024;
// stages of 64 columns in flight, and one more in the ring: as many as registers (16 of weights a stage) and LDS (2 KiB of rows per row tile) hold
constexpr int ahead(int nf) { return nf > 14 ? 3 : nf > 12 ? 4 : nf > 10 ? 5 : 6; }

// What is multiplied: bf16 by bf16, or e4m3 rows by e4m3 weights or by MXFP4 ones (e2m1 in blocks of 32, an E8M0 scale each).  Of rows of bytes K, ldx
// and a stage's columns count pairs: then a stage is 128 columns and as many bytes of rows and of e4m3 weights as one of 64 columns of bf16.
enum Numbers { BF16 = 0, FP8 = 1, MXFP4 = 2 };
struct Scales { const float* w; const float* x; const int* blocks; };  // of the outputs (e4m3 weights) and of the rows; of the blocks, [N/16][stages][16], a byte each

struct PanelArgs {
  const unsigned char* w; const __bf16* x; unsigned short* y;
  int N, K; long long ldx, ldy;
  int n_panels, features;  // of a panel: all eight waves', or four's
  unsigned int x_bytes;
  ExpertGate gate;
  GroupedRows groups;
};

// round to nearest even, NaN kept quiet (hardware conversion, two at a time)
__device__ inline unsigned int pack2(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  return __builtin_bit_cast(unsigned int, (bf16x2){(__bf16)a, (__bf16)b});
}
__device__ inline uint2 pack4(frag_cd v) { return make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3])); }

__device__ inline rsrc_t buffer_of(const void* p, unsigned int bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00027000); }
__device__ inline int load4(rsrc_t r, int lane_off, int off) { return __builtin_bit_cast(int, __builtin_amdgcn_raw_buffer_load_b32(r, lane_off, off, 0)); }
__device__ inline raw16 load16(rsrc_t r, int lane_off, int off) { return __builtin_bit_cast(raw16, __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0)); }
// one LDS-DMA piece: lane l's 16 bytes land at lds + 16 l
__device__ inline void dma16(rsrc_t r, int lane_off, int off, void* lds) { __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds, 16, lane_off, off, 0, 0); }

typedef __attribute__((ext_vector_type(8))) int raw32;
// an operand of 128 bytes' columns from its two pieces of 64
template <class T>
__device__ inline raw32 both(T a, T b) { return __builtin_shufflevector(__builtin_bit_cast(__attribute__((ext_vector_type(4))) int, a), __builtin_bit_cast(__attribute__((ext_vector_type(4))) int, b), 0, 1, 2, 3, 4, 5, 6, 7); }
// packed e2m1 weights (a lane has 4 x 8 columns, 32 apart) to the operand, where it has 32 in a row: a transposition over the quarters of the lanes
__device__ inline raw32 fp4_operand(raw16 w) {
  const auto a = __builtin_amdgcn_permlane16_swap(w[0], w[1], false, false), b = __builtin_amdgcn_permlane16_swap(w[2], w[3], false, false);
  const auto c = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false), d = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
  return (raw32){(int)c[0], (int)d[0], (int)c[1], (int)d[1], 0, 0, 0, 0};
}
constexpr int UNIT = 0x7f7f7f7f;  // block scales of one
template <int Q>
__device__ inline frag_cd product(raw32 w, raw32 x, frag_cd c, int blocks) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, x, c, Q == MXFP4 ? 4 : 0, 0, 0, Q == MXFP4 ? blocks : UNIT, 0, UNIT);
}

// The 8-row piece of a stage that slot i of a wave copies; where there are fewer pieces than slots a piece is copied twice (the same bytes), so
// that every wave has the same number in flight.
__device__ inline int piece_of(int wave, int i, int pieces) {
  const int p = wave + 8 * i;
  return p < pieces ? p : i > 0 ? p - 8 : p % pieces;
}

template <class F, int... U>
__device__ __attribute__((always_inline)) inline void each(const F& f, std::integer_sequence<int, U...>) { (f(std::integral_constant<int, U>{}), ...); }

// Where a tile's bytes of stage st lie behind its first (bf16 and e4m3: a stage is a block of two units, MXFP4: a unit); block: bytes from one to the next
template <int Q>
__device__ inline int stage_bytes(int st, int block) { return Q == MXFP4 ? (st >> 1) * block + (st & 1) * 1024 : st * block; }

// acc[i][j] += the wave's feature tile i x rows 16 j .. of NF row tiles (a multiple of two), over n stages of 64 columns.  MXFP4: sr, s0 and s1 of the
// block scales as wr, w0 and w1 of the weights.
template <int NF, int Q>
__device__ __attribute__((always_inline)) inline void multiply_rows(frag_cd (&acc)[2][16], rsrc_t wr, int w0, int w1, int block, rsrc_t sr, int s0, int s1, rsrc_t xr, const int (&xsrc)[4], unsigned char* ring, int n, int wave, int lane) {
  constexpr int AHEAD = ahead(NF), RING = AHEAD + 1, STAGE = NF * 2048;
  static_assert(RING * STAGE <= RING_BYTES, "ring");
  constexpr int PX = (2 * NF + 7) / 8, OPS = 4 + PX;  // pieces of x and memory operations per wave and stage
  constexpr int F = 2 * NF, NB = F / 4;               // row fragments of a stage (two k-steps), in batches of four
  const int r = lane & 15, q = lane >> 4;
  int xdst[PX];
#pragma unroll
  for (int i = 0; i < PX; ++i) xdst[i] = piece_of(wave, i, 2 * NF) * 1024;
  // rows of 128 bytes whose 16-byte chunks are swizzled by (row >> 1) & 7: a fragment read touches 16 distinct chunks per 16 lanes
  const int xo[2] = {r * 128 + ((q ^ (r >> 1)) << 4), r * 128 + (((4 + q) ^ (r >> 1)) << 4)};
  raw16 w[AHEAD][2][2];
  int scale[AHEAD][2];
  frag_ab b[2][4];  // of a batch: four row tiles' k-step, or two row tiles' both halves of a stage
  auto read = [&](int set, const unsigned char* img, int t) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int f = 4 * t + e;
      b[set][e] = *reinterpret_cast<const frag_ab*>(img + (Q == BF16 ? xo[f / NF] + f % NF * 2048 : xo[f & 1] + f / 2 * 2048));
    }
  };
  auto column = [&](int s) __attribute__((always_inline)) { return s < n ? s : n - 1; };  // of stage s (behind the end the last one is fetched again)
  // memory operations behind batch t: pieces of x spread over the stage, weights where those they replace have been multiplied
  auto fetch = [&](int t, int u, int st, unsigned char* dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PX; ++i)
      if (t == i * NB / PX) dma16(xr, xsrc[i], st * 128, dst + xdst[i]);
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (t == (k == 0 && Q == BF16 ? (NF - 1) / 4 : NB - 1)) {
        if (Q == MXFP4 && k == 1) {
          scale[u][0] = load4(sr, s0, st * 64);
          scale[u][1] = load4(sr, s1, st * 64);
        } else {
          w[u][k][0] = load16(wr, w0, stage_bytes<Q>(st, block) + k * 1024);
          w[u][k][1] = load16(wr, w1, stage_bytes<Q>(st, block) + k * 1024);
        }
      }
  };
#pragma unroll
  for (int s = 0; s < AHEAD; ++s)
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      fetch(t, s, column(s), ring + s * STAGE);
      __builtin_amdgcn_sched_barrier(0);  // (in the order of the loop: what is in flight at its top is the same on both ways in)
    }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 1) * OPS) : "memory");
  __builtin_amdgcn_s_barrier();
  read(0, ring, 0);
  int slot = 0;
  // The barrier before the last batch of stage s: everybody's pieces of stage s + 1, read from there on, have landed, and everybody's reads of stage s,
  // whose place stage s + RING takes, are answered.
  constexpr int BEFORE = [] {  // memory operations of a stage in front of its last batch
    int c = Q == BF16 && (NF - 1) / 4 < NB - 1 ? 2 : 0;
    for (int i = 0; i < PX; ++i) c += i * NB / PX < NB - 1;
    return c;
  }();
  auto stage = [&](auto uc, auto more, int s) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    const int next = slot + 1 == RING ? 0 : slot + 1;
    const unsigned char* cur = ring + slot * STAGE;
    const unsigned char* nxt = ring + next * STAGE;
    unsigned char* dst = ring + (slot == 0 ? RING - 1 : slot - 1) * STAGE;
    const int sa = column(s + AHEAD);
    raw32 a[2];
    int by[2];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const int set = (u * NB + t) & 1;
      if (t == NB - 1) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(more ? (AHEAD - 2) * OPS + BEFORE : (AHEAD - 2 - u) * OPS) : "memory");
        __builtin_amdgcn_s_barrier();
      }
      read(set ^ 1, t + 1 < NB ? cur : nxt, t + 1 < NB ? t + 1 : 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (Q == BF16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int f = 4 * t + e, k = f / NF, j = f % NF;
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(frag_ab, w[u][k][i]), b[set][e], acc[i][j], 0, 0, 0);
        }
      } else {
        if (t == 0) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            a[i] = Q == MXFP4 ? fp4_operand(w[u][0][i]) : both(w[u][0][i], w[u][1][i]);
            by[i] = Q == MXFP4 ? scale[u][i] >> (8 * q) : 0;
          }
        }
#pragma unroll
        for (int e = 0; e < 4; e += 2)
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[i][2 * t + e / 2] = product<Q>(a[i], both(b[set][e], b[set][e + 1]), acc[i][2 * t + e / 2], by[i]);
      }
      if constexpr (more) fetch(t, u, sa, dst);
      __builtin_amdgcn_sched_barrier(0);
    }
    slot = next;
  };
  int s = 0;
  static_assert(AHEAD * NB % 2 == 0, "a round of stages leaves the fragments' two sets as they were");
  for (; s + AHEAD <= n; s += AHEAD)
    each([&](auto uc) __attribute__((always_inline)) { stage(uc, std::true_type{}, s + decltype(uc)::value); }, std::make_integer_sequence<int, AHEAD>{});
  // (the last stages fetch nothing: the compiler would drop loads of weights that no stage multiplies, and the counts be wrong)
  each([&](auto uc) __attribute__((always_inline)) { if (s + decltype(uc)::value < n) stage(uc, std::false_type{}, s + decltype(uc)::value); }, std::make_integer_sequence<int, AHEAD - 1>{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no piece may be in flight when the workgroup gives its LDS back
}

template <int Q>
__device__ __attribute__((always_inline)) inline void multiply(int nf, frag_cd (&acc)[2][16], rsrc_t wr, int w0, int w1, int block, rsrc_t sr, int s0, int s1, rsrc_t xr, const int (&xsrc)[4], unsigned char* ring, int n, int wave, int lane) {
  switch (nf) {
    case 16: if constexpr (Q != MXFP4) multiply_rows<16, Q>(acc, wr, w0, w1, block, sr, s0, s1, xr, xsrc, ring, n, wave, lane); break;  // (of MXFP4 224 rows: what transposes its weights takes the registers)
    case 14: multiply_rows<14, Q>(acc, wr, w0, w1, block, sr, s0, s1, xr, xsrc, ring, n, wave, lane); break;
    case 12: multiply_rows<12, Q>(acc, wr, w0, w1, block, sr, s0, s1, xr, xsrc, ring, n, wave, lane); break;
    case 10: multiply_rows<10, Q>(acc, wr, w0, w1, block, sr, s0, s1, xr, xsrc, ring, n, wave, lane); break;
    case 8: multiply_rows<8, Q>(acc, wr, w0, w1, block, sr, s0, s1, xr, xsrc, ring, n, wave, lane); break;
    case 6: multiply_rows<6, Q>(acc, wr, w0, w1, block, sr, s0, s1, xr, xsrc, ring, n, wave, lane); break;
    case 4: multiply_rows<4, Q>(acc, wr, w0, w1, block, sr, s0, s1, xr, xsrc, ring, n, wave, lane); break;
    default: multiply_rows<2, Q>(acc, wr, w0, w1, block, sr, s0, s1, xr, xsrc, ring, n, wave, lane); break;
  }
}

// What a wave stores of its 32 features from f0 on.  acc[i][j][e]: feature 16 i + 4 q + e, row 16 j + r, to be multiplied by scale(j), and by of_features[i][e] if PER_FEATURE; gate(g, u) of a
// gated product; out(row): the row's outputs.
template <int MODE, bool PER_FEATURE, class Scale, class Gate, class Out>
__device__ __attribute__((always_inline)) inline void store_rows(const frag_cd (&acc)[2][16], const frag_cd (&of_features)[2], int rows, int f0, int lane, Scale scale, Gate gate, Out out) {
  const int r = lane & 15, q = lane >> 4;
#pragma unroll
  for (int j = 0; j < 16; j += 2) {
    if (16 * j >= rows) break;
    uint2 v[2][2];  // [row tile][half]: halves are feature tiles, or (gated) one half of the lanes has one and the other the other
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      frag_cd a = acc[0][j + t], b = acc[1][j + t];
      const float by = scale(j + t);
#pragma unroll
      for (int e = 0; e < 4; ++e) { a[e] *= PER_FEATURE ? of_features[0][e] * by : by; b[e] *= PER_FEATURE ? of_features[1][e] * by : by; }
      if constexpr (MODE == GATED) {  // a tile is 8 gate rows and their 8 up rows: the upper half of the lanes takes the other tile's
        frag_cd o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const auto gu = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[e]), __float_as_uint(b[e]), false, false);
          o[e] = gate(__uint_as_float(gu[0]), __uint_as_float(gu[1]));
        }
        v[0][t] = pack4(o);
      } else {
        if constexpr (MODE == SQUARED) {
#pragma unroll
          for (int e = 0; e < 4; ++e) { a[e] = fmaxf(a[e], 0.f); b[e] = fmaxf(b[e], 0.f); a[e] *= a[e]; b[e] *= b[e]; }
        }
        v[t][0] = pack4(a);
        v[t][1] = pack4(b);
      }
    }
#pragma unroll
    for (int t = 0; t < (MODE == GATED ? 1 : 2); ++t) {
      // sixteen lanes each: 0 the first half's (4 + 4 features), 1 the second's, 2 and 3 those eight features further
      const auto lo = __builtin_amdgcn_permlane16_swap(v[t][0].x, v[t][1].x, false, false), hi = __builtin_amdgcn_permlane16_swap(v[t][0].y, v[t][1].y, false, false);
      const raw16 o = {lo[0], hi[0], lo[1], hi[1]};
      const int row = 16 * (j + (MODE == GATED ? q & 1 : t)) + r;
      const int f = MODE == GATED ? f0 / 2 + 8 * (q >> 1) : f0 + 16 * (q & 1) + 8 * (q >> 1);
      if (row < rows) *reinterpret_cast<raw16*>(out(row) + f) = o;
    }
  }
}

// i of 0 .. n - 1, as workgroups come, to an index such that each XCD (i % 8) has a contiguous range
__device__ inline int xcd_range(int i, int n) {
  const int xcd = i & 7, qd = n >> 3, rm = n & 7;
  return (xcd < rm ? xcd * (qd + 1) : rm * (qd + 1) + (xcd - rm) * qd) + (i >> 3);
}

template <int MODE>
__global__ __launch_bounds__(512) void expert_panel_kernel(const PanelArgs p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // blockIdx -> (tile, panel): of those that exist, each XCD has a contiguous range, panels fastest (a tile's panels share its rows through that L2)
  const int nwg = p.groups.n_tiles[0] * p.n_panels;
  int id = blockIdx.x;
  {
    const int xcd = id & 7, qd = nwg >> 3, rm = nwg & 7;
    if ((id >> 3) >= qd + (xcd < rm ? 1 : 0)) return;
    id = xcd_range(id, nwg);
  }
  const int tile = id / p.n_panels, panel = id % p.n_panels;
  const int* row_of = p.groups.order + p.groups.tile_first[tile];
  const int rows = p.groups.tile_rows[tile];
  const int nf = (rows + 31) / 32 * 2, nks = p.K / 32;
  // the expert's panel; past its last feature reads give zeros (and ask no memory)
  const int ft = p.features / 16, tiles = p.N / 16 - panel * ft < ft ? p.N / 16 - panel * ft : ft;
  const rsrc_t wr = buffer_of(p.w + ((long long)p.groups.tile_expert[tile] * (p.N / 16) + panel * ft) * nks * 1024, (unsigned int)tiles * nks * 1024);
  const int w0 = 2 * wave * nks * 1024 + lane * 16, w1 = w0 + nks * 1024;
  const rsrc_t xr = buffer_of(p.x, p.x_bytes);
  int xsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 8 * piece_of(wave, i, 2 * nf) + (lane >> 3);
    const int pair = row_of[row < rows ? row : rows - 1];  // (rows past the end read the last one; nobody stores what becomes of them)
    xsrc[i] = (int)((unsigned int)(pair / p.groups.row_div) * (unsigned int)(p.ldx * 2)) + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
  }
  frag_cd acc[2][16];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[i][j] = (frag_cd){0.f, 0.f, 0.f, 0.f};
  multiply<BF16>(nf, acc, wr, w0, w1, FRAG_BLOCK * 1024, wr, 0, 0, xr, xsrc, ring, p.K / 64, wave, lane);
  const int f0 = panel * p.features + wave * 32;
  if (wave * 32 >= p.features || f0 >= p.N) return;
  store_rows<MODE, false>(acc, {}, rows, f0, lane, [](int) { return 1.f; }, [&](float g, float u) { return expert_gate(g, u, p.gate); },
                   [&](int row) { return p.y + (long long)row_of[row] * p.ldy; });
}

// ---- one matrix for all rows -----------------------------------------------------------------------------------------
// y[M, N] = x[M, K] W[N, K]^T, the matrix multiplied by panels of 256 features x `height` rows: workgroups of one matrix share what they read through
// the L2, panels in order, a panel's tiles next to one another.  The height is free in steps of 32, so that panels x tiles fill the CUs in whole rounds;
// the panels of a last round may have another.  Bound by the matrix cores and the power they draw (2048 x 28672 x 4096 of zeros takes 308 us, of random
// numbers 369) and by some 8 us per round outside the K loop.  Against tiles of up to 256 x 256 with both operands through LDS, 2048 rows:
// 28672 x 4096 411 -> 369 us (1.30 PFLOP/s), 9216 x 4096 147 -> 128, 16384 x 2048 123 -> 112, 4096 x 14336 206 -> 190, 5632 x 2048 51 -> 45.
struct DenseArgs {
  const unsigned char* w; const __bf16* x; unsigned short* y;
  int M, N, K; long long ldx, ldy;
  int height[2], tiles[2];  // of a tile, and tiles per panel: of the first `panels`, and of those behind them
  int panels;
  const float* row_ss; int ss_parts; float inv_k, eps; int gelu;
  Scales scales;
};

// of row i of a tile from row m0: the root of its mean square, and the scale of its bytes
template <int Q, class Args>
__device__ inline float scale_of_row(const Args& p, long long m) {
  float by = 1.f;
  if (p.row_ss != nullptr) {
    float ss = 0.f;
    for (int k = 0; k < p.ss_parts; ++k) ss += p.row_ss[m * p.ss_parts + k];
    by = rsqrtf(ss * p.inv_k + p.eps);
  }
  return Q == BF16 ? by : by * p.scales.x[m];
}

template <int MODE, int Q>
__device__ __attribute__((always_inline)) inline void dense_panel(const DenseArgs& p, unsigned char* ring) {
  float* const row_scale = reinterpret_cast<float*>(ring + RING_BYTES);  // [ROWS]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int first = p.panels * p.tiles[0];
  const bool behind = (int)blockIdx.x >= first;
  const int id = behind ? xcd_range(blockIdx.x - first, gridDim.x - first) : xcd_range(blockIdx.x, first);
  const int height = p.height[behind], tiles = p.tiles[behind];
  const int panel = (behind ? p.panels : 0) + id / tiles, m0 = id % tiles * height;
  const int rows = p.M - m0 < height ? p.M - m0 : height;
  const int nf = (rows + 31) / 32 * 2, nks = p.K / 32;
  const bool scaled = Q != BF16 || p.row_ss != nullptr;
  if (scaled && threadIdx.x < rows) row_scale[threadIdx.x] = scale_of_row<Q>(p, m0 + (int)threadIdx.x);
  const int have = p.N / 16 - panel * (FEATURES / 16) < FEATURES / 16 ? p.N / 16 - panel * (FEATURES / 16) : FEATURES / 16;  // feature tiles; past them reads give zeros
  const int tile_bytes = nks * (Q == MXFP4 ? 512 : 1024);
  const rsrc_t wr = buffer_of(p.w + (long long)panel * (FEATURES / 16) * tile_bytes, (unsigned int)have * tile_bytes);
  static_assert(FEATURES == 16 * FRAG_GROUP, "a panel is a group of tiles, where there are groups: the buffer ends with its last tile's bytes either way");
  const bool grouped = frag_grouped(p.N, tile_bytes / 1024, Q == MXFP4);
  const int next = frag_next(tile_bytes / 1024, grouped) * 1024, w0 = 2 * wave * next + lane * 16, w1 = w0 + next;
  const rsrc_t sr = Q == MXFP4 ? buffer_of(p.scales.blocks + (long long)panel * (FEATURES / 16) * nks * 8, (unsigned int)have * nks * 32) : wr;
  const int s0 = 2 * wave * nks * 32 + (lane & 15) * 4, s1 = s0 + nks * 32;
  const rsrc_t xr = buffer_of(p.x + m0 * p.ldx, (unsigned int)(((rows - 1) * p.ldx + p.K) * 2));
  int xsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 8 * piece_of(wave, i, 2 * nf) + (lane >> 3);
    xsrc[i] = (row < rows ? row : rows - 1) * (int)(p.ldx * 2) + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
  }
  frag_cd acc[2][16];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[i][j] = (frag_cd){0.f, 0.f, 0.f, 0.f};
  multiply<Q>(nf, acc, wr, w0, w1, frag_stride(grouped) * 1024, sr, s0, s1, xr, xsrc, ring, p.K / 64, wave, lane);
  if (scaled) __syncthreads();
  const int f0 = panel * FEATURES + wave * 32;
  if (f0 >= p.N) return;
  frag_cd of_features[2] = {{1.f, 1.f, 1.f, 1.f}, {1.f, 1.f, 1.f, 1.f}};
  if constexpr (Q == FP8) {
#pragma unroll
    for (int i = 0; i < 2; ++i) of_features[i] = *reinterpret_cast<const frag_cd*>(p.scales.w + f0 + 16 * i + 4 * (lane >> 4));
  }
  store_rows<MODE, Q == FP8>(acc, of_features, rows, f0, lane, [&](int j) { return scaled ? row_scale[16 * j + (lane & 15)] : 1.f; },
                   [&](float g, float u) {  // silu(z) = z sigmoid(z); gelu_tanh(z) = z sigmoid(2 sqrt(2 / pi) (z + 0.044715 z^3))
                     const float z = p.gelu ? 1.5957691216057308f * (g + 0.044715f * g * g * g) : g;
                     return g / (1.f + __expf(-z)) * u;
                   },
                   [&](int row) { return p.y + (m0 + row) * p.ldy; });
}

template <int MODE>
__global__ __launch_bounds__(512) void dense_panel_kernel(const DenseArgs p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
  dense_panel<MODE, BF16>(p, ring);
}

// Quantised weights and rows: the bytes of a stage and its time are those of bf16, its columns twice as many (the scaled matrix
// instruction takes 128 columns in the time of two of 32 of bf16).  A stage's fragments come in batches of two row tiles and both halves, and its weights
// stay until its last batch.  MXFP4 weights are half the bytes, a block's scales their own load; they are transposed once a stage.  Against tiles of 128 and 256 rows
// through LDS (us): e4m3 2048 x 28672 x 4096 269 -> 212 (2.27 PFLOP/s), 400 x 28672 x 4096 71 -> 49, 2048 x 6144 x 4096 67 -> 47, MXFP4 192 x 28672 x 4096
// 37 -> 27; narrow tiles e4m3 640 x 4096 x 14336 69 -> 52, MXFP4 400 x 4096 x 4096 26 -> 14.
template <int MODE, int Q>
__global__ __launch_bounds__(512) void quantised_rows_kernel(const DenseArgs p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
  dense_panel<MODE, Q>(p, ring);
}

// ---- few tiles: panels of 128 features x up to 128 rows, K shared out where that fills the CUs -----------------------------
// The same with one feature tile a wave (products of steps of some hundred rows: what counts is how fast one CU goes through its columns).  Eight stages
// ahead, weights 16 KB a stage straight to registers and rows up to 16 KB through the ring.  A CU takes in 59 GB/s of what has to come from HBM and
// 150 GB/s of what its L2 holds (measured; however much is in flight), so a stage of 64 columns is 0.27 us at best.
// By tiles of 128 x 128 of the kernel with both operands through LDS (four waves, one a SIMD) a stage was 0.52 to 0.62 us, by tiles
// of 32, 64 and 96 rows here 0.35, 0.39 and 0.44, of 128 0.53 (us: 256 x 3072 x 2048 22.5 -> 15.5, 1024 x 2048 x 2048 22.4 -> 16.8, 640 x 4096 x 4096 39.6 -> 34.2).
// Eight waves of 16 features: with two feature tiles a wave, as above, only four would share a tile of 128 and each would hold twice as many weights in flight.
struct NarrowArgs {
  const unsigned char* w; const __bf16* x; void* y;
  int M, N, K; long long ldx, ldy;
  int height, tiles, stages; long long slab;  // of a tile; tiles; of a share of K; elements of a share's sums
  const float* row_ss; int ss_parts; float inv_k, eps; int gelu;
  Scales scales;
};
enum NarrowMode { SUMS = 3 };  // beside Mode: fp32 sums of a share of K
constexpr int NARROW_FEATURES = 128, NARROW_AHEAD = 8;
__host__ __device__ constexpr int narrow_ring(int height) { return (NARROW_AHEAD + 1) * height * 128; }  // bytes: what lower tiles leave of the LDS is room for other kernels' workgroups
constexpr int NOWHERE = 0x7ffffff0;  // a lane's offset past any buffer (no scalar offset added to it comes round to its beginning)

template <int NF, int Q>
__device__ __attribute__((always_inline)) inline void multiply_narrow(frag_cd (&acc)[8], rsrc_t wr, int wlane, int w0, int block, rsrc_t sr, int slane, int s0, rsrc_t xr, const int (&xsrc)[2], unsigned char* ring, int c0, int n, int wave, int lane) {
  constexpr int AHEAD = NARROW_AHEAD, RING = AHEAD + 1, STAGE = NF * 2048;
  static_assert(RING * STAGE <= RING_BYTES, "ring");
  constexpr int PX = (2 * NF + 7) / 8, OPS = 2 + PX, BEFORE = Q == BF16 ? PX + 1 : PX;  // memory operations of a stage, and those in front of its barrier
  const int r = lane & 15, q = lane >> 4;
  int xdst[PX];
#pragma unroll
  for (int i = 0; i < PX; ++i) xdst[i] = piece_of(wave, i, 2 * NF) * 1024;
  const int xo[2] = {r * 128 + ((q ^ (r >> 1)) << 4), r * 128 + (((4 + q) ^ (r >> 1)) << 4)};
  raw16 w[AHEAD][2];
  int scale[AHEAD];
  frag_ab b[2][NF];  // of a batch: all row tiles' k-step, or half of the row tiles' both halves of a stage
  auto read = [&](int t, const unsigned char* img) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NF; ++j) b[t][j] = *reinterpret_cast<const frag_ab*>(img + (Q == BF16 ? xo[t] + j * 2048 : xo[j & 1] + (t * NF + j) / 2 * 2048));
  };
  auto weights = [&](int k, int u, int st) __attribute__((always_inline)) {
    const bool there = st < n;
    if (Q == MXFP4 && k == 1) scale[u] = load4(sr, there ? slane : NOWHERE, s0 + (c0 + st) * 64);
    else w[u][k] = load16(wr, there ? wlane : NOWHERE, w0 + stage_bytes<Q>(c0 + st, block) + k * 1024);
  };
  auto multiply = [&](int t, int u) __attribute__((always_inline)) {
    if constexpr (Q == BF16) {
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(frag_ab, w[u][t]), b[t][j], acc[j], 0, 0, 0);
    } else {
      const raw32 a = Q == MXFP4 ? fp4_operand(w[u][0]) : both(w[u][0], w[u][1]);
      const int by = Q == MXFP4 ? scale[u] >> (8 * q) : 0;
#pragma unroll
      for (int j = 0; j < NF; j += 2) acc[(t * NF + j) / 2] = product<Q>(a, both(b[t][j], b[t][j + 1]), acc[(t * NF + j) / 2], by);
    }
  };
  // stages behind the end: offsets past the buffers, where reads give zeros and ask no memory (the same number is in flight as long as stages are fetched)
  auto fetch = [&](int k, int u, int st, unsigned char* dst) __attribute__((always_inline)) {
    const bool there = st < n;
    if (k == 0) {
#pragma unroll
      for (int i = 0; i < PX; ++i) dma16(xr, there ? xsrc[i] : NOWHERE, (c0 + st) * 128, dst + xdst[i]);
    }
    if (Q == BF16) weights(k, u, st);  // (else both are multiplied to the stage's end)
    else if (k == 1) { weights(0, u, st); weights(1, u, st); }
  };
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) {
    fetch(0, s, s, ring + s * STAGE);
    __builtin_amdgcn_sched_barrier(0);
    fetch(1, s, s, ring + s * STAGE);
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 1) * OPS) : "memory");
  __builtin_amdgcn_s_barrier();
  read(0, ring);
  int slot = 0;
  auto stage = [&](auto uc, auto more, int s) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    const int next = slot + 1 == RING ? 0 : slot + 1;
    unsigned char* dst = ring + (slot == 0 ? RING - 1 : slot - 1) * STAGE;
    read(1, ring + slot * STAGE);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0, u);
    if constexpr (more) fetch(0, u, s + AHEAD, dst);
    __builtin_amdgcn_sched_barrier(0);
    // everybody's pieces of the next stage, read from here on, have landed, and everybody's reads of this one, whose place the next fetch takes, are answered
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(more ? (AHEAD - 2) * OPS + BEFORE : (AHEAD - 2 - u) * OPS) : "memory");
    __builtin_amdgcn_s_barrier();
    read(0, ring + next * STAGE);
    __builtin_amdgcn_sched_barrier(0);
    multiply(1, u);
    if constexpr (more) fetch(1, u, s + AHEAD, dst);
    __builtin_amdgcn_sched_barrier(0);
    slot = next;
  };
  int s = 0;
  for (; s + AHEAD <= n; s += AHEAD)
    each([&](auto uc) __attribute__((always_inline)) { stage(uc, std::true_type{}, s + decltype(uc)::value); }, std::make_integer_sequence<int, AHEAD>{});
  // (the last stages fetch nothing, as above)
  each([&](auto uc) __attribute__((always_inline)) { if (s + decltype(uc)::value < n) stage(uc, std::false_type{}, s + decltype(uc)::value); }, std::make_integer_sequence<int, AHEAD - 1>{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no piece may be in flight when the workgroup gives its LDS back
}

template <int MODE, int Q>
__global__ __launch_bounds__(512) void narrow_tiles_kernel(const NarrowArgs p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
  float* const row_scale = reinterpret_cast<float*>(ring + narrow_ring(p.height));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // blockIdx -> (share of K, panel, tile): each XCD has a contiguous range, a panel's tiles next to one another (they share its weights through that L2)
  const int id = xcd_range(blockIdx.x, gridDim.x), panels = p.N / NARROW_FEATURES;
  const int m0 = id % p.tiles * p.height, panel = id / p.tiles % panels, share = id / p.tiles / panels;
  const int rows = p.M - m0 < p.height ? p.M - m0 : p.height, nf = (rows + 31) / 32 * 2, nks = p.K / 32;
  const int c0 = share * p.stages, n = p.K / 64 - c0 < p.stages ? p.K / 64 - c0 : p.stages;
  const bool scaled = Q != BF16 || (MODE != SUMS && p.row_ss != nullptr);  // (sums: by the scale of the bytes alone)
  if (scaled && threadIdx.x < rows) row_scale[threadIdx.x] = MODE == SUMS ? p.scales.x[m0 + (int)threadIdx.x] : scale_of_row<Q>(p, m0 + (int)threadIdx.x);
  const int tile_bytes = nks * (Q == MXFP4 ? 512 : 1024);
  // (a group of tiles is two panels)
  const bool grouped = frag_grouped(p.N, tile_bytes / 1024, Q == MXFP4);
  const int from = grouped ? panel / (FRAG_GROUP * 16 / NARROW_FEATURES) * FRAG_GROUP : panel * (NARROW_FEATURES / 16), have = grouped ? FRAG_GROUP : NARROW_FEATURES / 16;
  const rsrc_t wr = buffer_of(p.w + (long long)from * tile_bytes, (unsigned int)have * tile_bytes);
  const rsrc_t sr = Q == MXFP4 ? buffer_of(p.scales.blocks + (long long)panel * (NARROW_FEATURES / 16) * nks * 8, (unsigned int)(NARROW_FEATURES / 16) * nks * 32) : wr;
  const rsrc_t xr = buffer_of(p.x + m0 * p.ldx, (unsigned int)(((rows - 1) * p.ldx + p.K) * 2));
  int xsrc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 8 * piece_of(wave, i, 2 * nf) + (lane >> 3);
    xsrc[i] = (row < rows ? row : rows - 1) * (int)(p.ldx * 2) + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
  }
  frag_cd acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = (frag_cd){0.f, 0.f, 0.f, 0.f};
  const int w0 = (panel * (NARROW_FEATURES / 16) - from + wave) * frag_next(tile_bytes / 1024, grouped) * 1024, s0 = wave * nks * 32;
  switch (nf) {
    case 8: multiply_narrow<8, Q>(acc, wr, lane * 16, w0, frag_stride(grouped) * 1024, sr, (lane & 15) * 4, s0, xr, xsrc, ring, c0, n, wave, lane); break;
    case 6: multiply_narrow<6, Q>(acc, wr, lane * 16, w0, frag_stride(grouped) * 1024, sr, (lane & 15) * 4, s0, xr, xsrc, ring, c0, n, wave, lane); break;
    case 4: multiply_narrow<4, Q>(acc, wr, lane * 16, w0, frag_stride(grouped) * 1024, sr, (lane & 15) * 4, s0, xr, xsrc, ring, c0, n, wave, lane); break;
    default: multiply_narrow<2, Q>(acc, wr, lane * 16, w0, frag_stride(grouped) * 1024, sr, (lane & 15) * 4, s0, xr, xsrc, ring, c0, n, wave, lane); break;
  }
  if (scaled) __syncthreads();
  // acc[j][e]: feature 4 q + e of the wave's 16, row 16 j + r
  const int r = lane & 15, q = lane >> 4, f0 = panel * NARROW_FEATURES + wave * 16;
  frag_cd of_features = {1.f, 1.f, 1.f, 1.f};
  if constexpr (Q == FP8) of_features = *reinterpret_cast<const frag_cd*>(p.scales.w + f0 + 4 * q);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int row = 16 * j + r;
    if (16 * j >= rows) break;
    const long long m = m0 + row;
    frag_cd v = acc[j];
    if (scaled) {
      const frag_cd by = of_features * row_scale[row];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= by[e];
    }
    if constexpr (MODE == SUMS) {
      if (row < rows) *reinterpret_cast<frag_cd*>(reinterpret_cast<float*>(p.y) + share * p.slab + m * p.ldy + f0 + 4 * q) = v;
    } else {
      unsigned short* const y = reinterpret_cast<unsigned short*>(p.y) + m * p.ldy;
      if constexpr (MODE == GATED) {  // a tile is 8 gate rows and their 8 up rows: lanes q < 2 have gates, q + 2 the ups of the same features
        frag_cd o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float up = __shfl_xor(v[e], 32, 64), z = p.gelu ? 1.5957691216057308f * (v[e] + 0.044715f * v[e] * v[e] * v[e]) : v[e];
          o[e] = v[e] / (1.f + __expf(-z)) * up;
        }
        if (q < 2 && row < rows) *reinterpret_cast<uint2*>(y + f0 / 2 + 4 * q) = pack4(o);
      } else {
        if constexpr (MODE == SQUARED) {
#pragma unroll
          for (int e = 0; e < 4; ++e) { v[e] = fmaxf(v[e], 0.f); v[e] *= v[e]; }
        }
        if (row < rows) *reinterpret_cast<uint2*>(y + f0 + 4 * q) = pack4(v);
      }
    }
  }
}

template <auto KERNEL, class Args>
int launch(const Args& a, int grid, hipStream_t s, int lds = RING_BYTES + ROWS * 4) {
  constexpr int LDS = RING_BYTES + ROWS * 4;
  static const hipError_t lds_ok = hipFuncSetAttribute((const void*)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (lds_ok != hipSuccess) return -2;
  hipLaunchKernelGGL(KERNEL, dim3(grid), dim3(512), lds, s, a);
  return (int)hipGetLastError();
}

template <int Q>
int launch_narrow(const NarrowArgs& a, int epi, int grid, hipStream_t s) {
  const int lds = narrow_ring(a.height) + a.height * 4;
  switch (epi) {
    case 0: return launch<narrow_tiles_kernel<PLAIN, Q>>(a, grid, s, lds);
    case 1: return launch<narrow_tiles_kernel<SUMS, Q>>(a, grid, s, lds);
    case 2: case 4: return launch<narrow_tiles_kernel<GATED, Q>>(a, grid, s, lds);
    case 5: if constexpr (Q == BF16) return launch<narrow_tiles_kernel<SQUARED, BF16>>(a, grid, s, lds);
  }
  return -1;
}

// Whether there are the scales that numbers need; of bytes, K and ldx in pairs.
bool in_pairs(int numbers, int& K, long long& ldx, const float* w_scale, const float* x_scale, const int* blocks) {
  if (numbers == BF16) return true;
  if ((numbers != FP8 && numbers != MXFP4) || (K & 127) || (ldx & 15) || !x_scale || (numbers == FP8 ? !w_scale || ((uintptr_t)w_scale & 15) : !blocks)) return false;
  K /= 2; ldx /= 2;
  return true;
}

}  // namespace

extern "C" {

// Wp holds the packed matrices [N, K] of all experts, one behind the other; row i of the tiled rows (kve_group, at most 256 a tile) is pair order[i],
// x's row is pair / row_div, y's row the pair.  mode 1: bf16 y[pairs, N / 2] with the experts' gate; 2: bf16 max(y, 0)^2 [pairs, N]; 0: bf16 y[pairs, N].
// features: of a panel, 256 or 128 (then four waves of a workgroup copy rows only).  N % 32 == 0, K % 64 == 0, rows of x and y of whole 16-byte pieces;
// x_rows rows of x must lie within 2 GiB (offsets are 32-bit).
int kv_expert_panels(const void* Wp, const void* x, void* y, int N, int K, long long ldx, long long ldy, long long x_rows, int mode, float limit, float slope, float shift, int* order, int* tiles, int max_tiles, int* n_tiles,
                     int row_div, int features, hipStream_t stream) {
  if ((features != FEATURES && features != FEATURES / 2) || N <= 0 || K <= 0 || (N & 31) || (K & 63) || K > (1 << 21) || (ldx & 7) || (ldy & 7) || max_tiles <= 0 || row_div <= 0 || x_rows <= 0 || mode < PLAIN || mode > SQUARED) return -1;
  const long long bytes = ((x_rows - 1) * ldx + K) * 2;
  if (bytes >= (1ll << 31) || ldx < K) return -1;
  PanelArgs a;
  a.w = (const unsigned char*)Wp; a.x = (const __bf16*)x; a.y = (unsigned short*)y;
  a.N = N; a.K = K; a.ldx = ldx; a.ldy = ldy;
  a.n_panels = (N + features - 1) / features;
  a.features = features;
  a.x_bytes = (unsigned int)bytes;
  a.gate = ExpertGate{limit, slope, shift};
  a.groups = GroupedRows{order, tiles, tiles + max_tiles, tiles + 2 * max_tiles, n_tiles, max_tiles, row_div};
  const int grid = max_tiles * a.n_panels;
  return mode == GATED ? launch<expert_panel_kernel<GATED>>(a, grid, stream) : mode == SQUARED ? launch<expert_panel_kernel<SQUARED>>(a, grid, stream) : launch<expert_panel_kernel<PLAIN>>(a, grid, stream);
}

// Wp: one packed matrix [N, K]; epi 0: bf16 y[M, N], 2: the gated y[M, N / 2] with silu, 4: with gelu (tanh form), 5: max(y, 0)^2 [M, N].  The first
// `panels` of the ceil(N / 256) panels are cut into tiles of `height` rows, those behind them of `height_behind` (multiples of 32 up to 256, of MXFP4 224).  row_ss
// (or null): fp32 [M][ss_parts] whose sums over K are the rows' mean squares; products are divided by the root of that.
// N % 32 == 0, K % 64 == 0, rows of x and y of whole 16-byte pieces that start at such; 256 rows of x must lie within 2 GiB.
// numbers (Numbers): of bytes, K and ldx count them (K % 128 == 0, no epi 5), x_scale[M] are the rows' scales, w_scale[N] those of e4m3 weights (in the order
// of whose fragments x then is), blocks those of MXFP4 ones (x in order).
int kv_dense_panels(const void* Wp, const void* x, void* y, int M, int N, int K, long long ldx, long long ldy, int epi, int height, int panels, int height_behind, const float* row_ss, int ss_parts, float eps,
                    int numbers, const float* w_scale, const float* x_scale, const int* blocks, hipStream_t stream) {
  const float inv_k = 1.f / (float)K;
  if (!in_pairs(numbers, K, ldx, w_scale, x_scale, blocks)) return -1;
  if (M <= 0 || N <= 0 || K <= 0 || (N & 31) || (K & 63) || K > (1 << 21) || (ldx & 7) || (ldy & 7) || ldx < K || ldx >= (1 << 22) || ((uintptr_t)x & 15) || ((uintptr_t)y & 15)) return -1;
  const int all = (N + FEATURES - 1) / FEATURES;
  for (int h : {height, height_behind})
    if (h <= 0 || h > (numbers == MXFP4 ? ROWS - 32 : ROWS) || (h & 31)) return -1;
  if (panels < 0 || panels > all) return -1;
  DenseArgs a;
  a.w = (const unsigned char*)Wp; a.x = (const __bf16*)x; a.y = (unsigned short*)y;
  a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldy = ldy;
  a.height[0] = height; a.height[1] = height_behind;
  a.tiles[0] = (M + height - 1) / height; a.tiles[1] = (M + height_behind - 1) / height_behind;
  a.panels = panels;
  a.row_ss = row_ss; a.ss_parts = ss_parts; a.inv_k = inv_k; a.eps = eps; a.gelu = epi == 4;
  a.scales = Scales{w_scale, x_scale, blocks};
  const long long grid = (long long)panels * a.tiles[0] + (long long)(all - panels) * a.tiles[1];
  if (grid > 0x7fffffffll) return -1;
  const bool gated = epi == 2 || epi == 4;
  if (!gated && epi != 0 && (epi != 5 || numbers != BF16)) return -1;
  switch (numbers) {
    case FP8: return gated ? launch<quantised_rows_kernel<GATED, FP8>>(a, (int)grid, stream) : launch<quantised_rows_kernel<PLAIN, FP8>>(a, (int)grid, stream);
    case MXFP4: return gated ? launch<quantised_rows_kernel<GATED, MXFP4>>(a, (int)grid, stream) : launch<quantised_rows_kernel<PLAIN, MXFP4>>(a, (int)grid, stream);
  }
  return gated ? launch<dense_panel_kernel<GATED>>(a, (int)grid, stream) : epi == 5 ? launch<dense_panel_kernel<SQUARED>>(a, (int)grid, stream) : launch<dense_panel_kernel<PLAIN>>(a, (int)grid, stream);
}

// Wp: one packed matrix [N, K].  Tiles of `height` rows (a multiple of 32 up to 128) x 128 features; epi 0, 2, 4, 5 as above, 1: fp32 sums
// [splits][M][N] of shares of `stages` x 64 columns (128 of bytes; `slab` elements apart; other epilogues: one share).  N % 128 == 0, the rest as above.
int kv_narrow_tiles(const void* Wp, const void* x, void* y, int M, int N, int K, long long ldx, long long ldy, int epi, int height, int splits, int stages, long long slab, const float* row_ss, int ss_parts, float eps,
                    int numbers, const float* w_scale, const float* x_scale, const int* blocks, hipStream_t stream) {
  const float inv_k = 1.f / (float)K;
  if (!in_pairs(numbers, K, ldx, w_scale, x_scale, blocks)) return -1;
  if (M <= 0 || N <= 0 || K <= 0 || N % NARROW_FEATURES || (K & 63) || K > (1 << 21) || (ldx & 7) || ldx < K || ldx >= (1 << 22) || ((uintptr_t)x & 15) || ((uintptr_t)y & 15) || (ldy & 3)) return -1;
  if (height <= 0 || height > 128 || (height & 31) || splits <= 0 || stages <= 0 || (long long)(splits - 1) * stages >= K / 64 || (long long)splits * stages < K / 64 || (epi != 1 && splits != 1)) return -1;
  NarrowArgs a;
  a.w = (const unsigned char*)Wp; a.x = (const __bf16*)x; a.y = y;
  a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldy = ldy;
  a.height = height; a.tiles = (M + height - 1) / height; a.stages = stages; a.slab = slab;
  a.row_ss = row_ss; a.ss_parts = ss_parts; a.inv_k = inv_k; a.eps = eps; a.gelu = epi == 4;
  a.scales = Scales{w_scale, x_scale, blocks};
  const long long grid = (long long)splits * (N / NARROW_FEATURES) * a.tiles;
  if (grid > 0x7fffffffll) return -1;
  switch (numbers) {
    case FP8: return launch_narrow<FP8>(a, epi, (int)grid, stream);
    case MXFP4: return launch_narrow<MXFP4>(a, epi, (int)grid, stream);
  }
  return launch_narrow<BF16>(a, epi, (int)grid, stream);
}

}  // extern "C"
