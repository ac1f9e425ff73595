// Latency statistics kernels for gfx950 (MI355X): LDS-binned histograms and exact quantiles.
//
// What this replaces: the reference reduces request/token latencies on the CPU by
// sorting a Python list once per percentile (analyze.py:59-81, ~25 sorts per run) and
// by a Python loop for its 20-bin histograms (analyze.py:84-122).  At per-token
// granularity (10^6..10^8 inter-token gaps per run) that is the harness's only
// compute-bound path, so it lives on the GPU:
//
//   kv_stream_hist      streaming histogram with 2048 log-spaced bins per metric, plus
//                        count / sum / min / max, accumulated into persistent device
//                        state (launch it on every new slice of token events; the state
//                        is never re-read from the samples).  Per-wavefront private
//                        sub-histograms live in LDS (4 waves x 2048 bins x 4 B = 32 KiB of
//                        the CU's 160 KiB) and are updated with LDS atomics; one global
//                        atomic per non-empty bin per workgroup flushes them.
//   kv_select_quantiles  exact order statistics by MSD radix select on order-preserving
//                        integer keys: 11-bit digits, i.e. the same 2048-bin LDS histogram,
//                        restricted to samples whose higher digits match the prefix of a
//                        target rank; the last workgroup of a pass turns the bin counts
//                        into the next prefix (kv_radix_pass_*: a launch of its own, for samples
//                        spread over ranks).  Up to 8 ranks are tracked at once (floor and
//                        ceil rank of p50/p95/p99), so three quantiles of 10^8 doubles cost 6
//                        streaming passes and no sort.  Rows of 16 k (doubles: 512) to 32 M samples take two
//                        passes instead, between values that a sample of them gives (kv_split_quantiles).
//                        The result is bit-exact: the CPU
//                        interpolates between the two selected samples exactly like
//                        analyze.py does.
//   kv_equal_hist       the 20-bin equal-width histogram over [min, max] (last bin closed),
//                        LDS-binned the same way, with min/max read from device memory.
//
// Batching: samples are a row-major [n_metrics, row_stride] matrix; NaN entries are
// skipped (analyze.py drops NaNs), so ragged metrics are NaN-padded and one launch with
// grid.y = metric handles latency / TTFT / TLLT / generation / per-token x all / cold /
// warm together.
//
// Wavefront width is 64 on CDNA; workgroups are 256 threads = 4 waves, one per SIMD.

#include <algorithm>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define KV_BINS 2048
#define KV_WAVES 4
#define KV_THREADS 256
#define KV_MAX_RANKS 8

namespace {

// ---------------------------------------------------------------------------------
// order-preserving keys
template <typename T> struct KeyOf;
template <> struct KeyOf<float> {
  using type = uint32_t;
  static constexpr int bits = 32;
  __device__ static inline uint32_t key(float v) {
    uint32_t b = __float_as_uint(v);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  }
};
template <> struct KeyOf<double> {
  using type = uint64_t;
  static constexpr int bits = 64;
  __device__ static inline uint64_t key(double v) {
    uint64_t b = (uint64_t)__double_as_longlong(v);
    return (b & 0x8000000000000000ull) ? ~b : (b | 0x8000000000000000ull);
  }
};

// log-spaced bin of a positive value: 2048 bins over [2^lo_log2, 2^hi_log2)
__device__ inline int log_bin(float v, float lo_log2, float inv_step) {
  if (!(v > 0.f)) return 0;
  float f = (__log2f(v) - lo_log2) * inv_step;
  int b = (int)f;
  return b < 0 ? 0 : (b >= KV_BINS ? KV_BINS - 1 : b);
}

// Histogram increment with wave-level aggregation of the common bin.  Latency samples
// are heavily clustered (most of a wave's 64 lanes hit the same bin), which would
// serialise 64 LDS atomics on one address; instead the lanes that share the first
// active lane's bin elect one lane to add their population count.  Must be called by
// exactly the lanes that hold a valid sample (the active set is the participant set).
__device__ inline void hist_add(unsigned int* h, unsigned int d) {
  unsigned int d0 = __builtin_amdgcn_readfirstlane(d);
  bool same = d == d0;
  unsigned long long mask = __ballot(same);
  if (same) {
    if ((int)__lane_id() == __ffsll((long long)mask) - 1) atomicAdd(&h[d0], (unsigned int)__popcll(mask));
  } else {
    atomicAdd(&h[d], 1u);
  }
}

__device__ inline double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ inline unsigned long long wave_sum_u64(unsigned long long v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
template <typename K> __device__ inline K wave_min(K v) {
  for (int o = 32; o > 0; o >>= 1) { K w = __shfl_xor(v, o, 64); v = w < v ? w : v; }
  return v;
}
template <typename K> __device__ inline K wave_max(K v) {
  for (int o = 32; o > 0; o >>= 1) { K w = __shfl_xor(v, o, 64); v = w > v ? w : v; }
  return v;
}

// Per-metric persistent state of the streaming histogram.
struct StreamState {
  unsigned long long count;
  double sum;
  unsigned long long min_key;  // order-preserving key of the minimum (init: ~0)
  unsigned long long max_key;  // order-preserving key of the maximum (init: 0)
};

// ---------------------------------------------------------------------------------
// kv_stream_hist: x[n_metrics][row_stride] (first n valid columns), hist[n_metrics][2048]
template <typename T>
__global__ __launch_bounds__(KV_THREADS) void stream_hist_kernel(const T* __restrict__ x, long long n, long long row_stride,
                                                                 unsigned int* __restrict__ hist, StreamState* __restrict__ state,
                                                                 float lo_log2, float inv_step) {
  __shared__ unsigned int lds[KV_WAVES * KV_BINS];
  const int tid = threadIdx.x, wave = tid >> 6;
  const int m = blockIdx.y;
  for (int i = tid; i < KV_WAVES * KV_BINS; i += KV_THREADS) lds[i] = 0;
  __syncthreads();

  const T* row = x + (long long)m * row_stride;
  unsigned int* my = lds + wave * KV_BINS;
  using KT = typename KeyOf<T>::type;
  unsigned long long cnt = 0;
  double sum = 0.0;
  KT kmin = ~(KT)0, kmax = 0;

  constexpr int VEC = 16 / sizeof(T);  // 16-byte loads: 4 floats or 2 doubles per lane
  const long long nvec = n / VEC;
  const long long stride = (long long)gridDim.x * KV_THREADS;
  struct alignas(16) Pack { T v[VEC]; };
  const bool aligned = (((uintptr_t)row) & 15) == 0;
  if (aligned) {
    const Pack* pv = reinterpret_cast<const Pack*>(row);
    auto consume = [&](const Pack& p) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        T v = p.v[j];
        if (v == v) {
          hist_add(my, (unsigned int)log_bin((float)v, lo_log2, inv_step));
          ++cnt; sum += (double)v;
          KT k = KeyOf<T>::key(v);
          kmin = k < kmin ? k : kmin; kmax = k > kmax ? k : kmax;
        }
      }
    };
    // four 16-byte loads in flight per lane: the LDS atomics of one pack hide the latency of
    // the next loads instead of serialising load -> bin -> load
    long long i = (long long)blockIdx.x * KV_THREADS + tid;
    for (; i + 3 * stride < nvec; i += 4 * stride) {
      const Pack p0 = pv[i], p1 = pv[i + stride], p2 = pv[i + 2 * stride], p3 = pv[i + 3 * stride];
      consume(p0); consume(p1); consume(p2); consume(p3);
    }
    for (; i < nvec; i += stride) consume(pv[i]);
  }
  // tail (or everything, when the row is not 16-byte aligned)
  for (long long i = (aligned ? nvec * VEC : 0) + (long long)blockIdx.x * KV_THREADS + tid; i < n; i += stride) {
    T v = row[i];
    if (v == v) {
      hist_add(my, (unsigned int)log_bin((float)v, lo_log2, inv_step));
      ++cnt; sum += (double)v;
      KT k = KeyOf<T>::key(v);
      kmin = k < kmin ? k : kmin; kmax = k > kmax ? k : kmax;
    }
  }
  __syncthreads();
  unsigned int* gh = hist + (long long)m * KV_BINS;
  for (int b = tid; b < KV_BINS; b += KV_THREADS) {
    unsigned int c = lds[b] + lds[KV_BINS + b] + lds[2 * KV_BINS + b] + lds[3 * KV_BINS + b];
    if (c) atomicAdd(&gh[b], c);
  }
  // scalars: wave reduction, then one atomic per wave
  cnt = wave_sum_u64(cnt);
  sum = wave_sum(sum);
  kmin = wave_min<KT>(kmin);
  kmax = wave_max<KT>(kmax);
  if ((tid & 63) == 0 && cnt) {
    StreamState* s = state + m;
    atomicAdd(&s->count, cnt);
    atomicAdd(&s->sum, sum);
    // widen 32-bit keys so one state layout serves both dtypes
    unsigned long long k0 = (unsigned long long)kmin << (64 - KeyOf<T>::bits);
    unsigned long long k1 = (unsigned long long)kmax << (64 - KeyOf<T>::bits);
    atomicMin(&s->min_key, k0);
    atomicMax(&s->max_key, k1);
  }
}

// ---------------------------------------------------------------------------------
// Radix select.  Per metric: U distinct prefixes (U <= 8).  hist[m][u][2048].
struct RadixState {
  unsigned long long prefix[KV_MAX_RANKS];  // key bits decided so far (high bits), per rank
  unsigned long long k[KV_MAX_RANKS];       // rank remaining inside the prefix
  unsigned long long uniq[KV_MAX_RANKS];    // distinct prefixes for the next histogram pass
  int slot[KV_MAX_RANKS];                   // rank -> index into uniq
  int n_uniq;
  int n_ranks;
  unsigned long long count;                 // samples
};

// Ranks from quantile levels: pos = p*(n-1), ranks floor(pos) and ceil(pos) — the definition of analyze.py:75-81.
struct Levels { double p[KV_MAX_RANKS / 2]; int n; };
__device__ inline unsigned long long rank_of(const Levels& lv, int r, unsigned long long n) {
  double p = lv.p[r >> 1];
  p = p < 0.0 ? 0.0 : (p > 1.0 ? 1.0 : p);
  const double pos = p * (double)(n - 1);
  return (unsigned long long)((r & 1) ? ceil(pos) : floor(pos));
}

// A pass counts the 11-bit digits behind each distinct prefix.  Latencies are clustered (a first digit is a quarter of an octave, and most
// of a wave's 64 samples share it), so what bounds a pass is LDS atomics that meet on one address: a workgroup of 16 waves keeps the histogram
// 16 times (fewer times when there are more prefixes), bin by bin next to each other, and a lane uses copy lane % 16 — at most 4 lanes
// of an instruction meet, in different banks.  One global atomic per non-empty bin and workgroup adds it up, so there are few workgroups,
// one a CU.  3 x 4 M floats: 25 us a pass, picking included, where one histogram a wave with ballot aggregation took 48 and picking 14 more.
constexpr int SEL_THREADS = 1024;
constexpr int SEL_WORDS = 16 * KV_BINS;  // LDS words of the copies: 128 KiB
constexpr int PER = KV_MAX_RANKS * KV_BINS / SEL_THREADS;  // bins per thread, of all prefixes
constexpr int SEL_ROW = KV_BINS + KV_BINS / 32;  // LDS words of a summed histogram, 33 per 32 bins (a lane's 32 bins then start in a bank of their own)

// (clearing and summing the copies takes a few us: a few thousand samples meet seldom enough in fewer)
__device__ inline int log2_copies(int prefixes, long long n) {
  const int room = prefixes <= 1 ? 4 : prefixes == 2 ? 3 : prefixes <= 4 ? 2 : 1, wanted = n <= 2048 ? 0 : n <= 8192 ? 2 : 4;
  return room < wanted ? room : wanted;
}

// visit(v) for the samples first, first + stride, ... (in 16-byte pieces) of a row, `first` consecutive in a wave.  All lanes of a wave visit together:
// those that are past the end, a NaN.  after_piece(): after 16 bytes of each lane, or less.
struct Nothing { __device__ void operator()() const {} };
template <typename T, typename F, typename G = Nothing>
__device__ __forceinline__ void for_samples(const T* __restrict__ row, long long n, long long first, long long stride, F&& visit, G&& after_piece = G{}) {
  constexpr int VEC = 16 / sizeof(T);
  struct alignas(16) Pack { T v[VEC]; };
  const T none = (T)__builtin_nanf("");
  const long long lane = threadIdx.x & 63;
  // (rows need not start at a multiple of 16 bytes: the samples in front of the first whole piece and behind the last go one by one)
  long long head = (VEC - (long long)((uintptr_t)row / sizeof(T)) % VEC) % VEC;
  head = head < n ? head : n;
  const Pack* pv = reinterpret_cast<const Pack*>(row + head) + lane;
  const long long nvec = (n - head) / VEC, tail = head + nvec * VEC;
  auto visit_pack = [&](const Pack& p) {
#pragma unroll
    for (int j = 0; j < VEC; ++j) visit(p.v[j]);
    after_piece();
  };
  constexpr int AHEAD = 4;  // loads in flight per lane while the ones before are counted
  Pack p[AHEAD];
  // (of the wave's first lane: the loops are the same for all)
  const long long start = (long long)((unsigned long long)(unsigned int)__builtin_amdgcn_readfirstlane((int)(first >> 32)) << 32 | (unsigned int)__builtin_amdgcn_readfirstlane((int)first));
  long long i = start;
  if (i + (AHEAD - 1) * stride + 63 < nvec) {
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) p[k] = pv[i + k * stride];
    for (;;) {
      i += AHEAD * stride;
      const bool more = i + (AHEAD - 1) * stride + 63 < nvec;
      Pack q[AHEAD];
      if (more) {
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) q[k] = pv[i + k * stride];
      }
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) visit_pack(p[k]);
      if (!more) break;
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) p[k] = q[k];
    }
  }
  for (; i < nvec; i += stride) {
    Pack q;
#pragma unroll
    for (int j = 0; j < VEC; ++j) q.v[j] = none;
    if (i + lane < nvec) q = pv[i];
    visit_pack(q);
  }
  if (start < head) visit(first < head ? row[first] : none);
  if (tail + start < n) visit(tail + first < n ? row[tail + first] : none);
  after_piece();
}

// counts the digits of the samples first, first + stride, ... (in 16-byte pieces) of a row into h[prefix][bin][copy]; MOST: at least U prefixes
// (0: the first pass, which has none)
template <typename T, int MOST>
__device__ void count_digits(const T* __restrict__ row, long long n, long long first, long long stride, unsigned int* h, const unsigned long long* uniq, int U, int shift, int digit_bits) {
  using KT = typename KeyOf<T>::type;
  const int cl = log2_copies(U, n), copy = threadIdx.x & ((1 << cl) - 1);
  const KT dmask = (KT)((1u << digit_bits) - 1u);
  const int hi_shift = shift + digit_bits;  // bits above the current digit
  KT pre[MOST > 0 ? MOST : 1] = {};
#pragma unroll
  for (int u = 0; u < MOST; ++u) pre[u] = (KT)((KT)(uniq[u < U ? u : 0] >> (64 - KeyOf<T>::bits)) >> hi_shift);  // (unused ones repeat the first)
  for_samples(row, n, first, stride, [&](T v) {
    if (!(v == v)) return;
    const KT key = KeyOf<T>::key(v);
    int bin = (int)((key >> shift) & dmask);
    if constexpr (MOST > 0) {
      const KT hi = (KT)(key >> hi_shift);
      int at = -1;
#pragma unroll
      for (int u = MOST - 1; u >= 0; --u) at = hi == pre[u] ? u : at;
      if (at < 0) return;
      bin += at * KV_BINS;
    }
    atomicAdd(&h[(bin << cl) + copy], 1u);
  });
}

// the copies of bin i (counted over all prefixes)
__device__ inline unsigned int sum_copies(const unsigned int* h, int i, int cl) {
  if (cl < 2) return cl == 0 ? h[i] : h[2 * i] + h[2 * i + 1];
  unsigned int c = 0;
  for (int k = 0; k < 1 << cl; k += 4) {
    const uint4 v = *reinterpret_cast<const uint4*>(h + (i << cl) + k);
    c += v.x + v.y + v.z + v.w;
  }
  return c;
}

// The whole workgroup: every rank picks the bin that holds it, appends the digit to its prefix and keeps its rank inside; then the distinct
// prefixes.  A wave per rank.  sums: LDS, [prefix][SEL_ROW].  `levels` (first pass): the ranks follow from the number of samples counted.
__device__ void pick_digits(RadixState* s, const unsigned int* sums, int shift, bool first_pass, const Levels* levels) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int R = levels ? 2 * levels->n : s->n_ranks;
  if (wave < R) {
    const unsigned int* p = sums + (first_pass ? 0 : s->slot[wave]) * SEL_ROW + lane * 33;
    unsigned int t[32];
    unsigned long long local = 0;
#pragma unroll
    for (int j = 0; j < 32; ++j) t[j] = p[j];
#pragma unroll
    for (int j = 0; j < 32; ++j) local += t[j];
    unsigned long long upto = local;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned long long v = __shfl_up(upto, o, 64);
      if (lane >= o) upto += v;
    }
    const unsigned long long total = __shfl(upto, 63, 64);
    const unsigned long long k = levels ? (total ? rank_of(*levels, wave, total) : 0) : s->k[wave];
    unsigned long long run = upto - local;
    if (k >= run && k < upto) {
      int bin = 0;
      unsigned long long below = 0;
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        if (k >= run && k < run + t[j]) { bin = lane * 32 + j; below = run; }
        run += t[j];
      }
      s->prefix[wave] |= (unsigned long long)bin << shift;
      s->k[wave] = k - below;
    }
    if (levels && wave == 0 && lane == 0) s->count = total;
  }
  __syncthreads();
  if (wave == 0) {  // a lane per rank: the first rank with the same prefix, and how many such firsts there are in front of it
    const unsigned long long mine = s->prefix[lane < KV_MAX_RANKS ? lane : 0];
    int first = lane;
#pragma unroll
    for (int r = KV_MAX_RANKS - 1; r >= 0; --r) {
      const unsigned long long other = __shfl(mine, r, 64);
      if (r < R && other == mine) first = r;
    }
    const unsigned long long firsts = __ballot(lane < R && first == lane);
    if (lane < R) {
      const int at = __popcll(firsts & ((1ull << first) - 1));
      s->slot[lane] = at;
      if (first == lane) s->uniq[at] = mine;
    }
    if (lane == 0) {
      s->n_uniq = __popcll(firsts);
      s->n_ranks = R;
    }
  }
  __syncthreads();
}

// What a selection leaves per metric: the keys of the ranks (left-aligned in 64 bits) and the number of samples.
constexpr int SEL_OUT = KV_MAX_RANKS + 1;

__device__ inline void copy_state(RadixState* to, const RadixState* from) {
  static_assert(sizeof(RadixState) % 4 == 0 && sizeof(RadixState) / 4 <= SEL_THREADS, "a word per thread");
  if (threadIdx.x < sizeof(RadixState) / 4) reinterpret_cast<unsigned int*>(to)[threadIdx.x] = reinterpret_cast<const unsigned int*>(from)[threadIdx.x];
}
__device__ inline void clear_state(RadixState* s) {
  if (threadIdx.x < sizeof(RadixState) / 4) reinterpret_cast<unsigned int*>(s)[threadIdx.x] = 0;
}

// a pass's workgroup: its samples' digits in h, counted
template <typename T>
__device__ void count_pass(const T* row, long long n, int part, int parts, unsigned int* h, const RadixState* s, int U, int shift, int digit_bits, bool first_pass) {
  for (int i = threadIdx.x; i < U * KV_BINS << log2_copies(U, n); i += SEL_THREADS) h[i] = 0;
  __syncthreads();
  const long long first = (long long)part * SEL_THREADS + threadIdx.x, stride = (long long)parts * SEL_THREADS;
  if (first_pass) count_digits<T, 0>(row, n, first, stride, h, s->uniq, U, shift, digit_bits);
  else if (U <= 1) count_digits<T, 1>(row, n, first, stride, h, s->uniq, U, shift, digit_bits);
  else if (U <= 4) count_digits<T, 4>(row, n, first, stride, h, s->uniq, U, shift, digit_bits);
  else count_digits<T, KV_MAX_RANKS>(row, n, first, stride, h, s->uniq, U, shift, digit_bits);
  __syncthreads();
}

// One pass: grid (workgroups, metrics).  PICK: the last workgroup of a metric to finish picks the digits (`done` counts them, and is zero again
// behind it) and clears the histogram for the next pass; with out also what the selection leaves.
template <typename T, bool PICK>
__global__ __launch_bounds__(SEL_THREADS) void select_pass_kernel(const T* __restrict__ x, long long n, long long row_stride, RadixState* st, unsigned int* hist, int shift, int digit_bits, bool first_pass,
                                                                  Levels levels, unsigned int* done, unsigned long long* out) {
  extern __shared__ __attribute__((aligned(16))) unsigned int h[];
  __shared__ RadixState s;
  __shared__ bool last;
  const int tid = threadIdx.x, m = blockIdx.y;
  copy_state(&s, st + m);
  __syncthreads();
  const int U = first_pass ? 1 : s.n_uniq, cl = log2_copies(U, n);
  count_pass<T>(x + (long long)m * row_stride, n, blockIdx.x, gridDim.x, h, &s, U, shift, digit_bits, first_pass);
  unsigned int* gh = hist + (long long)m * KV_MAX_RANKS * KV_BINS;
  for (int i = tid; i < U * KV_BINS; i += SEL_THREADS) {
    const unsigned int c = sum_copies(h, i, cl);
    if (c) atomicAdd(&gh[i], c);
  }
  if constexpr (PICK) {
    // The adds above are asynchronous, and neither the barrier nor a workgroup-scope release waits for them on this target: every wave waits until
    // its own have been performed, then the barrier, and only then is the arrival counted — whoever sees the full count sees all adds.  No fence:
    // what the last workgroup reads was written by device-scope atomics alone (a fence would write an XCD's L2 back, from every wave 80 us a pass).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // also a compiler barrier: no add may sink below it
    __syncthreads();
    if (tid == 0) last = __hip_atomic_fetch_add(&done[m], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    unsigned int c[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j)  // (all on their way at once)
      c[j] = tid + j * SEL_THREADS < U * KV_BINS ? __hip_atomic_load(&gh[tid + j * SEL_THREADS], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = tid + j * SEL_THREADS;
      if (i >= U * KV_BINS) break;
      h[i + (i >> 5)] = c[j];
      gh[i] = 0;
    }
    if (tid == 0) done[m] = 0;
    __syncthreads();
    pick_digits(&s, h, shift + 64 - KeyOf<T>::bits, first_pass, first_pass ? &levels : nullptr);
    copy_state(st + m, &s);
    if (out && tid < SEL_OUT) out[(long long)m * SEL_OUT + tid] = tid < KV_MAX_RANKS ? s.prefix[tid] : s.count;
  }
}

// a sample's key; a NaN's is the largest, which no sample has (that one is a NaN's too)
template <typename T>
__device__ inline typename KeyOf<T>::type key_or_last(T v) {
  using KT = typename KeyOf<T>::type;
  return v == v ? KeyOf<T>::key(v) : ~(KT)0;
}

// How many of keys[from ... from + stretch) (whole 16 bytes) come in front of the key at `at`; of equal ones the one in front is the smaller.  A wave's
// lanes have the same stretch.
template <typename KT>
__device__ inline unsigned int count_in_front(const KT* keys, int from, int stretch, int at, KT key) {
  constexpr int VEC = 16 / sizeof(KT);
  struct alignas(16) Some { KT k[VEC]; };
  unsigned int less = 0;
  auto count = [&](auto&& in_front) {
#pragma unroll 4
    for (int j = from; j < from + stretch; j += VEC) {
      const Some k = *reinterpret_cast<const Some*>(&keys[j]);
#pragma unroll
      for (int i = 0; i < VEC; ++i) less += in_front(k.k[i], j + i);
    }
  };
  // a stretch in front of this key counts those up to it, one behind it those below: one comparison each (NaNs count nowhere)
  const KT upto = from + stretch <= at && key != ~(KT)0 ? key + 1 : key;
  if (__any(from <= at && at < from + stretch)) count([&](KT k, int j) { return k < key || (k == key && j < at); });
  else count([&](KT k, int) { return k < upto; });
  return less;
}

// Up to 512 samples (a run's requests): each is ranked among all, by as many threads as there are per sample.  A workgroup per metric.
constexpr int SEL_RANKED = 512;
template <typename T>
__global__ __launch_bounds__(SEL_THREADS) void select_by_rank_kernel(const T* __restrict__ x, int n, long long row_stride, Levels levels, unsigned long long* out) {
  using KT = typename KeyOf<T>::type;
  __shared__ __attribute__((aligned(16))) KT keys[SEL_RANKED];
  __shared__ unsigned int before[SEL_RANKED];
  const int tid = threadIdx.x, m = blockIdx.x;
  if (tid < SEL_RANKED) {
    keys[tid] = tid < n ? key_or_last(x[(long long)m * row_stride + tid]) : ~(KT)0;
    before[tid] = 0;
  }
  const int count = __syncthreads_count(tid < n && keys[tid < n ? tid : 0] != ~(KT)0);
  int together = 64;
  while (together < n) together *= 2;
  const int stretch = together * together / SEL_THREADS, at = tid % together;
  const KT key = keys[at];
  atomicAdd(&before[at], count_in_front(keys, tid / together * stretch, stretch, at, key));
  __syncthreads();
  unsigned long long* o = out + (long long)m * SEL_OUT;
  if (tid == 0) o[KV_MAX_RANKS] = (unsigned long long)count;
  if (tid < n && key != ~(KT)0)
    for (int r = 0; r < 2 * levels.n; ++r)
      if (rank_of(levels, r, (unsigned long long)count) == (unsigned long long)before[tid]) o[r] = (unsigned long long)key << (64 - KeyOf<T>::bits);
}

// Some thousand samples: all passes in one launch, a workgroup per metric.
template <typename T>
__global__ __launch_bounds__(SEL_THREADS) void select_few_kernel(const T* __restrict__ x, long long n, long long row_stride, Levels levels, unsigned long long* out) {
  extern __shared__ __attribute__((aligned(16))) unsigned int h[];
  __shared__ RadixState s;
  const int tid = threadIdx.x, m = blockIdx.x;
  clear_state(&s);
  __syncthreads();
  for (int top = KeyOf<T>::bits; top > 0;) {
    const bool first = top == KeyOf<T>::bits;
    const int digit_bits = top >= 11 ? 11 : top, U = first ? 1 : s.n_uniq, cl = log2_copies(U, n);
    top -= digit_bits;
    count_pass<T>(x + (long long)m * row_stride, n, 0, 1, h, &s, U, top, digit_bits, first);
    unsigned int c[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = tid + j * SEL_THREADS;
      c[j] = i < U * KV_BINS ? sum_copies(h, i, cl) : 0;
    }
    __syncthreads();  // (the sums lie where the copies were)
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = tid + j * SEL_THREADS;
      if (i < U * KV_BINS) h[i + (i >> 5)] = c[j];
    }
    __syncthreads();
    pick_digits(&s, h, top + 64 - KeyOf<T>::bits, first, first ? &levels : nullptr);
  }
  if (tid < SEL_OUT) out[(long long)m * SEL_OUT + tid] = tid < KV_MAX_RANKS ? s.prefix[tid] : s.count;
}

// ---------------------------------------------------------------------------------
// Many samples, in two passes over them instead of one per digit (3 for floats, 6 for doubles).  What bounds a digit's pass is not memory but one
// LDS atomic per sample.  Here 2048 samples (of long rows 4096), one from each stretch of the row, say between which two values a level's order statistics lie: an
// interval that holds a few per cent of the samples.  The first pass counts the samples below each interval in registers, and only those inside
// go to a histogram, a thousand linear bins of the interval's keys; the second collects the few hundred of the bins that hold the ranks, and the
// last workgroup to finish ranks them.  Exact whatever the samples are: where an interval misses a rank (4 standard deviations aside: about one
// call in 5000) the row's count of samples says so and the digits' passes answer for it.  Where a bin of several values holds more than fit all the same
// (Spans says what is done against that) the count says that the two passes are to be made again, between the least and the most of that bin.
// Whole calls by digits and so, 3 rows: 33 k floats 54 and 48 us, 1 M 69 and 52, 4 M 88 and 64;
// 4 M doubles 198 and 79.  Of the 50 us of kernels for 3 x 4 M floats the sample takes 10, the first pass 21 and the second 19, the last workgroup's ranking
// among them: beside reading (10 us a pass at 5 TB/s) chains of dependent steps, about one us each.  Fewer bins (512, 256) are not faster: their sums are not what counts.
constexpr int SAMPLE_PARTS = 64;                     // workgroups that rank a row's sample, at most
constexpr int SPANS = KV_MAX_RANKS / 2;              // intervals: one per level, fewer where they overlap
constexpr int SPAN_BINS = 1024, SPAN_COPIES = 2;     // LDS: 4 x 1024 x 2 counts, 32 KiB (a lane uses copy lane % 2: values that many samples share)
constexpr int PIECES = 32, PIECE_BINS = SPAN_BINS / PIECES;  // of an interval with a gap
constexpr int FOUND = 16384;                         // samples of a bin that are ranked
constexpr unsigned long long UNDECIDED = ~0ull;      // as a count: the digits' passes have to answer
constexpr unsigned long long CROWDED = ~0ull - 1;    // as a count: the intervals are narrower now, the passes have to be made again
constexpr long long SPLIT_MOST = 1ll << 25;          // of a row: beyond, what a sample says is too wide for FOUND (60 M floats: 182 us, by digits 179)

// What the sample says about a row, and what the passes count.  Keys are the samples' own, in the low bits.
struct SplitState {
  unsigned long long cuts[SPANS][PIECES + 1];        // level -> sampled keys at the ends of its interval and, evenly many apart, between them
  unsigned long long below[SPANS];                   // samples in front of each interval, as Spans orders them
  unsigned long long count;                          // samples
  unsigned long long least[KV_MAX_RANKS], most[KV_MAX_RANKS];  // of the samples in a chosen bin
  unsigned int found[KV_MAX_RANKS];                  // how many those are
  unsigned int done;
  unsigned int open;                                 // ends (two per level) beyond which the interval goes on: no sampled key is as far out as it has to be
  int together[SPANS];                               // level -> a bin with this many pieces between cuts, or more, is too full for FOUND
};
constexpr int SPLIT_WORDS = sizeof(SplitState) / 4;
constexpr long long SPLIT_BYTES = sizeof(SplitState) + SPANS * SPAN_BINS * 4 + (long long)KV_MAX_RANKS * FOUND * 8;
static_assert(sizeof(SplitState) % 16 == 0, "16-byte reads of the bins behind it");

// Sampled ranks between a level and the ends of its interval, of `got`
__host__ __device__ inline double margin(int got, double p) { return 4.0 * sqrt((double)got * p * (1.0 - p)) + 2.0; }

struct SplitRow {
  SplitState* state;
  unsigned int* bins;           // [SPANS][SPAN_BINS]
  unsigned long long* found;    // [KV_MAX_RANKS][FOUND]
  __device__ SplitRow(void* work, int metric) {
    char* p = (char*)work + metric * SPLIT_BYTES;
    state = (SplitState*)p;
    bins = (unsigned int*)(p + sizeof(SplitState));
    found = (unsigned long long*)(bins + SPANS * SPAN_BINS);
  }
};

// What the first pass keeps for the second: each wave the samples inside the intervals, up to `room`, and how many there were.  15 % of a row at the usual three
// levels, so that the second pass reads those and not the row again; a wave that had more goes through its samples again.  Where a workgroup has more than 32 k
// samples (room -1: nothing is kept): calls of 3 x 4 M floats (47 k) 68.5 -> 62.7 us, the second pass 27 -> 19.6, of 30 M (117 k) 111 -> 97.5, of 64 x 1 M 205 -> 158; of
// 1 x 4 M doubles (16 k) and 3 x 1 M floats (12 k) the same, of a thousand samples 1.4 more (and kernels that know both ways half of that).  And where the levels' intervals
// fit what is kept: quartiles of 2048 samples have 24 % inside, and what would be kept in vain is up to 2 % of a call (3 x 4 M floats 69.4, 70.7, doubles 78.9, 81.1, 64 x 1 M
// 210, 214); of 4096 17 % (30 M floats 113 -> 104).  A row of which half is one value is kept in vain all the same (78.4, 79.7; doubles 85.5, 88.2; 64 x 1 M 251, 256): the sample
// could say so, by the values a little outside, and 2 to 4 us of a call of 64 rows would be back, but every other call takes 0.3 to 1 longer for it.
constexpr int WAVES = SEL_THREADS / 64, MOST_PARTS = 256, SPARE = 32;  // of a workgroup; workgroups per row, at most; of a wave, beside 3 / 16 of its samples
template <typename T>
struct Kept {
  unsigned int* counts;  // [parts][WAVES]
  T* samples;            // [parts][WAVES][room]
  int room;
  __device__ Kept(void* kept, long long row_bytes, int metric, int r) {
    char* p = (char*)kept + metric * row_bytes;
    counts = (unsigned int*)p;
    samples = (T*)(p + MOST_PARTS * WAVES * 4);
    room = r;
  }
  __device__ unsigned int& count(int part, int wave) const { return counts[part * WAVES + wave]; }
  __device__ T* of(int part, int wave) const { return samples + ((long long)part * WAVES + wave) * room; }
};
inline int kept_room(long long n, int parts) { return n / parts > 32768 ? (int)(n * 3 / 16 / (parts * WAVES)) + SPARE : -1; }
// samples of a row that are ranked (a larger sample of longer rows: it takes 6 us more, and what lies beyond its largest has to fit FOUND)
inline int sampled(long long n) { return (n <= 1 << 22 ? 2 : 4) * SEL_THREADS; }
// the share of a row that lies inside the levels' intervals
inline double inside(Levels lv, long long n) {
  std::sort(lv.p, lv.p + lv.n);
  double all = 0.0, upto = 0.0;
  for (int i = 0; i < lv.n; ++i) {
    const double p = std::clamp(lv.p[i], 0.0, 1.0), apart = margin(sampled(n), p) / sampled(n), end = std::min(p + apart, 1.0);
    all += std::max(0.0, end - std::max(p - apart, upto));
    upto = std::max(upto, end);
  }
  return all;
}
inline long long kept_bytes(long long n, int dtype) { return MOST_PARTS * WAVES * 4 + (n * 3 / 16 + MOST_PARTS * WAVES * SPARE) / 2 * 2 * (dtype == 0 ? 4 : 8); }

// Linear bins of `wide` + 1 keys: key - first >> bin_shift
template <int BINS>
__device__ inline int bin_shift(unsigned long long wide) {
  static_assert((BINS & (BINS - 1)) == 0, "a power of two");
  return wide < BINS ? 0 : 64 - __clzll((long long)wide) - (31 - __builtin_clz(BINS));
}

// The levels' intervals in order, those that overlap as one, with linear bins.  Where so many cuts fall into one bin that it is too full for FOUND (a gap takes nearly all bins: hits
// and misses of a cache, with a rank between them) and no intervals overlap, each has 32 pieces between its cuts instead, of 32 linear bins: 3 x 4 M floats in two clusters 75 us
// a call, by passes made again 137, by digits 98.  Not for all rows: linear bins need no search for the piece (1 to 2 us), and the piece around a small gap
// holds more than any of them (clusters of 5 % 82 and 69 us).
template <typename KT>
struct Spans {
  unsigned long long lo[SPANS], hi[SPANS];  // ends
  unsigned long long from[SPANS];           // the bins are those of from ... upto: the first takes in what is below, the last what is above
  int shift[SPANS];
  int of[SPANS];                            // level -> interval
  int n;
  bool crowded;                             // a bin is too full: there are pieces, of use if no intervals overlap
  KT search[SPANS * PIECES];                // keys from here on ...
  KT base[SPANS * PIECES];                  // ... in linear bins from here on, the first takes in what is below, the last what is above
  int piece_shift[SPANS * PIECES];
};
// By one thread, in registers: the intervals.
template <typename T>
__device__ inline void find_linear(const SplitState& s, int levels, Spans<typename KeyOf<T>::type>* to) {
  unsigned long long lo[SPANS], hi[SPANS], from[SPANS], upto[SPANS];
  int level[SPANS];
  const unsigned int open = s.open;
#pragma unroll
  for (int i = 0; i < SPANS; ++i) {
    from[i] = i < levels ? s.cuts[i][0] : ~0ull;
    upto[i] = i < levels ? s.cuts[i][PIECES] : ~0ull;
    // (as values: both zeros, which compare as one, are in or out together)
    lo[i] = open >> 2 * i & 1 ? KeyOf<T>::key(-(T)INFINITY) : from[i] == KeyOf<T>::key((T)0) ? KeyOf<T>::key(-(T)0) : from[i];
    hi[i] = open >> (2 * i + 1) & 1 ? KeyOf<T>::key((T)INFINITY) : upto[i] == KeyOf<T>::key(-(T)0) ? KeyOf<T>::key((T)0) : upto[i];
    if (i >= levels) lo[i] = ~0ull;  // (no key: behind all others)
    level[i] = i;
  }
#pragma unroll
  for (int i = 1; i < SPANS; ++i)
#pragma unroll
    for (int j = i; j > 0; --j)
      if (lo[j - 1] > lo[j]) {
        const unsigned long long a = lo[j], b = hi[j], c = from[j], d = upto[j];
        const int l = level[j];
        lo[j] = lo[j - 1]; hi[j] = hi[j - 1]; from[j] = from[j - 1]; upto[j] = upto[j - 1]; level[j] = level[j - 1];
        lo[j - 1] = a; hi[j - 1] = b; from[j - 1] = c; upto[j - 1] = d; level[j - 1] = l;
      }
  int n = 0;
  unsigned long long first = 0, last = 0, in = 0, out = 0;
#pragma unroll
  for (int i = 0; i < SPANS; ++i) {
    if (i >= levels) break;
    const bool apart = n == 0 || lo[i] > last;
    n += apart;
    first = apart ? lo[i] : first;
    last = apart || hi[i] > last ? hi[i] : last;
    in = apart || from[i] < in ? from[i] : in;
    out = apart || upto[i] > out ? upto[i] : out;
    to->lo[n - 1] = first;
    to->hi[n - 1] = last;
    to->from[n - 1] = in;
    to->shift[n - 1] = bin_shift<SPAN_BINS>(out - in);
    to->of[level[i]] = n - 1;
    to->search[(n - 1) * PIECES] = (typename KeyOf<T>::type)first;
  }
  for (int i = n; i < SPANS; ++i) to->search[i * PIECES] = ~(typename KeyOf<T>::type)0;
  to->n = n;
}
// By a wave, meanwhile: the pieces, two a lane.
template <typename T>
__device__ inline void find_pieces(const SplitState& s, int levels, Spans<typename KeyOf<T>::type>* to) {
  using KT = typename KeyOf<T>::type;
  static_assert(SPANS * PIECES == 2 * 64, "of all levels");
  constexpr int LANES = PIECES / 2;  // of a level
  const int lane = threadIdx.x & 63, l = lane / LANES, j = lane % LANES * 2, q = s.together[l];
  const unsigned long long before = s.cuts[l][j > 0 ? j - 1 : 0], cut[3] = {s.cuts[l][j], s.cuts[l][j + 1], s.cuts[l][j + 2]};
  const unsigned long long from = __shfl(cut[0], l * LANES, 64), upto = __shfl(cut[2], l * LANES + LANES - 1, 64);
  const int shift = bin_shift<SPAN_BINS>(upto - from), bin[2] = {(int)((cut[0] - from) >> shift), (int)((cut[1] - from) >> shift)};
  bool full = false;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int k = j + e + q, at = (l * LANES + k / 2) & 63, even = __shfl(bin[0], at, 64), odd = __shfl(bin[1], at, 64);
    full = full || (k < PIECES && (k & 1 ? odd : even) == bin[e]);
  }
  int place = 0;  // of the level's interval among all
#pragma unroll
  for (int i = 0; i < SPANS; ++i) place += i < levels && __shfl(from, i * LANES, 64) < from;
  const bool crowded = __ballot(full && l < levels && shift > 0) != 0;
  if (lane == 0) to->crowded = crowded;
  if (!crowded) return;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    // (a key that is several cuts, a timeout, say, has a piece of its own: the last of them begins behind it)
    const bool again = e == 0 ? j > 0 && cut[0] == before : cut[1] == cut[0];
    const unsigned long long base = cut[e] + (again && cut[e + 1] != cut[e] ? 1 : 0);
    const int p = (l < levels ? place : l) * PIECES + j + e;
    to->base[p] = l < levels ? (KT)base : ~(KT)0;
    if (j + e > 0) to->search[p] = l < levels ? (KT)base : ~(KT)0;
    to->piece_shift[p] = cut[e + 1] > base ? bin_shift<PIECE_BINS>(cut[e + 1] - base) : 0;
  }
}
template <typename T>
__device__ inline void find_spans(const SplitState& s, int levels, Spans<typename KeyOf<T>::type>* to) {
  if (threadIdx.x == 0) find_linear<T>(s, levels, to);
  if (threadIdx.x / 64 == 1) find_pieces<T>(s, levels, to);
  __syncthreads();
}
template <typename KT>
__device__ inline bool pieced(const Spans<KT>& s, int levels) { return s.crowded && s.n == levels; }

// The levels' intervals, from EACH samples per thread.  Grid (workgroups, metrics): each takes in all sampled keys, ranks its share of them against all, and writes those whose
// rank is that of an end.  (One workgroup that selects by digits took 45 us: a chain of loads, LDS sums and scans on one compute unit.)
template <typename T, int EACH>
__global__ __launch_bounds__(SEL_THREADS) void select_sample_kernel(const T* __restrict__ x, long long n, long long row_stride, Levels levels, void* work) {
  using KT = typename KeyOf<T>::type;
  constexpr int SAMPLED = EACH * SEL_THREADS;
  __shared__ __attribute__((aligned(16))) KT keys[SAMPLED];
  __shared__ unsigned int before[SEL_THREADS];
  __shared__ unsigned int rank[KV_MAX_RANKS];  // of the levels' ends
  const int tid = threadIdx.x, m = blockIdx.y;
  const SplitRow row(work, m);
  const T* xr = x + (long long)m * row_stride;
  T v[EACH];
#pragma unroll
  for (int j = 0; j < EACH; ++j) {
    // somewhere in the stretch: samples at even distances would all be, say, a request's first (mixed as 32-bit xxHash ends, by Yann Collet)
    const unsigned long long at = tid + j * SEL_THREADS, from = at * (unsigned long long)n / SAMPLED, len = (at + 1) * (unsigned long long)n / SAMPLED - from;
    unsigned int r = (unsigned int)at * 2654435761u + (unsigned int)m * 40503u;
    r ^= r >> 15; r *= 2246822519u; r ^= r >> 13; r *= 3266489917u; r ^= r >> 16;
    v[j] = xr[from + (((unsigned long long)r * len) >> 32)];
  }
  int got = 0;
#pragma unroll
  for (int j = 0; j < EACH; ++j) {
    keys[tid + j * SEL_THREADS] = key_or_last(v[j]);
    got += __syncthreads_count(v[j] == v[j]);
  }
  if (tid < KV_MAX_RANKS) {
    double p = levels.p[tid >> 1];
    p = p < 0.0 ? 0.0 : (p > 1.0 ? 1.0 : p);
    const double at = p * (double)(got - 1), apart = margin(got, p);
    const double end = (tid & 1) ? ceil(at + apart) : floor(at - apart);
    const bool open = end < 0.0 || end > (double)(got - 1);
    rank[tid] = end < 0.0 ? 0 : end > (double)(got - 1) ? (unsigned int)(got - 1) : (unsigned int)end;
    const unsigned int opens = (unsigned int)__ballot(open);
    if (blockIdx.x == 0) {
      // samples of a piece: those of the row over those of the sample, times the ranks between two cuts
      const float ranks = (float)(rank[tid | 1] - rank[tid & ~1] + 1), each = (float)n * ranks * __builtin_amdgcn_rcpf((float)got * PIECES);
      if (tid & 1) row.state->together[tid >> 1] = 1 + (int)fminf(0.75f * FOUND * __builtin_amdgcn_rcpf(each), (float)PIECES);
      row.state->least[tid] = ~0ull;
      row.state->most[tid] = 0;
      row.state->found[tid] = 0;
      if (tid < SPANS) row.state->below[tid] = 0;
      if (tid == 0) { row.state->count = 0; row.state->done = 0; row.state->open = opens; }
    }
  }
  if (got == 0 && blockIdx.x == 0 && tid < SPANS * (PIECES + 1)) row.state->cuts[tid / (PIECES + 1)][tid % (PIECES + 1)] = KeyOf<T>::key(tid % (PIECES + 1) == PIECES ? (T)INFINITY : -(T)INFINITY);
  for (int i = blockIdx.x * SEL_THREADS + tid; i < SPANS * SPAN_BINS; i += gridDim.x * SEL_THREADS) row.bins[i] = 0;
  // as many threads per key as there are, each for a stretch of the others
  const int ours = SAMPLED / (int)gridDim.x, together = ours < SEL_THREADS ? ours : SEL_THREADS, stretch = SAMPLED / (SEL_THREADS / together);
  const int mine = tid % together, from = tid / together * stretch;
  for (int base = 0; base < ours; base += together) {
    const int at = (int)blockIdx.x * ours + base + mine;
    before[tid] = 0;
    __syncthreads();
    const KT key = keys[at];
    atomicAdd(&before[mine], count_in_front(keys, from, stretch, at, key));
    __syncthreads();
    if (tid < together && key != ~(KT)0)
      for (int l = 0; l < levels.n; ++l) {
        const unsigned int at = before[tid] - rank[2 * l], wide = rank[2 * l + 1] - rank[2 * l];
        if (at > wide) continue;
        // the cuts j with wide j / PIECES = at, whole numbers: few, from one that the quotient names (it is rounded) or a neighbour on
        const int j = (int)((float)(at * PIECES) * __builtin_amdgcn_rcpf((float)wide));
        for (unsigned int k = wide && j > 0 ? j - 1 : 0; k <= PIECES && wide * k / PIECES <= at; ++k)
          if (wide * k / PIECES == at) row.state->cuts[l][k] = key;
      }
    __syncthreads();
  }
}

constexpr int QUEUE_BYTES = 2048;  // of a wave: room for fewer than 64 samples that wait and 16 bytes of each lane

template <typename K> __device__ inline auto value_of(K key) {
  if constexpr (sizeof(K) == 4) return __uint_as_float(key & 0x80000000u ? key & 0x7fffffffu : ~key);
  else return __longlong_as_double((long long)(key & 0x8000000000000000ull ? key & 0x7fffffffffffffffull : ~key));
}

// The same in all lanes: kept in scalar registers, not read from LDS again for each sample that needs one of several.
__device__ inline uint32_t in_sgpr(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ inline uint64_t in_sgpr(uint64_t v) { return (uint64_t)in_sgpr((uint32_t)(v >> 32)) << 32 | in_sgpr((uint32_t)v); }

// The first pass of a workgroup: V intervals.
//
// What bounds it is instructions per sample, not memory: the samples are compared as they are (two instructions per interval, the masks they leave
// counted by the scalar unit), and those inside queue up per wave, so that the two dozen instructions that bin one run on full waves and not on the five lanes
// of 64 that have one.  (With each instruction's few lanes on their own the pass over 3 x 4 M floats took 2 us more of its 20.)
template <typename T, int V, bool PIECED, bool KEEP>
__device__ void split_pass(const T* row, long long n, int part, int parts, const Spans<typename KeyOf<T>::type>& s, T* queue, unsigned int* h, unsigned int* below, unsigned int* valid, const Kept<T>& kept) {
  using KT = typename KeyOf<T>::type;
  constexpr int QUEUE = QUEUE_BYTES / sizeof(T);
  T lo[V], hi[V];
  KT from[V];
  int shift[V];
  unsigned int under[V] = {}, on = 0;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    lo[i] = value_of(in_sgpr((KT)s.lo[i]));
    hi[i] = value_of(in_sgpr((KT)s.hi[i]));
    from[i] = in_sgpr((KT)s.from[i]);
    shift[i] = (int)in_sgpr((uint32_t)s.shift[i]);
  }
  const int copy = threadIdx.x & (SPAN_COPIES - 1), lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  T* const mine = kept.of(part, wave);
  const int room = kept.room;
  unsigned int queued = 0, binned = 0;  // of this wave; the queue is a ring
  auto bin_one = [&](T v) {
    const KT key = KeyOf<T>::key(v);
    if constexpr (PIECED) {
      int at = 0;
#pragma unroll
      for (int step = SPANS * PIECES / 2; step > 0; step /= 2) at += s.search[at + step] <= key ? step : 0;
      const KT begin = s.base[at], in_piece = (key > begin ? key - begin : 0) >> s.piece_shift[at];
      atomicAdd(&h[(at * PIECE_BINS + (int)(in_piece < PIECE_BINS ? in_piece : PIECE_BINS - 1)) * SPAN_COPIES + copy], 1u);
      return;
    }
    KT first = from[0];
    int sh = shift[0], base = 0;
    asm("" : "+s"(first), "+s"(sh));
#pragma unroll
    for (int i = 1; i < V; ++i) {
      KT f = from[i];
      int t = shift[i];
      asm("" : "+s"(f), "+s"(t));  // values: the compiler would choose between their addresses and read memory
      const bool up = v >= lo[i];  // (the intervals ascend)
      first = up ? f : first;
      sh = up ? t : sh;
      base = up ? i * SPAN_BINS : base;
    }
    const KT bin = (key > first ? key - first : 0) >> sh;
    atomicAdd(&h[(base + (int)(bin < SPAN_BINS ? bin : SPAN_BINS - 1)) * SPAN_COPIES + copy], 1u);
  };
  for_samples(row, n, (long long)part * SEL_THREADS + threadIdx.x, (long long)parts * SEL_THREADS, [&](T v) {
    on += __popcll(__ballot(v == v));
    asm("" : "+s"(on));  // now: put off, the masks of a dozen samples take more scalar registers than there are
    unsigned long long who = 0;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const unsigned long long low = __ballot(v < lo[i]);
      under[i] += __popcll(low);
      asm("" : "+s"(under[i]));
      who |= __ballot(v <= hi[i]) & ~low;
    }
    if (__builtin_amdgcn_inverse_ballot_w64(who)) queue[(queued + __builtin_amdgcn_mbcnt_hi((unsigned int)(who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)who, 0u))) & (QUEUE - 1)] = v;
    queued += __popcll(who);
  }, [&] {
    for (; queued - binned >= 64; binned += 64) {
      const T v = queue[(binned + lane) & (QUEUE - 1)];
      if (KEEP && (int)binned + 64 <= room) mine[binned + lane] = v;
      bin_one(v);
    }
  });
  if (lane < (int)(queued - binned)) {
    const T v = queue[(binned + lane) & (QUEUE - 1)];
    if (KEEP && (int)binned + lane < room) mine[binned + lane] = v;
    bin_one(v);
  }
  if (lane == 0) {
    if (KEEP) kept.count(part, wave) = queued;
#pragma unroll
    for (int i = 0; i < V; ++i) atomicAdd(&below[i], under[i]);
    atomicAdd(valid, on);
  }
}

constexpr int SPLIT_LDS = SPANS * SPAN_BINS * SPAN_COPIES * 4 + SEL_THREADS / 64 * QUEUE_BYTES;

// Grid (workgroups, metrics).
template <typename T, bool KEEP>
__global__ __launch_bounds__(SEL_THREADS) void select_split_kernel(const T* __restrict__ x, long long n, long long row_stride, int levels, void* work, void* kept_, long long kept_row, int room) {
  extern __shared__ __attribute__((aligned(16))) unsigned int h[];  // [SPANS][SPAN_BINS][SPAN_COPIES], then the waves' queues
  __shared__ Spans<typename KeyOf<T>::type> s;
  __shared__ unsigned int below[SPANS + 1];
  const int tid = threadIdx.x, m = blockIdx.y;
  const SplitRow row(work, m);
  for (int i = tid; i < SPANS * SPAN_BINS * SPAN_COPIES; i += SEL_THREADS) h[i] = 0;
  if (tid <= SPANS) below[tid] = 0;
  const Kept<T> kept(kept_, kept_row, m, room);
  T* queue = reinterpret_cast<T*>(reinterpret_cast<char*>(h + SPANS * SPAN_BINS * SPAN_COPIES) + (tid >> 6) * QUEUE_BYTES);
  find_spans<T>(*row.state, levels, &s);
  const T* xr = x + (long long)m * row_stride;
  const int V = s.n;
  auto pass = [&](auto v) {
    if (pieced(s, levels)) split_pass<T, decltype(v)::value, true, KEEP>(xr, n, blockIdx.x, gridDim.x, s, queue, h, below, below + SPANS, kept);
    else split_pass<T, decltype(v)::value, false, KEEP>(xr, n, blockIdx.x, gridDim.x, s, queue, h, below, below + SPANS, kept);
  };
  if (V <= 1) pass(std::integral_constant<int, 1>{});
  else if (V == 2) pass(std::integral_constant<int, 2>{});
  else if (V == 3) pass(std::integral_constant<int, 3>{});
  else pass(std::integral_constant<int, SPANS>{});
  __syncthreads();
  for (int i = tid; i < V * SPAN_BINS; i += SEL_THREADS) {
    const unsigned int c = sum_copies(h, i, 1);
    if (c) atomicAdd(&row.bins[i], c);
  }
  if (tid < V) atomicAdd(&row.state->below[tid], (unsigned long long)below[tid]);
  if (tid == SPANS) atomicAdd(&row.state->count, (unsigned long long)below[SPANS]);
}

// A wave: the bin that holds the k-th sample, and its place in there; -1: there are not as many.
template <int BINS>
__device__ inline int pick_bin(const unsigned int* bins, unsigned long long k, unsigned long long* place) {
  constexpr int EACH = BINS / 64;
  const int lane = threadIdx.x & 63;
  const uint4* p = reinterpret_cast<const uint4*>(bins) + lane * (EACH / 4);
  unsigned int t[EACH];
#pragma unroll
  for (int j = 0; j < EACH / 4; ++j) { const uint4 v = p[j]; t[4 * j] = v.x; t[4 * j + 1] = v.y; t[4 * j + 2] = v.z; t[4 * j + 3] = v.w; }
  unsigned long long local = 0;
#pragma unroll
  for (int j = 0; j < EACH; ++j) local += t[j];
  unsigned long long upto = local;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long v = __shfl_up(upto, o, 64);
    if (lane >= o) upto += v;
  }
  unsigned long long run = upto - local;
  const unsigned long long here = __ballot(k >= run && k < upto);
  if (here == 0) return -1;
  int bin = 0;
  unsigned long long below = 0;
#pragma unroll
  for (int j = 0; j < EACH; ++j) {
    if (k >= run && k < run + t[j]) { bin = lane * EACH + j; below = run; }
    run += t[j];
  }
  const int at = __ffsll((long long)here) - 1;
  *place = k - __shfl(below, at, 64);
  return __shfl(bin, at, 64);
}

// The bins that hold ranks, as every workgroup of the second pass finds them again.
struct Chosen {
  unsigned long long lo[KV_MAX_RANKS], wide[KV_MAX_RANKS];  // keys of a bin
  unsigned long long place[KV_MAX_RANKS];                   // of a rank in its bin
  int id[KV_MAX_RANKS];                                     // of a rank's bin, -1: its interval misses it
  int bin_of[KV_MAX_RANKS];                                 // rank -> bin
};

// The last workgroup: ranks what was found in the U chosen bins.  Each rank has its own, narrower bins of them, again and again until what is left
// is one value or fits a wave's lanes: at once for most samples, at most log(keys) / log(RANK_BINS) times.
// (Inlined: as a call the compiler's choice, it cost the passes 4 us.)
constexpr int RANK_BINS = 1024;
template <typename T>
__device__ __forceinline__ void rank_found(const SplitRow& row, const Chosen& c, int R, int U, unsigned int* h, unsigned long long count, unsigned long long* out) {
  __shared__ unsigned long long few[KV_MAX_RANKS][64], from[KV_MAX_RANKS], upto[KV_MAX_RANKS], least[KV_MAX_RANKS], most[KV_MAX_RANKS];  // of a rank
  __shared__ unsigned long long answer[KV_MAX_RANKS];
  __shared__ int bin_of[KV_MAX_RANKS], picked[KV_MAX_RANKS], held[KV_MAX_RANKS], cnt[KV_MAX_RANKS];
  __shared__ bool undecided, crowded[KV_MAX_RANKS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, rest = 64 - KeyOf<T>::bits;
  if (tid == 0) undecided = false;
  if (tid < KV_MAX_RANKS) {
    crowded[tid] = false;
    const unsigned int f = tid < U ? __hip_atomic_load(&row.state->found[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    cnt[tid] = f <= FOUND ? (int)f : 0;
  }
  __syncthreads();
  if (tid < KV_MAX_RANKS) {
    int u = tid < R ? c.bin_of[tid] : -1;
    if (tid < R && u < 0) undecided = true;
    if (u >= 0) {
      const unsigned int in_bin = row.bins[c.id[tid]];
      from[tid] = __hip_atomic_load(&row.state->least[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      upto[tid] = __hip_atomic_load(&row.state->most[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool first = c.place[tid] == 0;
      if (first || c.place[tid] + 1 == in_bin || from[tid] == upto[tid]) {  // the least, the most, one value
        answer[tid] = first ? from[tid] : upto[tid];
        u = -1;
      } else if (cnt[u] == 0) {
        crowded[tid] = true;
        u = -1;
      }
    }
    bin_of[tid] = u;  // -1: nothing left to do
  }
  __syncthreads();
  constexpr int HELD = 4;  // samples per thread that stay in registers
  int total = 0;
  for (int u = 0; u < U; ++u) total += cnt[u];
  unsigned long long key[HELD];
  int bin[HELD];
  auto read = [&](int first) {
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
      int i = first + j * SEL_THREADS + tid;
      bin[j] = -1;
      key[j] = 0;
      for (int u = 0; u < U && i >= 0; i -= cnt[u++])
        if (i < cnt[u]) { bin[j] = u; key[j] = __hip_atomic_load(&row.found[(long long)u * FOUND + i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    }
  };
  auto each = [&](auto visit) {  // visit(rank, key, its bin) for what may be the rank's
    int of[KV_MAX_RANKS], shift[KV_MAX_RANKS];
    unsigned long long lo[KV_MAX_RANKS], wide[KV_MAX_RANKS];
#pragma unroll
    for (int r = 0; r < KV_MAX_RANKS; ++r) {  // (all on their way at once)
      of[r] = r < R ? bin_of[r] : -1;
      lo[r] = from[r];
      wide[r] = upto[r] - lo[r];
    }
#pragma unroll
    for (int r = 0; r < KV_MAX_RANKS; ++r) shift[r] = bin_shift<RANK_BINS>(wide[r]);
    for (int first = 0; first < total; first += HELD * SEL_THREADS) {
      if (total > HELD * SEL_THREADS) read(first);
#pragma unroll
      for (int j = 0; j < HELD; ++j) {
        if (bin[j] < 0) continue;
#pragma unroll
        for (int r = 0; r < KV_MAX_RANKS; ++r)
          if (of[r] == bin[j] && key[j] - lo[r] <= wide[r]) visit(r, key[j], (int)((key[j] - lo[r]) >> shift[r]));
      }
    }
  };
  if (total <= HELD * SEL_THREADS) read(0);
  unsigned long long place = wave < R ? c.place[wave] : 0;
  bool more = true;
  while (more) {
    for (int i = tid; i < R * RANK_BINS; i += SEL_THREADS) h[i] = 0;
    if (tid < KV_MAX_RANKS) { least[tid] = ~0ull; most[tid] = 0; held[tid] = 0; }
    __syncthreads();
    each([&](int r, unsigned long long, int bin) { atomicAdd(&h[r * RANK_BINS + bin], 1u); });
    __syncthreads();
    if (wave < R && bin_of[wave] >= 0) {
      const int bin = pick_bin<RANK_BINS>(h + wave * RANK_BINS, place, &place);
      if (lane == 0) picked[wave] = bin;
    }
    __syncthreads();
    each([&](int r, unsigned long long key, int bin) {
      if (bin != picked[r]) return;
      const int i = atomicAdd(&held[r], 1);
      if (i < 64) few[r][i] = key;
      atomicMin(&least[r], key);
      atomicMax(&most[r], key);
    });
    __syncthreads();
    bool left = false;
    if (wave < R && bin_of[wave] >= 0) {
      const int have = held[wave];
      left = have > 64 && least[wave] != most[wave];
      if (least[wave] == most[wave]) {
        if (lane == 0) answer[wave] = least[wave];
      } else if (!left) {
        const unsigned long long key = lane < have ? few[wave][lane] : ~0ull;
        unsigned int before = 0;
        for (int j = 0; j < have; ++j) before += few[wave][j] < key || (few[wave][j] == key && j < lane);
        if (lane < have && before == place) answer[wave] = key;
      }
      if (lane == 0) {
        from[wave] = least[wave];
        upto[wave] = most[wave];
        if (!left) bin_of[wave] = -1;
      }
    }
    more = __syncthreads_or(left);
  }
  if (wave > 0) return;  // (behind the loop's last barrier)
  const bool again = __ballot(lane < R && crowded[lane < R ? lane : 0]) != 0;
  if (lane < R) out[lane] = answer[lane] << rest;
  if (lane == 0) out[KV_MAX_RANKS] = undecided ? UNDECIDED : again ? CROWDED : count;
  if (again && lane < R / 2) {
    // a level's ranks follow one another: beside one in a crowded bin the other is in there too, or it would be the bin's first or last and not be crowded
    const int l = 2 * lane, r = crowded[l] ? l : l + 1;
    row.state->cuts[lane][0] = crowded[r] ? from[r] : answer[l];
    row.state->cuts[lane][PIECES] = crowded[r] ? upto[r] : answer[l + 1];
    row.state->together[lane] = PIECES;  // (linear bins)
    if (lane == 0) row.state->open = 0;
  }
}

// The second pass.  Grid (workgroups, metrics).
template <typename T, bool KEEP>
__global__ __launch_bounds__(SEL_THREADS) void select_collect_kernel(const T* __restrict__ x, long long n, long long row_stride, Levels levels, void* work, unsigned long long* out, void* kept_, long long kept_row, int room) {
  using KT = typename KeyOf<T>::type;
  constexpr int ROOM = 6144;
  static_assert(ROOM * 2 >= KV_MAX_RANKS * RANK_BINS, "rank_found's bins");
  __shared__ __attribute__((aligned(16))) unsigned long long keys[ROOM];  // what this workgroup finds, [bin][ours]
  __shared__ Spans<typename KeyOf<T>::type> s;
  __shared__ Chosen c;
  __shared__ unsigned int found[KV_MAX_RANKS], from[KV_MAX_RANKS];
  __shared__ unsigned long long least[KV_MAX_RANKS], most[KV_MAX_RANKS];
  __shared__ bool last;
  const int tid = threadIdx.x, m = blockIdx.y, wave = tid >> 6, lane = tid & 63;
  const SplitRow row(work, m);
  const unsigned long long count = row.state->count;
  const int R = count ? 2 * levels.n : 0;
  if (tid < KV_MAX_RANKS) { found[tid] = 0; least[tid] = ~0ull; most[tid] = 0; c.id[tid] = -1; }
  find_spans<T>(*row.state, levels.n, &s);
  if (wave < R) {  // a wave per rank
    const int span = s.of[wave >> 1];
    const unsigned long long rank = rank_of(levels, wave, count), below = row.state->below[span];
    unsigned long long place = 0;
    const int bin = rank >= below ? pick_bin<SPAN_BINS>(row.bins + span * SPAN_BINS, rank - below, &place) : -1;
    if (lane == 0 && bin >= 0) { c.id[wave] = span * SPAN_BINS + bin; c.place[wave] = place; }
  }
  __syncthreads();
  int first = lane;  // a lane per rank: the first rank with the same bin, and how many such firsts there are in front of it
  const int id = c.id[lane < KV_MAX_RANKS ? lane : 0];
#pragma unroll
  for (int r = KV_MAX_RANKS - 1; r >= 0; --r) first = __shfl(id, r, 64) == id ? r : first;
  const unsigned long long firsts = __ballot(lane < R && id >= 0 && first == lane);
  const int U = __popcll(firsts);
  if (tid < KV_MAX_RANKS) {
    const int u = tid < R && id >= 0 ? __popcll(firsts & ((1ull << first) - 1)) : -1;
    c.bin_of[tid] = u;
    if (u >= 0 && first == tid) {
      const int span = id / SPAN_BINS;
      const bool in_pieces = pieced(s, levels.n);
      const int p = id / PIECE_BINS, bins = in_pieces ? PIECE_BINS : SPAN_BINS, bin = id % bins, shift = in_pieces ? s.piece_shift[p] : s.shift[span];
      const unsigned long long from = in_pieces ? s.base[p] : s.from[span], begin = from + ((unsigned long long)bin << shift);
      const unsigned long long first = bin > 0 ? begin : in_pieces ? s.search[p] : s.lo[span], end = in_pieces && (p + 1) % PIECES ? s.search[p + 1] - 1 : s.hi[span];
      // by what is left up to the end of the interval or piece: the bin's own end, as a key, can lie past the last one and come round to zero
      const unsigned long long whole = (1ull << shift) - 1;
      c.lo[u] = first;
      c.wide[u] = bin == bins - 1 || end < begin || end - begin <= whole ? end - first : begin - first + whole;
    }
  }
  __syncthreads();
  const Kept<T> kept(kept_, kept_row, m, room);
  const int our_wave = __builtin_amdgcn_readfirstlane(wave);
  const unsigned int have = KEEP ? in_sgpr((uint32_t)kept.count(blockIdx.x, our_wave)) : 0;
  const T* const mine = kept.of(blockIdx.x, our_wave);
  const unsigned int ours = U ? (ROOM / U < FOUND ? ROOM / U : FOUND) : 0;
  auto pass = [&](auto most_bins) {
    constexpr int MOST = decltype(most_bins)::value;
    KT lo[MOST], wide[MOST];
#pragma unroll
    for (int u = 0; u < MOST; ++u) { lo[u] = in_sgpr((KT)c.lo[u < U ? u : 0]); wide[u] = in_sgpr((KT)c.wide[u < U ? u : 0]); }  // (unused ones repeat the first)
    auto visit = [&](T v) __attribute__((always_inline)) {
      const KT key = key_or_last(v);
      int at = -1;
#pragma unroll
      for (int u = MOST - 1; u >= 0; --u) at = (KT)(key - lo[u]) <= wide[u] ? u : at;
      if (at < 0) return;
      if (found[at] <= ours) {
        const unsigned int i = atomicAdd(&found[at], 1u);
        if (i < ours) keys[at * ours + i] = key;
      }
      if ((unsigned long long)key < least[at]) atomicMin(&least[at], (unsigned long long)key);
      if ((unsigned long long)key > most[at]) atomicMax(&most[at], (unsigned long long)key);
    };
    if (!KEEP || have > (unsigned int)room) {
      for_samples(x + (long long)m * row_stride, n, (long long)blockIdx.x * SEL_THREADS + tid, (long long)gridDim.x * SEL_THREADS, visit);
      return;
    }
    constexpr int AT_ONCE = 8;
    for (unsigned int i = lane; i < have + lane; i += AT_ONCE * 64) {  // (the same for all lanes)
      T v[AT_ONCE];
#pragma unroll
      for (int j = 0; j < AT_ONCE; ++j) v[j] = i + j * 64 < have ? mine[i + j * 64] : (T)__builtin_nanf("");
#pragma unroll
      for (int j = 0; j < AT_ONCE; ++j) visit(v[j]);
    }
  };
  if (U == 1) pass(std::integral_constant<int, 1>{});
  else if (U > 1 && U <= 3) pass(std::integral_constant<int, 3>{});
  else if (U > 3) pass(std::integral_constant<int, KV_MAX_RANKS>{});
  __syncthreads();
  if (tid < U && found[tid]) {
    from[tid] = atomicAdd(&row.state->found[tid], found[tid] <= ours ? found[tid] : FOUND + 1u);  // (too many here: too many in all)
    atomicMin(&row.state->least[tid], least[tid]);
    atomicMax(&row.state->most[tid], most[tid]);
  }
  __syncthreads();
  for (int u = 0; u < U; ++u) {
    if (found[u] > ours) continue;
    for (unsigned int j = tid; j < found[u] && from[u] + j < FOUND; j += SEL_THREADS)
      __hip_atomic_store(&row.found[u * FOUND + from[u] + j], keys[u * ours + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (as in select_pass_kernel: every wave's own have been performed before its workgroup is counted)
  __syncthreads();
  if (tid == 0) last = __hip_atomic_fetch_add(&row.state->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  __syncthreads();
  if (last) rank_found<T>(row, c, R, U, reinterpret_cast<unsigned int*>(keys), count, out + (long long)m * SEL_OUT);
}

// Before the passes are made again between the ends that the last ones left.  Grid (workgroups, metrics).
__global__ __launch_bounds__(SEL_THREADS) void select_again_kernel(void* work) {
  const SplitRow row(work, blockIdx.y);
  const int i = blockIdx.x * SEL_THREADS + threadIdx.x;
  if (i < SPANS * SPAN_BINS) row.bins[i] = 0;
  if (i < SPANS) row.state->below[i] = 0;
  if (i < KV_MAX_RANKS) {
    row.state->least[i] = ~0ull;
    row.state->most[i] = 0;
    row.state->found[i] = 0;
  }
  if (i == 0) { row.state->count = 0; row.state->done = 0; }
}

// clears a selection's state, histograms and counters (a kernel, not a memset: callers may capture it)
__global__ __launch_bounds__(SEL_THREADS) void select_clear_kernel(unsigned int* words, int n) {
  const int i = blockIdx.x * SEL_THREADS + threadIdx.x;
  if (i < n) words[i] = 0;
}

// Samples spread over ranks: the digits of the summed histograms.  Grid: metrics.
__global__ __launch_bounds__(SEL_THREADS) void select_scan_kernel(RadixState* st, unsigned int* hist, int shift, bool first_pass) {
  extern __shared__ __attribute__((aligned(16))) unsigned int h[];
  __shared__ RadixState s;
  const int tid = threadIdx.x, m = blockIdx.x;
  copy_state(&s, st + m);
  unsigned int* gh = hist + (long long)m * KV_MAX_RANKS * KV_BINS;
  for (int i = tid; i < KV_MAX_RANKS * KV_BINS; i += SEL_THREADS) {
    h[i + (i >> 5)] = gh[i];
    gh[i] = 0;
  }
  __syncthreads();
  pick_digits(&s, h, shift, first_pass, nullptr);
  copy_state(st + m, &s);
}

// ... and the ranks of the samples they have together (device array of levels, the count as the streaming state holds it)
__global__ void radix_init_kernel(const StreamState* __restrict__ stream, RadixState* __restrict__ st, const double* __restrict__ ps, int n_ps) {
  const int m = blockIdx.x;
  if (threadIdx.x != 0) return;
  RadixState* s = st + m;
  Levels lv{};
  lv.n = n_ps;
  for (int i = 0; i < n_ps && i < KV_MAX_RANKS / 2; ++i) lv.p[i] = ps[i];
  s->count = stream[m].count;
  const int r = s->count ? 2 * lv.n : 0;
  for (int i = 0; i < KV_MAX_RANKS; ++i) {
    s->prefix[i] = 0; s->uniq[i] = 0; s->slot[i] = 0;
    s->k[i] = i < r ? rank_of(lv, i, s->count) : 0;
  }
  s->n_uniq = r ? 1 : 0;
  s->n_ranks = r;
}

// ---------------------------------------------------------------------------------
// 20-bin (n_bins <= 64) equal-width histogram over [min, max] taken from StreamState.
template <typename T>
__global__ __launch_bounds__(KV_THREADS) void equal_hist_kernel(const T* __restrict__ x, long long n, long long row_stride,
                                                                const StreamState* __restrict__ state, unsigned long long* __restrict__ out, int n_bins) {
  __shared__ unsigned int lds[KV_WAVES * 64];
  const int tid = threadIdx.x, wave = tid >> 6;
  const int m = blockIdx.y;
  for (int i = tid; i < KV_WAVES * 64; i += KV_THREADS) lds[i] = 0;
  __syncthreads();
  const StreamState* s = state + m;
  // decode min/max keys back to values
  auto unkey = [](unsigned long long k) -> double {
    if (sizeof(T) == 4) {
      uint32_t b = (uint32_t)(k >> 32);
      b = (b & 0x80000000u) ? (b & 0x7fffffffu) : ~b;
      return (double)__uint_as_float(b);
    }
    unsigned long long b = (k & 0x8000000000000000ull) ? (k & 0x7fffffffffffffffull) : ~k;
    return __longlong_as_double((long long)b);
  };
  const double lo = unkey(s->min_key), hi = unkey(s->max_key);
  const double width = (hi - lo) / (double)n_bins;
  const T* row = x + (long long)m * row_stride;
  const long long stride = (long long)gridDim.x * KV_THREADS;
  if (s->count && hi > lo) {
    for (long long i = (long long)blockIdx.x * KV_THREADS + tid; i < n; i += stride) {
      T v = row[i];
      if (v == v) {
        int b = (int)(((double)v - lo) / width);
        b = b >= n_bins ? n_bins - 1 : (b < 0 ? 0 : b);
        hist_add(lds + wave * 64, (unsigned int)b);
      }
    }
  }
  __syncthreads();
  if (tid < n_bins) {
    unsigned int c = lds[tid] + lds[64 + tid] + lds[128 + tid] + lds[192 + tid];
    if (c) atomicAdd(&out[(long long)m * 64 + tid], (unsigned long long)c);
  }
}

inline int grid_x(long long n, int per_thread) {
  long long blocks = (n + (long long)KV_THREADS * per_thread - 1) / ((long long)KV_THREADS * per_thread);
  if (blocks < 1) blocks = 1;
  // 256 CUs x 2 blocks; grid-stride covers the rest.  Every block ends with one global atomic
  // per non-empty bin on the SAME few hundred addresses: with 2048 blocks that flush (about a
  // million contended atomics) cost more than streaming the samples.
  if (blocks > 512) blocks = 512;
  return (int)blocks;
}

// ---------------------------------------------------------------------------------------------
// Live inter-token gaps from raw token events.  events: int64 [n][3] = (request id, token index,
// t_ns) in arrival order, as the load generator's SSE parser appended them; token index < 0 marks
// the end of a request.  The gap of an event with index k > 0 is its time minus the time of the
// same request's previous event: event (req, k - 1) of this batch if it is here, else the time the
// request was last seen in an earlier batch (last_t[req], -1: never).  Three launches:
//   insert: (req, index) -> t of every event into a batch-local open-addressing table
//   emit  : gaps[i] (ms, fp32; NaN for events without a gap) — what stream_hist_kernel then bins
//   commit: last_t[req] = max(last_t[req], t) over the batch (timestamps of a request only grow)
// so the host does no per-event work at all: one copy of the ring's new slice, then launches.
__device__ inline unsigned long long event_key(long long req, long long idx) {
  return ((((unsigned long long)req) << 24) | ((unsigned long long)idx & 0xFFFFFFull)) + 1ull;  // 0 = empty slot
}
__device__ inline unsigned int event_hash(unsigned long long k) {
  k ^= k >> 33; k *= 0xff51afd7ed558ccdull; k ^= k >> 33; k *= 0xc4ceb9fe1a85ec53ull; k ^= k >> 33;
  return (unsigned int)k;
}

__global__ __launch_bounds__(256) void gap_insert_kernel(const long long* __restrict__ ev, int n, unsigned long long* __restrict__ keys, long long* __restrict__ vals,
                                                         unsigned int mask) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const long long req = ev[3 * i], idx = ev[3 * i + 1], t = ev[3 * i + 2];
  if (idx < 0 || req < 0) return;
  const unsigned long long key = event_key(req, idx);
  unsigned int h = event_hash(key) & mask;
  for (unsigned int probe = 0; probe <= mask; ++probe) {  // the table holds at least 2 n slots: a free one exists
    const unsigned long long old = atomicCAS(&keys[h], 0ull, key);
    if (old == 0ull || old == key) { vals[h] = t; return; }
    h = (h + 1) & mask;
  }
}

__global__ __launch_bounds__(256) void gap_emit_kernel(const long long* __restrict__ ev, int n, const unsigned long long* __restrict__ keys,
                                                       const long long* __restrict__ vals, unsigned int mask, const long long* __restrict__ last_t, long long n_last,
                                                       float* __restrict__ gaps) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const long long req = ev[3 * i], idx = ev[3 * i + 1], t = ev[3 * i + 2];
  float gap = __builtin_nanf("");
  if (idx > 0 && req >= 0) {
    long long prev = -1;
    const unsigned long long key = event_key(req, idx - 1);
    unsigned int h = event_hash(key) & mask;
    for (unsigned int probe = 0; probe <= mask; ++probe) {
      const unsigned long long k = keys[h];
      if (k == key) { prev = vals[h]; break; }
      if (k == 0ull) break;
      h = (h + 1) & mask;
    }
    if (prev < 0 && req < n_last) prev = last_t[req];
    if (prev >= 0) gap = (float)((double)(t - prev) * 1e-6);
  }
  gaps[i] = gap;
}

__global__ __launch_bounds__(256) void gap_commit_kernel(const long long* __restrict__ ev, int n, long long* __restrict__ last_t, long long n_last) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const long long req = ev[3 * i], idx = ev[3 * i + 1], t = ev[3 * i + 2];
  if (idx < 0 || req < 0 || req >= n_last) return;
  atomicMax(&last_t[req], t);
}

// Which form a row's length takes, by whole calls of 3 rows (us).  Up to 512 samples each is ranked (512: 26, with one thread for each 33; by digits
// 34 for floats, 56 for doubles).  Longer rows of floats go by digits in one workgroup per row up to SEL_FEW: 1025 take 34, 4096 36, 16384 44, by the
// sample's intervals 41 to 44 whatever the length; 32768 take 50 and 45.  Doubles have twice the digits and go by intervals from there: 1025 take 41
// for 57.
constexpr long long SEL_FEW = 16384;

long long select_work_bytes(int n_metrics) { return (long long)n_metrics * (sizeof(RadixState) + KV_MAX_RANKS * KV_BINS * 4 + 8); }

void radix_pass_geometry(int dtype, int pass, int* shift, int* digit_bits) {
  int top = dtype == 0 ? 32 : 64;
  for (int i = 0;; ++i) {
    const int db = top >= 11 ? 11 : top;
    if (i == pass) { *shift = top - db; *digit_bits = db; return; }
    top -= db;
  }
}

// LDS above 64 KiB has to be asked for, once per kernel
template <typename K>
bool big_lds(K kernel) { return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, SEL_WORDS * 4) == hipSuccess; }

// workgroups per row: one a CU, each with at least 32 KiB of samples
int select_parts(long long n, int n_metrics, int dtype) {
  const long long want = (n * (dtype == 0 ? 4 : 8) + 32767) / 32768, most = n_metrics < 256 ? 256 / n_metrics : 1;
  return (int)(want < 1 ? 1 : want < most ? want : most);
}

Levels levels_of(const double* ps, int n_ps) {
  Levels lv{};
  lv.n = n_ps;
  for (int i = 0; i < n_ps; ++i) lv.p[i] = ps[i];
  return lv;
}

template <typename T>
int select_split(const T* x, long long n, long long row_stride, int n_metrics, int dtype, const Levels& lv, void* work, void* kept, unsigned long long* out, bool again, hipStream_t stream) {
  if (again) {
    hipLaunchKernelGGL(select_again_kernel, dim3(SPANS * SPAN_BINS / SEL_THREADS, n_metrics), dim3(SEL_THREADS), 0, stream, work);
  } else {
    int parts = SAMPLE_PARTS;
    while (parts > 1 && parts * n_metrics > 256) parts /= 2;
    auto sample = sampled(n) == 2 * SEL_THREADS ? select_sample_kernel<T, 2> : select_sample_kernel<T, 4>;
    hipLaunchKernelGGL(sample, dim3(parts, n_metrics), dim3(SEL_THREADS), 0, stream, x, n, row_stride, lv, work);
  }
  const dim3 grid(select_parts(n, n_metrics, dtype), n_metrics);
  static const bool ok = big_lds(select_split_kernel<T, true>) && big_lds(select_split_kernel<T, false>);
  if (!ok) return -2;
  const int room = kept ? kept_room(n, grid.x) : -1;
  const long long row = kept_bytes(n, dtype);
  auto passes = [&](auto keep) {
    hipLaunchKernelGGL((select_split_kernel<T, decltype(keep)::value>), grid, dim3(SEL_THREADS), SPLIT_LDS, stream, x, n, row_stride, lv.n, work, kept, row, room);
    hipLaunchKernelGGL((select_collect_kernel<T, decltype(keep)::value>), grid, dim3(SEL_THREADS), 0, stream, x, n, row_stride, lv, work, out, kept, row, room);
  };
  if (room >= 0) passes(std::true_type{});
  else passes(std::false_type{});
  return (int)hipGetLastError();
}

template <typename T>
int select(const T* x, long long n, long long row_stride, int n_metrics, int dtype, const Levels& lv, void* work, unsigned long long* out, hipStream_t stream) {
  static const bool ok = big_lds(select_few_kernel<T>) && big_lds(select_pass_kernel<T, true>);
  if (!ok) return -2;
  if (n <= SEL_RANKED) {
    hipLaunchKernelGGL(select_by_rank_kernel<T>, dim3(n_metrics), dim3(SEL_THREADS), 0, stream, x, (int)n, row_stride, lv, out);
    return (int)hipGetLastError();
  }
  if (n <= SEL_FEW) {
    hipLaunchKernelGGL(select_few_kernel<T>, dim3(n_metrics), dim3(SEL_THREADS), SEL_WORDS * 4, stream, x, n, row_stride, lv, out);
    return (int)hipGetLastError();
  }
  RadixState* st = (RadixState*)work;
  unsigned int* hist = (unsigned int*)(st + n_metrics);
  unsigned int* done = hist + (long long)n_metrics * KV_MAX_RANKS * KV_BINS;
  const int words = (int)(select_work_bytes(n_metrics) / 4);
  hipLaunchKernelGGL(select_clear_kernel, dim3((words + SEL_THREADS - 1) / SEL_THREADS), dim3(SEL_THREADS), 0, stream, (unsigned int*)work, words);
  const dim3 grid(select_parts(n, n_metrics, dtype), n_metrics);
  const int passes = (dtype == 0 ? 3 : 6);
  for (int p = 0; p < passes; ++p) {
    int shift = 0, digit_bits = 0;
    radix_pass_geometry(dtype, p, &shift, &digit_bits);
    hipLaunchKernelGGL((select_pass_kernel<T, true>), grid, dim3(SEL_THREADS), SEL_WORDS * 4, stream, x, n, row_stride, st, hist, shift, digit_bits, p == 0, lv, done, p == passes - 1 ? out : nullptr);
  }
  return (int)hipGetLastError();
}

}  // namespace

extern "C" {

// keys / vals: scratch tables of `slots` entries (a power of two >= 2 n); keys must be zero on entry
// (the caller clears it: hipMemsetAsync in the binding).  last_t: int64 [n_last], -1 = never seen.
int kv_token_gaps(const long long* ev, int n, unsigned long long* keys, long long* vals, int slots, long long* last_t, long long n_last, float* gaps, hipStream_t stream) {
  if (n <= 0) return 0;
  if (slots < 2 * n || (slots & (slots - 1)) != 0 || n_last < 0) return -1;
  const dim3 grid((n + 255) / 256), block(256);
  hipLaunchKernelGGL(gap_insert_kernel, grid, block, 0, stream, ev, n, keys, vals, (unsigned int)(slots - 1));
  hipLaunchKernelGGL(gap_emit_kernel, grid, block, 0, stream, ev, n, keys, vals, (unsigned int)(slots - 1), last_t, n_last, gaps);
  hipLaunchKernelGGL(gap_commit_kernel, grid, block, 0, stream, ev, n, last_t, n_last);
  return (int)hipGetLastError();
}

size_t kv_stream_state_bytes() { return sizeof(StreamState); }
size_t kv_radix_state_bytes() { return sizeof(RadixState); }

// dtype: 0 = float32, 1 = float64
int kv_stream_hist(const void* x, long long n, long long row_stride, int n_metrics, int dtype, unsigned int* hist, void* state,
                   float lo_log2, float hi_log2, hipStream_t stream) {
  if (n <= 0 || n_metrics <= 0) return 0;
  float inv_step = (float)KV_BINS / (hi_log2 - lo_log2);
  dim3 grid(grid_x(n, 16), n_metrics);
  if (dtype == 0)
    hipLaunchKernelGGL(stream_hist_kernel<float>, grid, dim3(KV_THREADS), 0, stream, (const float*)x, n, row_stride, hist, (StreamState*)state, lo_log2, inv_step);
  else
    hipLaunchKernelGGL(stream_hist_kernel<double>, grid, dim3(KV_THREADS), 0, stream, (const double*)x, n, row_stride, hist, (StreamState*)state, lo_log2, inv_step);
  return (int)hipGetLastError();
}

// Initialise the selection state from quantile levels ``ps`` (device array, n_ps <= 4)
// and the sample counts that kv_stream_hist accumulated.
int kv_radix_init(const void* stream_state, void* st, const double* ps, int n_ps, int n_metrics, hipStream_t stream) {
  hipLaunchKernelGGL(radix_init_kernel, dim3(n_metrics), dim3(64), 0, stream, (const StreamState*)stream_state, (RadixState*)st, ps, n_ps);
  return (int)hipGetLastError();
}

// Selection of the order statistics around n_ps <= 4 quantile levels of every row of x, in scratch memory `work` (kv_select_work_bytes; nothing
// in it needs to be set).  out: [n_metrics][9], the order-preserving keys of the floor and ceil ranks (left-aligned in 64 bits) and the count.
long long kv_select_work_bytes(int n_metrics) { return select_work_bytes(n_metrics); }

int kv_radix_num_passes(int dtype) { return dtype == 0 ? 3 : 6; }

int kv_select_quantiles(const void* x, long long n, long long row_stride, int n_metrics, int dtype, const double* ps, int n_ps, void* work, unsigned long long* out, hipStream_t stream) {
  if (n <= 0 || n_metrics <= 0 || n_metrics > 65535 || n_ps < 1 || n_ps > KV_MAX_RANKS / 2) return -1;
  const Levels lv = levels_of(ps, n_ps);
  return dtype == 0 ? select((const float*)x, n, row_stride, n_metrics, dtype, lv, work, out, stream) : select((const double*)x, n, row_stride, n_metrics, dtype, lv, work, out, stream);
}

// The same by a sample's intervals, for the rows that kv_split_takes (scratch memory: kv_split_work_bytes, and what the passes keep of rows of n samples,
// kv_split_kept_bytes — enough for calls of fewer rows as well; null: nothing is kept): a count of kv_undecided() says that
// kv_select_quantiles has to answer, one of kv_crowded() that this has to be called again with what it left in the scratch memory.
int kv_split_takes(long long n, int n_metrics, int dtype) { return n > (dtype == 0 ? SEL_FEW : SEL_RANKED) && n <= SPLIT_MOST && n_metrics <= 64; }
long long kv_split_work_bytes(int n_metrics) { return n_metrics * SPLIT_BYTES; }
long long kv_split_kept_bytes(long long n, int n_metrics, int dtype, const double* ps, int n_ps) {
  return kept_room(n, select_parts(n, n_metrics, dtype)) < 0 || inside(levels_of(ps, n_ps), n) > 3. / 16 ? 0 : n_metrics * kept_bytes(n, dtype);
}
unsigned long long kv_undecided() { return UNDECIDED; }
unsigned long long kv_crowded() { return CROWDED; }

int kv_split_quantiles(const void* x, long long n, long long row_stride, int n_metrics, int dtype, const double* ps, int n_ps, void* work, void* kept, unsigned long long* out, int again, hipStream_t stream) {
  if (n_metrics <= 0 || !kv_split_takes(n, n_metrics, dtype) || n_ps < 1 || n_ps > KV_MAX_RANKS / 2) return -1;
  const Levels lv = levels_of(ps, n_ps);
  return dtype == 0 ? select_split((const float*)x, n, row_stride, n_metrics, dtype, lv, work, kept, out, again != 0, stream)
                    : select_split((const double*)x, n, row_stride, n_metrics, dtype, lv, work, kept, out, again != 0, stream);
}

// The same selection one pass at a time, for samples spread over several ranks: every rank runs
// pass_hist on its own samples, the ranks SUM the digit histograms (one all-reduce of
// [n_metrics][8][2048] counts per pass), and every rank runs pass_scan on the summed counts — the
// selection state stays identical everywhere and ends at the exact order statistics of the union.
// The state must have been initialised from the GLOBAL sample count.
int kv_radix_pass_hist(const void* x, long long n, long long row_stride, int n_metrics, int dtype, void* st, unsigned int* hist, int pass, hipStream_t stream) {
  if (n_metrics <= 0 || pass < 0 || pass >= kv_radix_num_passes(dtype)) return -1;
  if (n <= 0) return 0;  // a rank without samples contributes zeros
  int shift = 0, digit_bits = 0;
  radix_pass_geometry(dtype, pass, &shift, &digit_bits);
  const dim3 grid(select_parts(n, n_metrics, dtype), n_metrics);
  static const bool ok = big_lds(select_pass_kernel<float, false>) && big_lds(select_pass_kernel<double, false>);
  if (!ok) return -2;
  if (dtype == 0)
    hipLaunchKernelGGL((select_pass_kernel<float, false>), grid, dim3(SEL_THREADS), SEL_WORDS * 4, stream, (const float*)x, n, row_stride, (RadixState*)st, hist, shift, digit_bits, pass == 0, Levels{}, nullptr, nullptr);
  else
    hipLaunchKernelGGL((select_pass_kernel<double, false>), grid, dim3(SEL_THREADS), SEL_WORDS * 4, stream, (const double*)x, n, row_stride, (RadixState*)st, hist, shift, digit_bits, pass == 0, Levels{}, nullptr, nullptr);
  return (int)hipGetLastError();
}

int kv_radix_pass_scan(void* st, unsigned int* hist, int n_metrics, int dtype, int pass, hipStream_t stream) {
  if (n_metrics <= 0 || pass < 0 || pass >= kv_radix_num_passes(dtype)) return -1;
  int shift = 0, digit_bits = 0;
  radix_pass_geometry(dtype, pass, &shift, &digit_bits);
  const int key_bits = dtype == 0 ? 32 : 64;
  static const bool ok = big_lds(select_scan_kernel);
  if (!ok) return -2;
  hipLaunchKernelGGL(select_scan_kernel, dim3(n_metrics), dim3(SEL_THREADS), KV_MAX_RANKS * SEL_ROW * 4, stream, (RadixState*)st, hist, shift + (64 - key_bits), pass == 0);
  return (int)hipGetLastError();
}

int kv_equal_hist(const void* x, long long n, long long row_stride, int n_metrics, int dtype, const void* state, unsigned long long* out, int n_bins,
                  hipStream_t stream) {
  if (n <= 0 || n_metrics <= 0) return 0;
  if (n_bins > 64) return -1;
  dim3 grid(grid_x(n, 8), n_metrics);
  if (dtype == 0)
    hipLaunchKernelGGL(equal_hist_kernel<float>, grid, dim3(KV_THREADS), 0, stream, (const float*)x, n, row_stride, (const StreamState*)state, out, n_bins);
  else
    hipLaunchKernelGGL(equal_hist_kernel<double>, grid, dim3(KV_THREADS), 0, stream, (const double*)x, n, row_stride, (const StreamState*)state, out, n_bins);
  return (int)hipGetLastError();
}

}  // extern "C"
