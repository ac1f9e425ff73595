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
//                        streaming passes and no sort.  The result is bit-exact: the CPU
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

#include <hip/hip_runtime.h>
#include <stdint.h>

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

// counts the digits of the samples first, first + stride, ... (in 16-byte pieces) of a row into h[prefix][bin][copy]; MOST: at least U prefixes
// (0: the first pass, which has none)
template <typename T, int MOST>
__device__ void count_digits(const T* __restrict__ row, long long n, long long first, long long stride, unsigned int* h, const unsigned long long* uniq, int U, int shift, int digit_bits) {
  using KT = typename KeyOf<T>::type;
  constexpr int VEC = 16 / sizeof(T);
  const int cl = log2_copies(U, n), copy = threadIdx.x & ((1 << cl) - 1);
  const KT dmask = (KT)((1u << digit_bits) - 1u);
  const int hi_shift = shift + digit_bits;  // bits above the current digit
  KT pre[MOST > 0 ? MOST : 1] = {};
#pragma unroll
  for (int u = 0; u < MOST; ++u) pre[u] = (KT)((KT)(uniq[u < U ? u : 0] >> (64 - KeyOf<T>::bits)) >> hi_shift);  // (unused ones repeat the first)
  auto visit = [&](T v) {
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
  };
  struct alignas(16) Pack { T v[VEC]; };
  // (rows need not start at a multiple of 16 bytes: the samples in front of the first whole piece and behind the last go one by one)
  long long head = (VEC - (long long)((uintptr_t)row / sizeof(T)) % VEC) % VEC;
  head = head < n ? head : n;
  const Pack* pv = reinterpret_cast<const Pack*>(row + head);
  const long long nvec = (n - head) / VEC, tail = head + nvec * VEC;
  auto visit_pack = [&](const Pack& p) {
#pragma unroll
    for (int j = 0; j < VEC; ++j) visit(p.v[j]);
  };
  constexpr int AHEAD = 4;  // loads in flight per lane while the ones before are counted
  Pack p[AHEAD];
  long long i = first;
  if (i + (AHEAD - 1) * stride < nvec) {
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) p[k] = pv[i + k * stride];
    for (;;) {
      i += AHEAD * stride;
      const bool more = i + (AHEAD - 1) * stride < nvec;
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
  for (; i < nvec; i += stride) visit_pack(pv[i]);
  if (first < head) visit(row[first]);
  if (tail + first < n) visit(row[tail + first]);
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

// Up to 1024 samples (a run's requests): a thread per sample counts how many come in front of it.  A workgroup per metric.
template <typename T>
__global__ __launch_bounds__(SEL_THREADS) void select_by_rank_kernel(const T* __restrict__ x, int n, long long row_stride, Levels levels, unsigned long long* out) {
  __shared__ __attribute__((aligned(16))) unsigned long long keys[SEL_THREADS + 1];
  const int tid = threadIdx.x, m = blockIdx.x;
  const T v = tid < n ? x[(long long)m * row_stride + tid] : (T)0;
  const bool on = tid < n && v == v;
  const unsigned long long key = (unsigned long long)KeyOf<T>::key(v) << (64 - KeyOf<T>::bits);
  const int count = __syncthreads_count(on);
  keys[tid] = on ? key : ~0ull;  // (no sample's key: that one is a NaN's)
  if (tid == 0) keys[SEL_THREADS] = ~0ull;
  __syncthreads();
  int before = 0;
  const int pairs = (tid & ~63) < n ? n : 0;  // (waves without a sample need not count)
#pragma unroll 4
  for (int j = 0; j < pairs; j += 2) {
    const ulonglong2 k = *reinterpret_cast<const ulonglong2*>(&keys[j]);
    before += (k.x < key || (k.x == key && j < tid) ? 1 : 0) + (k.y < key || (k.y == key && j + 1 < tid) ? 1 : 0);
  }
  unsigned long long* o = out + (long long)m * SEL_OUT;
  if (tid == 0) o[KV_MAX_RANKS] = (unsigned long long)count;
  if (on)
    for (int r = 0; r < 2 * levels.n; ++r)
      if (rank_of(levels, r, (unsigned long long)count) == (unsigned long long)before) o[r] = key;
}

// Few samples: all passes in one launch, a workgroup per metric.
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

// Up to SEL_FEW samples a row one workgroup per row makes all passes, beyond a launch per pass (and one that clears) spreads them.  The line lies where
// whole calls take as long: 3 x 32768 floats 59 us in the one form, one sample more a row 63 in the other; 5000 take 43, 100000 65.
constexpr long long SEL_FEW = 32768;

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

template <typename T>
int select(const T* x, long long n, long long row_stride, int n_metrics, int dtype, const Levels& lv, void* work, unsigned long long* out, hipStream_t stream) {
  static const bool ok = big_lds(select_few_kernel<T>) && big_lds(select_pass_kernel<T, true>);
  if (!ok) return -2;
  if (n <= SEL_THREADS) {
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
  Levels lv{};
  lv.n = n_ps;
  for (int i = 0; i < n_ps; ++i) lv.p[i] = ps[i];
  return dtype == 0 ? select((const float*)x, n, row_stride, n_metrics, dtype, lv, work, out, stream) : select((const double*)x, n, row_stride, n_metrics, dtype, lv, work, out, stream);
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
