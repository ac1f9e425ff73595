// Gated delta rule with one decay per key channel, for gfx950.  Per head, with the 32-bit state S [dim, vdim]:
//     S <- diag(g) S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
// q, k, v come out of short causal convolutions (silu behind them), q and k are unit vectors (q also times dim^-1/2),
// g = exp(-exp(A) softplus(z + dt_bias)), beta = sigmoid(b).  o leaves through an RMS norm over vdim and a gate.
//
//   delta_step_kernel     one token per sequence (decoding): convolution, norms, decay, state update, read-out, output norm and
//                         gate in one launch.  A workgroup owns one head's state: every state byte is read and written once, in
//                         whole rows.
//   delta_prep_kernel     portions of several tokens: everything in front of the recurrence, for all tokens in parallel
//   delta_scan_kernel     ... the recurrence token by token: a wave owns a few columns of S in registers, the key channels
//                         spread over its lanes (columns do not interact), no barrier in the loop
//   delta_out_kernel      ... output norm and gate
//   conv_tail_kernel      ... the convolution inputs the next portion still needs
//
// Per-sequence state, indexed by the sequence's slot: S fp32 [slots][heads][dim][vdim] and a ring of the last convolution
// inputs, T [slots][taps][channels], where position p sits at p % taps.  Nothing has to be cleared when a slot changes hands:
// a portion that starts at position 0 takes S as zero, and inputs before position 0 are zero by their index.
// Channels are ordered q [kv_heads dim], k [kv_heads dim], v [heads vdim].

#include <type_traits>

#include "elem.h"
#include "state_rows.h"

namespace {
using namespace elem;

struct DeltaArgs {
  // projections of the step: proj [T, ldp] (q, k, v, beta logits), low [T, ldl] (decay inputs, then output-gate logits)
  long long ldp, ldl;
  int q_off, k_off, v_off, b_off, z_off, gate_off;
  const float* conv_w;   // [taps][channels]
  const float* a_log;    // [heads]
  const float* dt_bias;  // [heads dim]
  const float* o_norm;   // [vdim]
  float* state;
  const int* tok_seq; const int* positions;
  const int* tok_kind;   // 0 padding, 1 the only token of its sequence in this step, 2 a token of a longer portion
  const int* tok_off;    // index of the token inside its portion
  int heads, kv_heads, dim, vdim, taps, channels;
  float eps, out_scale;
  long long ldo; int o_off;
};

// column of channel c of the projections
__device__ inline int chan_col(const DeltaArgs& a, int c) {
  const int qk = a.kv_heads * a.dim;
  return c < qk ? a.q_off + c : c < 2 * qk ? a.k_off + c - qk : a.v_off + c - 2 * qk;
}

// a convolution's sum: the first product is not rounded, the second one is (said here, else it is the compiler's choice at each place)
template <int TAPS>
__device__ inline float taps_sum(const float (&w)[TAPS], const float (&x)[TAPS]) {
  if constexpr (TAPS == 1) return w[0] * x[0];
  else {
    float y = __builtin_fmaf(w[0], x[0], w[1] * x[1]);
#pragma unroll
    for (int j = 2; j < TAPS; ++j) y = __builtin_fmaf(w[j], x[j], y);
    return y;
  }
}

// silu(convolution) of channel c at row t; `back` = rows of the same portion in front of t.  TAPS: compile-time taps (0: a.taps)
template <typename T, int TAPS>
__device__ inline float conv_silu(const DeltaArgs& a, const T* __restrict__ proj, const T* __restrict__ ring, long long t, int pos, int back, int slot, int c) {
  const T* p = proj + t * a.ldp + chan_col(a, c);
  const int taps = TAPS ? TAPS : a.taps;
  auto weight = [&](int j) { return a.conv_w[(taps - 1 - j) * a.channels + c]; };
  auto input = [&](int j) {
    const T* src = j <= back ? p - j * a.ldp : ring + ((long long)slot * taps + (j <= pos ? pos - j : 0) % taps) * a.channels + c;
    const float x = ld(src);
    return j <= pos ? x : 0.f;
  };
  if constexpr (TAPS > 0) {
    float w[TAPS], x[TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) { w[j] = weight(j); x[j] = j ? input(j) : ld(p); }
    return silu(taps_sum<TAPS>(w, x));
  }
  float y = weight(0) * ld(p);
  for (int j = 1; j < taps; ++j) y += weight(j) * input(j);
  return silu(y);
}

__device__ inline float decay_log(const DeltaArgs& a, float z, int h, int d) { return -fast_exp(a.a_log[h]) * softplus(z + a.dt_bias[h * a.dim + d]); }

// ---- decoding ----------------------------------------------------------------------------------------------------
// grid (listed rows, heads), 256 threads: thread = (row group, 4 columns); ROWS = rows of S per thread, EARLY = items of a thread that are asked for ahead of S.  With many rows the state bounds it (read and written, 5 TB/s);
// with few of them a chain of dependent steps does: loads answer in the order they were asked for, so what the convolutions, decays and gates need is asked for ahead
// of the state, and all of that is worked out while the state is on its way from HBM; nothing is loaded behind it.  Key and query are normed where they are used, so that
// the sums of their squares and their product cost no barrier of their own.  6 rows of 16 heads of 128 x 128 11.7 -> 9.8 us, 61 of 32 heads 62.9 -> 50.9.
template <typename T, int ROWS, int TAPS, int EARLY>
__global__ __launch_bounds__(256) void delta_step_kernel(const int* __restrict__ rows, const T* __restrict__ proj, const T* __restrict__ low, T* __restrict__ ring, T* __restrict__ out, DeltaArgs a) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const long long t = rows[blockIdx.x];
  const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (t < 0) return;  // unused entry
  const int kind = a.tok_kind[t], slot = a.tok_seq[t], pos = a.positions[t];
  if (kind != 1) return;  // a padding row
  const int rep = a.heads / a.kv_heads, g = h / rep;
  const StateRows own = state_rows(tid, a.dim, a.vdim);
  const int nrg = own.groups, rg = own.group, col = own.col;
  const bool on = own.on();
  float* qs = sm;                       // [dim]
  float* ks = qs + a.dim;               // [dim]
  float* ds = ks + a.dim;               // [dim] decay factors
  float* vs = ds + a.dim;               // [vdim]
  float* red = vs + a.vdim;             // [2][nrg][vdim]
  __shared__ float scal[4][4];
  const int qk = a.kv_heads * a.dim;
  // What the state meets: queries, keys, decays, values, dealt over the waves in parts of 64.  Each kind begins with a part (heads of more than 256: with the first
  // wave's), so that the lanes that add up squares are the same whatever lies in front of them, and a part is of one kind
  const int section = a.dim <= 256 ? (a.dim + 63) & ~63 : (a.dim + 255) & ~255, parts = (3 * section + a.vdim + 63) >> 6;
  struct Item { int kind, d; bool there; };  // kind: 0 query, 1 key, 2 decay, 3 value
  auto item = [&](int part) {
    Item it;
    it.kind = (64 * part >= section) + (64 * part >= 2 * section) + (64 * part >= 3 * section);
    it.d = 64 * part - it.kind * section + lane;
    const int size = it.kind == 3 ? a.vdim : a.dim;
    it.there = it.d < size;
    it.d = it.d < size - 1 ? it.d : size - 1;  // (behind the last one: that one again)
    return it;
  };
  const int q_channel = g * a.dim, k_channel = qk + q_channel, v_channel = 2 * qk + h * a.vdim;
  const int q_column = a.q_off + q_channel, k_column = a.k_off + q_channel, v_column = a.v_off + h * a.vdim;  // of the projections
  auto channel = [&](const Item& it) { return (it.kind == 3 ? v_channel : it.kind == 1 ? k_channel : q_channel) + it.d; };
  auto column = [&](const Item& it) { return (it.kind == 3 ? v_column : it.kind == 1 ? k_column : q_column) + it.d; };

  // the first EARLY items of a thread, as loaded: no branches and no conversions, which would wait for them
  static_assert(EARLY == 0 || TAPS >= 2, "a convolution of known taps has at least the two words of a decay");
  constexpr int SIZE = TAPS >= 2 ? TAPS : 2;
  unsigned int x[2][SIZE];
  float w[2][SIZE];
#pragma unroll
  for (int e = 0; e < EARLY; ++e) {
    const Item it = item(wave + 4 * e);
    const bool decay = it.kind == 2;
    const int c = decay ? 0 : channel(it), d = decay ? h * a.dim + it.d : 0;
    x[e][0] = raw(decay ? low + t * a.ldl + a.z_off + d : proj + t * a.ldp + column(it));
    w[e][0] = *(decay ? a.dt_bias + d : a.conv_w + (TAPS - 1) * a.channels + c);
#pragma unroll
    for (int m = 1; m < TAPS; ++m) {
      x[e][m] = raw(ring + ((long long)slot * TAPS + (m <= pos ? pos - m : 0) % TAPS) * a.channels + c);
      w[e][m] = *(decay ? a.a_log + h : a.conv_w + (TAPS - 1 - m) * a.channels + c);
    }
  }
  const T* pr = proj + t * a.ldp;
  const T* gates = low + t * a.ldl + a.gate_off + h * a.vdim;
  const int dv = tid < a.vdim ? tid : 0;
  const unsigned int beta_of = raw(pr + a.b_off + h), gate_of = raw(gates + dv);
  const float gain_of = a.o_norm[dv];
  __builtin_amdgcn_sched_barrier(0);

  float* st = a.state + ((long long)slot * a.heads + h) * a.dim * a.vdim;
  float4 s[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) s[i] = ld4(st + own.at(i));
  __builtin_amdgcn_sched_barrier(0);

  float sq = 0.f, sk = 0.f;
  auto keep = [&](const Item& it, float y) {
    sm[it.kind * a.dim + it.d] = y;  // (q, k, decays and v lie one behind another; what several lanes write is the same)
    y = it.there && it.kind < 2 ? y : 0.f;
    const float q = it.kind == 0 ? y : 0.f, k = it.kind == 1 ? y : 0.f;
    sq = __builtin_fmaf(q, q, sq);
    sk = __builtin_fmaf(k, k, sk);
  };
#pragma unroll
  for (int e = 0; e < EARLY; ++e) {
    if (wave + 4 * e >= parts) continue;
    const Item it = item(wave + 4 * e);
    if (it.kind == 2) {
      keep(it, fast_exp(-fast_exp(w[e][1]) * softplus(number<T>(x[e][0]) + w[e][0])));
    } else {
      float v[SIZE];
#pragma unroll
      for (int m = 0; m < SIZE; ++m) v[m] = m <= pos ? number<T>(x[e][m]) : 0.f;
      keep(it, silu(taps_sum<SIZE>(w[e], v)));
    }
  }
  for (int part = wave + 4 * EARLY; part < parts; part += 4) {
    const Item it = item(part);
    keep(it, it.kind == 2 ? fast_exp(decay_log(a, ld(low + t * a.ldl + a.z_off + h * a.dim + it.d), h, it.d)) : conv_silu<T, TAPS>(a, proj, ring, t, pos, 0, slot, channel(it)));
  }
  sq = wave_sum(sq);
  sk = wave_sum(sk);
  if (lane == 0) { scal[0][wave] = sq; scal[1][(wave - section / 64) & 3] = sk; }  // by their part of 64 of a head
  // the ring entry of this position was last used for position pos - taps, which nobody reads any more
  T* rw = ring + ((long long)slot * a.taps + pos % a.taps) * a.channels;
  auto pass_on = [&](const Item& it, float v) { elem::st(rw + channel(it), v); };
  auto passed_on = [&](const Item& it) { return it.there && (it.kind == 3 || (it.kind != 2 && h % rep == 0)); };
#pragma unroll
  for (int e = 0; e < EARLY; ++e)
    if (const Item it = item(wave + 4 * e); passed_on(it)) pass_on(it, number<T>(x[e][0]));
  for (int part = wave + 4 * EARLY; part < parts; part += 4)
    if (const Item it = item(part); passed_on(it)) pass_on(it, ld(pr + column(it)));
  __syncthreads();
  const float nq = 1.f / (sqrtf(scal[0][0] + scal[0][1] + scal[0][2] + scal[0][3] + 1e-6f) * sqrtf((float)a.dim));
  const float nk = 1.f / sqrtf(scal[1][0] + scal[1][1] + scal[1][2] + scal[1][3] + 1e-6f);
  float kq = 0.f;
  for (int d = tid; d < a.dim; d += 256) kq += (qs[d] * nq) * (ks[d] * nk);
  kq = wave_sum(kq);
  if (lane == 0) scal[2][wave] = kq;
  if (pos == 0) {  // (here and not around the loads: where ways with and without them meet, all of them would be waited for)
#pragma unroll
    for (int i = 0; i < ROWS; ++i) s[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // decay, and both products with the decayed state at once: o = S'^T q = (diag(g) S)^T q + (k . q) u
  float4 ak = make_float4(0.f, 0.f, 0.f, 0.f), aq = ak;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    if (i < own.count) {
      const int r = rg + i * nrg;
      const float dr = ds[r], kv = ks[r] * nk, qv = qs[r] * nq;
      s[i].x *= dr; s[i].y *= dr; s[i].z *= dr; s[i].w *= dr;
      ak.x += s[i].x * kv; ak.y += s[i].y * kv; ak.z += s[i].z * kv; ak.w += s[i].w * kv;
      aq.x += s[i].x * qv; aq.y += s[i].y * qv; aq.z += s[i].z * qv; aq.w += s[i].w * qv;
    }
  }
  if (on) {
    st4(red + rg * a.vdim + col, ak);
    st4(red + (nrg + rg) * a.vdim + col, aq);
  }
  __syncthreads();
  kq = scal[2][0] + scal[2][1] + scal[2][2] + scal[2][3];
  const float beta = sigmoid(number<T>(beta_of));
  float oss = 0.f;
  for (int d = tid; d < a.vdim; d += 256) {
    float xk = 0.f, xq = 0.f;
    for (int r = 0; r < nrg; ++r) {
      xk += red[r * a.vdim + d];
      xq += red[(nrg + r) * a.vdim + d];
    }
    const float u = beta * (vs[d] - xk);
    const float o = xq + kq * u;
    vs[d] = u;
    red[d] = o;  // (row group 0's partial of this column, read by this thread only)
    oss += o * o;
  }
  oss = wave_sum(oss);
  if (lane == 0) scal[3][wave] = oss;
  __syncthreads();
  if (on) {
    const float4 u = ld4(vs + col);
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      if (i < own.count) {
        const float kv = ks[rg + i * nrg] * nk;
        s[i].x += kv * u.x; s[i].y += kv * u.y; s[i].z += kv * u.z; s[i].w += kv * u.w;
        st4(st + own.at(i), s[i]);
      }
    }
  }
  const float rs = a.out_scale / sqrtf((scal[3][0] + scal[3][1] + scal[3][2] + scal[3][3]) / (float)a.vdim + a.eps);
  T* dst = out + t * a.ldo + a.o_off + h * a.vdim;
  for (int d = tid; d < a.vdim; d += 256) {
    const bool first = d < 256;
    elem::st(dst + d, red[d] * rs * (first ? gain_of : a.o_norm[d]) * sigmoid(first ? number<T>(gate_of) : ld(gates + d)));
  }
}

// ---- portions ----------------------------------------------------------------------------------------------------
// One wave per (token, unit); units: q heads, k heads (unit vectors), v heads (with beta), decay heads.  Rows of qn, kn and dec
// are dimp wide (dim rounded up to 8; zero, for dec one, behind dim).
template <typename T>
__global__ __launch_bounds__(256) void delta_prep_kernel(const T* __restrict__ proj, const T* __restrict__ low, const T* __restrict__ ring, float* __restrict__ qn, float* __restrict__ kn,
                                                         float* __restrict__ vv, float* __restrict__ dec, float* __restrict__ beta, int dimp, int min_kind, DeltaArgs a) {
  const long long t = blockIdx.x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int unit = blockIdx.y * 4 + wave;
  if (a.tok_kind[t] < min_kind) return;
  if (unit >= 2 * a.kv_heads + 2 * a.heads) return;
  const int slot = a.tok_seq[t], pos = a.positions[t], back = a.tok_off[t];
  if (unit < 2 * a.kv_heads) {
    const bool is_q = unit < a.kv_heads;
    float* dst = (is_q ? qn : kn) + (t * a.kv_heads + (is_q ? unit : unit - a.kv_heads)) * dimp;
    float ss = 0.f;
    for (int d = lane; d < a.dim; d += 64) {
      const float y = conv_silu<T, 0>(a, proj, ring, t, pos, back, slot, unit * a.dim + d);
      dst[d] = y;
      ss += y * y;
    }
    ss = wave_sum(ss);
    const float n = is_q ? 1.f / (sqrtf(ss + 1e-6f) * sqrtf((float)a.dim)) : 1.f / sqrtf(ss + 1e-6f);
    for (int d = lane; d < dimp; d += 64) dst[d] = d < a.dim ? dst[d] * n : 0.f;  // (the lane's own entries)
  } else if (unit < 2 * a.kv_heads + a.heads) {
    const int h = unit - 2 * a.kv_heads;
    for (int d = lane; d < a.vdim; d += 64)
      vv[(t * a.heads + h) * a.vdim + d] = conv_silu<T, 0>(a, proj, ring, t, pos, back, slot, 2 * a.kv_heads * a.dim + h * a.vdim + d);
    if (lane == 0) beta[t * a.heads + h] = sigmoid(ld(proj + t * a.ldp + a.b_off + h));
  } else {
    const int h = unit - 2 * a.kv_heads - a.heads;
    float* dst = dec + (t * a.heads + h) * dimp;
    for (int d = lane; d < dimp; d += 64) dst[d] = d < a.dim ? fast_exp(decay_log(a, ld(low + t * a.ldl + a.z_off + h * a.dim + d), h, d)) : 1.f;
  }
}

// Portions: seg arrays [n_segs] first row, tokens (0 = unused), first position, slot.  RG lanes share a column, 8 rows of S per lane.
template <int RG>
__global__ __launch_bounds__(256) void delta_scan_kernel(const float* __restrict__ qn, const float* __restrict__ kn, const float* __restrict__ vv, const float* __restrict__ dec,
                                                         const float* __restrict__ beta, float* __restrict__ o, const int* __restrict__ seg_row, const int* __restrict__ seg_n,
                                                         const int* __restrict__ seg_pos, const int* __restrict__ seg_slot, int min_n, int dimp, float* __restrict__ state, int heads,
                                                         int kv_heads, int dim, int vdim) {
  constexpr int CPW = 64 / RG, RPL = 8;
  const int sg = blockIdx.z, h = blockIdx.y;
  const int n = seg_n[sg];
  if (n < min_n || n == 0) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int rgi = lane / CPW;
  const int col = (blockIdx.x * 4 + wave) * CPW + lane % CPW;
  const bool on = col < vdim;
  const int colc = on ? col : vdim - 1;
  const int r0 = rgi * RPL;
  const bool rows_on = r0 < dimp;
  const int g = h / (heads / kv_heads);
  const long long row0 = seg_row[sg];
  float* st = state + ((long long)seg_slot[sg] * heads + h) * dim * vdim + colc;
  float s[RPL];
  const bool fresh = seg_pos[sg] == 0;
#pragma unroll
  for (int i = 0; i < RPL; ++i) s[i] = (!fresh && r0 + i < dim) ? st[(long long)(r0 + i) * vdim] : 0.f;
  float4 q0, q1, k0, k1, d0, d1;
  float v, b;
  const int r0c = rows_on ? r0 : 0;
#define KV_FETCH(ROW)                                                            \
  do {                                                                           \
    const float* qp = qn + ((ROW) * kv_heads + g) * dimp + r0c;                  \
    const float* kp = kn + ((ROW) * kv_heads + g) * dimp + r0c;                  \
    const float* dp = dec + ((ROW) * heads + h) * dimp + r0c;                    \
    q0 = ld4(qp); q1 = ld4(qp + 4); k0 = ld4(kp); k1 = ld4(kp + 4);              \
    d0 = ld4(dp); d1 = ld4(dp + 4);                                              \
    v = vv[((ROW) * heads + h) * vdim + colc];                                   \
    b = beta[(ROW) * heads + h];                                                 \
  } while (0)
  KV_FETCH(row0);
  for (int i = 0; i < n; ++i) {
    const float q[RPL] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    float k[RPL] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
    const float d[RPL] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
    const float vi = v, bi = b;
    const long long row = row0 + i;
    if (i + 1 < n) KV_FETCH(row + 1);
    float xk = 0.f;
#pragma unroll
    for (int r = 0; r < RPL; ++r) {
      if (!rows_on) k[r] = 0.f;
      s[r] *= d[r];
      xk += s[r] * k[r];
    }
    xk = lanes::meet_up<CPW, 64>(xk, lanes::Sum{});
    const float u = bi * (vi - xk);
    float xq = 0.f;
#pragma unroll
    for (int r = 0; r < RPL; ++r) {
      s[r] += k[r] * u;
      xq += s[r] * q[r];
    }
    xq = lanes::meet_up<CPW, 64>(xq, lanes::Sum{});
    if (rgi == 0 && on) o[(row * heads + h) * vdim + col] = xq;
  }
#undef KV_FETCH
  if (on) {
#pragma unroll
    for (int i = 0; i < RPL; ++i)
      if (r0 + i < dim) st[(long long)(r0 + i) * vdim] = s[i];
  }
}

// LPR lanes per (token, head), four columns per lane and pass
template <typename T, int LPR>
__global__ __launch_bounds__(256) void delta_out_kernel(const float* __restrict__ o, const T* __restrict__ low, T* __restrict__ out, int min_kind, DeltaArgs a) {
  const long long t = blockIdx.x;
  const int h = blockIdx.y * (256 / LPR) + threadIdx.x / LPR, lane = threadIdx.x % LPR;
  if (h >= a.heads || a.tok_kind[t] < min_kind) return;
  T* dst = out + t * a.ldo + a.o_off + h * a.vdim;
  const float* src = o + (t * a.heads + h) * a.vdim;
  const T* gl = low + t * a.ldl + a.gate_off + h * a.vdim;
  if ((a.vdim & 3) == 0) {
    float ss = 0.f;
    for (int d = 4 * lane; d < a.vdim; d += 4 * LPR) {
      const float4 v = ld4(src + d);
      ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    }
    ss = lanes::meet_up<1, LPR>(ss, lanes::Sum{});
    const float rs = a.out_scale / sqrtf(ss / (float)a.vdim + a.eps);
    for (int d = 4 * lane; d < a.vdim; d += 4 * LPR) {
      float4 v = ld4(src + d);
      const float4 z = ld4(gl + d), n = ld4(a.o_norm + d);
      v.x *= rs * n.x * sigmoid(z.x); v.y *= rs * n.y * sigmoid(z.y); v.z *= rs * n.z * sigmoid(z.z); v.w *= rs * n.w * sigmoid(z.w);
      st4(dst + d, v);
    }
  } else {
    float ss = 0.f;
    for (int d = lane; d < a.vdim; d += LPR) ss += src[d] * src[d];
    ss = lanes::meet_up<1, LPR>(ss, lanes::Sum{});
    const float rs = a.out_scale / sqrtf(ss / (float)a.vdim + a.eps);
    for (int d = lane; d < a.vdim; d += LPR) st(dst + d, src[d] * rs * a.o_norm[d] * sigmoid(ld(gl + d)));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void conv_tail_kernel(const T* __restrict__ proj, T* __restrict__ ring, const int* __restrict__ seg_row, const int* __restrict__ seg_n,
                                                        const int* __restrict__ seg_pos, const int* __restrict__ seg_slot, int min_n, DeltaArgs a) {
  const int sg = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
  const int n = seg_n[sg];
  if (n < min_n || n == 0 || c >= a.channels) return;
  const int keep = n < a.taps ? n : a.taps;
  const T* p = proj + (long long)seg_row[sg] * a.ldp + chan_col(a, c);
  T* rw = ring + (long long)seg_slot[sg] * a.taps * a.channels + c;
  for (int i = n - keep; i < n; ++i) rw[(long long)((seg_pos[sg] + i) % a.taps) * a.channels] = p[i * a.ldp];
}

// ---- portions in tiles of 16 tokens (key sizes up to 256) ----------------------------------------------------------
// With G_i the running sum of log decays inside a tile (per key channel), kb_i = k_i e^{G_i}, qb_i = q_i e^{G_i},
// A_ij = sum_d k_i k_j e^{G_i - G_j} (j < i), B_ij = sum_d q_i k_j e^{G_i - G_j} (j <= i) and S the state in front of the tile:
//     u_i = beta_i (v_i - S^T kb_i - sum_{j<i} A_ij u_j),   o_i = S^T qb_i + sum_{j<=i} B_ij u_j,
//     S' = diag(e^{G_15}) S + sum_j (k_j e^{G_15 - G_j}) u_j^T.
// Every exponent is <= 0 (differences are taken before the exponential), so strong decays only underflow.
// delta_tile_kernel solves the triangular part of a tile for all columns at once (forward substitution on [kb | v]), in parallel
// over tiles and heads:  u = tv - tk S,  o = ov + qe S,  with ke_j = k_j e^{G_15 - G_j}.  delta_chain_kernel then walks the tiles
// of a portion with S in matrix-core accumulators (fp32 in and out): two products and one update per tile.
// Workspace of a (tile, head), in the order in which the lanes of the chain read it, 16 bytes each: tk and qe [dkp / 4][16 tokens][4 channels],
// ke [dkp / 16][4][16 channels][4 tokens], gc [dkp], tv and ov [4][dvp][4 tokens].
__host__ __device__ inline long long tile_floats(int dkp, int dvp) { return 49LL * dkp + 32LL * dvp; }

typedef __attribute__((ext_vector_type(4))) float f4;

// What counts in delta_tile_kernel is how many workgroups a CU holds, and that none of them waits for long.  Partial sums of the pairs with j < i alone (the
// 36 blocks of 2 x 2) make that four, of 40 KB, with 128 channels and columns.  All rows that a workgroup reads are on their way before the first is used, a
// row of 16 tokens is summed by sixteen lanes, and all lanes have pairs with j < i to work out (on the diagonal B is the product of the unit vectors, summed as
// they are made).  4 x 560 tokens of 32 heads, us a layer in the profile of a step: 72 (one column's rows at a time, sums over a wave, 28 lanes of 64
// idle over the pairs 100); the bytes it writes alone would take 37.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ inline rsrc_t rows_of(const void* p) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, -1, 0x00027000); }
template <typename T> __device__ inline T load(rsrc_t from, unsigned lane_off, unsigned off);
template <> __device__ inline float load<float>(rsrc_t from, unsigned lane_off, unsigned off) { return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, lane_off, off, 0)); }
template <> __device__ inline bf16raw load<bf16raw>(rsrc_t from, unsigned lane_off, unsigned off) { return __builtin_amdgcn_raw_buffer_load_b16(from, lane_off, off, 0); }
// the sum over the sixteen lanes of a row, in each of them
__device__ inline float row16_sum(float v) {
  auto turned = [&](auto by) __attribute__((always_inline)) { return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x120 + decltype(by)::value, 0xf, 0xf, true)); };
  v += turned(std::integral_constant<int, 8>{});
  v += turned(std::integral_constant<int, 4>{});
  v += turned(std::integral_constant<int, 2>{});
  return v + turned(std::integral_constant<int, 1>{});
}
// where the pair (i, j) of a tile's rows is kept
constexpr int PAIRS = 144;
__device__ inline int pair_of(int i, int j) { return ((i >> 1) * ((i >> 1) + 1) / 2 + (j >> 1)) * 4 + (i & 1) * 2 + (j & 1); }

template <typename T, int TAPS, int DKP>
__global__ __launch_bounds__(256, 4) void delta_tile_kernel(const T* __restrict__ proj, const T* __restrict__ low, const T* __restrict__ ring, float* __restrict__ ws,
                                                         const int* __restrict__ tile_row, const int* __restrict__ tile_n, const int* __restrict__ tile_pos,
                                                         const int* __restrict__ tile_slot, int dvp, DeltaArgs a) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  constexpr int dkp = DKP, rs = DKP + 4;
  const int b = blockIdx.y, h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = tile_n[b];
  if (n == 0) return;
  float* qs = sm;              // [16][rs]
  float* ks = qs + 16 * rs;    // [16][rs]
  float* gs = ks + 16 * rs;    // [16][rs] running log2 decays
  float* vs = gs + 16 * rs;    // [16][dvp]
  float* pp = vs + 16 * dvp;   // [4 waves][2][PAIRS] partial A, B
  float* am = pp + 8 * PAIRS;  // [16][20] beta_i A_ij
  float* bm = am + 320;        // [16][20]
  __shared__ float beta[16], own[16];  // own: B_ii, a product without a decay
  const long long row0 = tile_row[b];
  const int pos0 = tile_pos[b], slot = tile_slot[b], back0 = a.tok_off[row0];
  const int rep = a.heads / a.kv_heads, g = h / rep, qk = a.kv_heads * a.dim;
  const float beta_in = ld(proj + (row0 + (tid < n ? tid : 0)) * a.ldp + a.b_off + h);
  // A task is a column of q, k, the decay inputs or v.  The rows of two are on their way at once, each by as many loads, whatever it is: behind a branch the
  // first one's would be waited for together with the second's.  A row's place is a scalar, the column a lane's.
  struct Task { T x[TAPS + 15]; float w[TAPS ? TAPS : 1], bias; int kind, d; bool live; };
  auto fetch = [&](Task& t, int first) __attribute__((always_inline)) {  // first: of the wave's (sizes are multiples of 64 but for the last kind's)
    t.kind = first < 3 * dkp ? first / dkp : 3;
    t.d = first - t.kind * dkp + lane;
    const bool gate = t.kind == 2;
    const int most = t.kind == 3 ? a.vdim : a.dim, at = t.d < most ? t.d : most - 1;
    t.live = t.d < most;
    const int c = gate ? 0 : t.kind == 0 ? g * a.dim + at : t.kind == 1 ? qk + g * a.dim + at : 2 * qk + h * a.vdim + at;
    const unsigned col = gate ? a.z_off + h * a.dim + at : chan_col(a, c), ld_bytes = (unsigned)(gate ? a.ldl : a.ldp) * sizeof(T);
#pragma unroll
    for (int i = 1 - TAPS; i < 0; ++i) {  // inputs in front of the tile: of the same portion, else from the ring
      const bool same = -i <= back0 && !gate;
      const T* from = same ? proj + (row0 + i) * a.ldp : ring + ((long long)slot * TAPS + (pos0 + i >= 0 ? pos0 + i : 0) % TAPS) * a.channels;
      t.x[i + TAPS - 1] = from[same ? col : (unsigned)c];
    }
    const rsrc_t from = rows_of(gate ? low + row0 * a.ldl : proj + row0 * a.ldp);
    unsigned row = 0;  // (rows past the tile's last one: the last one again)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      t.x[TAPS - 1 + i] = load<T>(from, col * sizeof(T), row);
      row += i + 1 < n ? ld_bytes : 0;
    }
#pragma unroll
    for (int j = 0; j < TAPS; ++j) t.w[j] = a.conv_w[j * a.channels + c];
    t.bias = a.dt_bias[h * a.dim + (gate ? at : 0)];
  };
  auto finish = [&](const Task& t) __attribute__((always_inline)) {
    if (t.kind == 3 && t.d >= dvp) return;
    const int stride = t.kind == 3 ? dvp : rs;
    float* dst = (t.kind == 0 ? qs : t.kind == 1 ? ks : t.kind == 2 ? gs : vs) + t.d;
    if (t.kind == 2) {
      const float rate = -1.4426950408889634f * fast_exp(a.a_log[h]);
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float step = rate * softplus(ld(&t.x[TAPS - 1 + i]) + t.bias);
        sum += i < n ? step : 0.f;
        dst[i * stride] = t.live ? sum : 0.f;
        if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
      return;
    }
    float x[TAPS + 15];
#pragma unroll
    for (int i = 0; i < TAPS + 15; ++i) x[i] = i >= TAPS - 1 || pos0 + i - (TAPS - 1) >= 0 ? ld(&t.x[i]) : 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float y = 0.f;
#pragma unroll
      for (int j = TAPS - 1; j >= 0; --j) y += t.w[j] * x[i + j];
      y = silu(y);
      dst[i * stride] = t.live && i < n ? y : 0.f;
      if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  };
  const int tasks = 3 * dkp + dvp;
  if constexpr (TAPS > 0) {
    for (int t0 = 64 * __builtin_amdgcn_readfirstlane(wave); t0 < tasks; t0 += 512) {
      Task one, two;
      const bool more = t0 + 256 < tasks;
      fetch(one, t0);
      fetch(two, more ? t0 + 256 : t0);
      __builtin_amdgcn_sched_barrier(0);
      finish(one);
      __builtin_amdgcn_sched_barrier(0);
      if (more) finish(two);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    for (int task = tid; task < tasks; task += 256) {
      const int kind = task < 3 * dkp ? task / dkp : 3, d = task - kind * dkp, stride = kind == 3 ? dvp : rs;
      float* dst = (kind == 0 ? qs : kind == 1 ? ks : kind == 2 ? gs : vs) + d;
      const bool live = d < (kind == 3 ? a.vdim : a.dim);
      const int c = kind == 0 ? g * a.dim + d : kind == 1 ? qk + g * a.dim + d : 2 * qk + h * a.vdim + d;
      float sum = 0.f;
      for (int i = 0; i < 16; ++i) {
        if (kind == 2 && live && i < n) sum += 1.4426950408889634f * decay_log(a, ld(low + (row0 + i) * a.ldl + a.z_off + h * a.dim + d), h, d);
        dst[i * stride] = kind == 2 ? sum : live && i < n ? conv_silu<T, 0>(a, proj, ring, row0 + i, pos0 + i, back0 + i, slot, c) : 0.f;
      }
    }
  }
  if (tid < 16) beta[tid] = tid < n ? sigmoid(beta_in) : 0.f;
  __syncthreads();
  {  // sixteen lanes a row
    const int i = tid >> 4, d0 = 4 * (tid & 15);
    float sq = 0.f, sk = 0.f, sb = 0.f;
    for (int d = d0; d < dkp; d += 64) {
      const f4 q = *reinterpret_cast<const f4*>(qs + i * rs + d), k = *reinterpret_cast<const f4*>(ks + i * rs + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sq += q[e] * q[e];
        sk += k[e] * k[e];
      }
    }
    sq = row16_sum(sq);
    sk = row16_sum(sk);
    const float nq = 1.f / (sqrtf(sq + 1e-6f) * sqrtf((float)a.dim)), nk = 1.f / sqrtf(sk + 1e-6f);
    for (int d = d0; d < dkp; d += 64) {
      const f4 q = *reinterpret_cast<const f4*>(qs + i * rs + d) * nq, k = *reinterpret_cast<const f4*>(ks + i * rs + d) * nk;
      *reinterpret_cast<f4*>(qs + i * rs + d) = q;
      *reinterpret_cast<f4*>(ks + i * rs + d) = k;
#pragma unroll
      for (int e = 0; e < 4; ++e) sb += q[e] * k[e];
    }
    sb = row16_sum(sb);
    if (d0 == 0) own[i] = sb;  // (of the normed rows: where a square overflows the norm makes zeros of them)
  }
  __syncthreads();
  {  // partial A, B: a wave has a quarter of the channels, two lanes every other four of them for the pairs (2 bi + x, 2 bj + y), bi > bj; a lane on
     // the diagonal, where only (2 bi + 1, 2 bi) is left, has that pair twice, and (x, x) of its products count
    const int bi = lane >> 3, bj = lane & 7, hi = bi > bj ? bi : bj, lo = bi > bj ? bj : bi, quarter = dkp >> 2;
    int oi[2], oj[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      oi[x] = (2 * hi + (hi == lo ? 1 : x)) * rs + wave * quarter + (hi == lo ? 4 * x : bi < bj ? 4 : 0);
      oj[x] = (2 * lo + (hi == lo ? 0 : x)) * rs + wave * quarter + (hi == lo ? 4 * x : bi < bj ? 4 : 0);
    }
    float pa[2][2] = {{0.f, 0.f}, {0.f, 0.f}}, pb[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
#pragma unroll 1
    for (int d = 0; d < quarter; d += 8) {
      f4 ki[2], qi[2], gi[2], kj[2], gj[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        ki[x] = *reinterpret_cast<const f4*>(ks + oi[x] + d);
        qi[x] = *reinterpret_cast<const f4*>(qs + oi[x] + d);
        gi[x] = *reinterpret_cast<const f4*>(gs + oi[x] + d);
        kj[x] = *reinterpret_cast<const f4*>(ks + oj[x] + d);
        gj[x] = *reinterpret_cast<const f4*>(gs + oj[x] + d);
      }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float w = kj[y][e] * __builtin_amdgcn_exp2f(gi[x][e] - gj[y][e]);  // (on the diagonal, x != y: may overflow, not used)
            pa[x][y] += ki[x][e] * w;
            pb[x][y] += qi[x][e] * w;
          }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        const float oa = __shfl(pa[x][y], 8 * bj + bi), ob = __shfl(pb[x][y], 8 * bj + bi);
        if (bi > bj) {
          const int i = pair_of(2 * bi + x, 2 * bj + y);
          pp[wave * 2 * PAIRS + i] = pa[x][y] + oa;
          pp[(wave * 2 + 1) * PAIRS + i] = pb[x][y] + ob;
        }
      }
    if (bi == bj) {
      const int i = pair_of(2 * bi + 1, 2 * bi);
      pp[wave * 2 * PAIRS + i] = pa[0][0] + pa[1][1];
      pp[(wave * 2 + 1) * PAIRS + i] = pb[0][0] + pb[1][1];
    }
  }
  __syncthreads();
  {
    const int i = tid >> 4, j = tid & 15;
    const float* p = pp + (j < i ? pair_of(i, j) : 2);  // (2: the pair (1, 0))
    am[i * 20 + j] = j < i ? beta[i] * (p[0] + p[2 * PAIRS] + p[4 * PAIRS] + p[6 * PAIRS]) : 0.f;
    bm[i * 20 + j] = j < i ? p[PAIRS] + p[3 * PAIRS] + p[5 * PAIRS] + p[7 * PAIRS] : j == i ? own[i] : 0.f;
  }
  __syncthreads();
  float* w = ws + ((long long)b * a.heads + h) * tile_floats(dkp, dvp);
  auto solve = [&](float (&x)[16], float (&y)[16], float sgn) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      f4 ar[4], br[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * j <= i) {
          ar[j] = *reinterpret_cast<const f4*>(am + i * 20 + 4 * j);
          br[j] = *reinterpret_cast<const f4*>(bm + i * 20 + 4 * j);
        }
      float s = beta[i] * x[i];
#pragma unroll
      for (int j = 0; j < i; ++j) s -= ar[j >> 2][j & 3] * x[j];
      x[i] = s;
      float r = 0.f;
#pragma unroll
      for (int j = 0; j <= i; ++j) r += br[j >> 2][j & 3] * x[j];
      y[i] += sgn * r;
      asm volatile("" ::: "memory");  // (a row's coefficients are read when they are needed: all of them at once would fill the registers)
    }
  };
  {  // keys: their columns go back to where the rows of q and k were, and from there to memory
    float x[16], y[16];
    if (tid < dkp) {
      const int c = tid;
      const float gl = gs[15 * rs + c];
      f4 kv[4];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float gg = gs[i * rs + c], kk = ks[i * rs + c], eg = __builtin_amdgcn_exp2f(gg);
        x[i] = kk * eg;
        y[i] = qs[i * rs + c] * eg;
        kv[i >> 2][i & 3] = kk * __builtin_amdgcn_exp2f(gl - gg);
        if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<f4*>(w + 32 * dkp + (c >> 4) * 256 + i * 64 + (c & 15) * 4) = kv[i];
      w[48 * dkp + c] = __builtin_amdgcn_exp2f(gl);
    }
    __syncthreads();
    if (tid < dkp) {
      solve(x, y, -1.f);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        qs[i * rs + tid] = x[i];
        ks[i * rs + tid] = y[i];
      }
    }
  }
  for (int c0 = tid + (tid < dkp ? 256 : 0) - dkp; c0 < dvp; c0 += 256) {
    int c = c0;
    asm volatile("" : "+v"(c));  // (the rows' places are worked out where they are needed and not in front of the loop, where they would fill the registers)
    float x[16], y[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      x[i] = vs[i * dvp + c];
      y[i] = 0.f;
    }
    solve(x, y, 1.f);
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      *reinterpret_cast<f4*>(w + 49 * dkp + (i * dvp + 4 * c)) = (f4){x[i], x[i + 1], x[i + 2], x[i + 3]};
      *reinterpret_cast<f4*>(w + 49 * dkp + ((16 + i) * dvp + 4 * c)) = (f4){y[i], y[i + 1], y[i + 2], y[i + 3]};
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = tid; j < 8 * dkp; j += 256) {
    const int piece = j % (4 * dkp);
    *reinterpret_cast<f4*>(w + 4 * j) = *reinterpret_cast<const f4*>((j < 4 * dkp ? qs : ks) + (piece & 15) * rs + (piece >> 4) * 4);
  }
}

// A workgroup has 16 CT columns of S and the dkp = 64 RT key channels over four waves (RT row tiles of 16 each).
// mfma_f32_16x16x4: A lane (row l & 15, k l >> 4), B lane (column l & 15, k l >> 4), D lane rows 4 (l >> 4) + r.  The k order of the
// products with S is chosen so that an accumulator register is a B operand as it is: step s takes the channels 4 q + s.
// LEAN: addresses are scalars and four 32-bit offsets of a lane; as pointers of a lane they take some thirty registers, and a long chain is 2 % faster
// (1 x 2048 tokens: 251 us, 257).
template <typename T, int RT, int CT, bool LEAN>
__device__ __attribute__((always_inline)) inline void delta_chain(f4* lds, int y, int n, const float* __restrict__ ws, float* __restrict__ o, const T* __restrict__ proj, T* __restrict__ ring, const int* __restrict__ seg_row,
                                                                  const int* __restrict__ seg_pos, const int* __restrict__ seg_slot, const int* __restrict__ seg_tile, int dkp, int dvp, const DeltaArgs& a) {
  f4(*part)[4][2 * CT][64] = reinterpret_cast<f4(*)[4][2 * CT][64]>(lds);
  const int h = blockIdx.x, sg = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const int col = y * (16 * CT) + lr, base = wave * RT * 16;  // (and the columns 16 further)
  bool col_on[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) col_on[c] = col + 16 * c < a.vdim;
  const int pos0 = seg_pos[sg], slot = seg_slot[sg], nt = (n + 15) >> 4;
  const long long row0 = seg_row[sg];
  const long long tf = tile_floats(dkp, dvp), step = tf * a.heads;
  const float* w = ws + ((long long)seg_tile[sg] * a.heads + h) * tf;
  float* sp = a.state + ((long long)slot * a.heads + h) * a.dim * a.vdim + col;
  f4 s[CT][RT];
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = base + 16 * t + 4 * lq + r;
        s[c][t][r] = (pos0 > 0 && col_on[c] && d < a.dim) ? sp[(long long)d * a.vdim + 16 * c] : 0.f;
      }
  // two tiles in flight: a tile's coefficients come from beyond this XCD's L2 the first time, and one tile takes less time than that
  struct Tile { f4 tk[RT], qe[RT], ke[RT], gc[RT], tv[CT]; float ov[CT]; };
  Tile ta, tb;
  const unsigned int at_row = base * 64 + lane * 16, at_gc = (base + 4 * lq) * 4, at_col = (lq * dvp + col) * 16;
  auto fetch = [&](Tile& x, int i) __attribute__((always_inline)) {
    const float* p = w + step * (i < nt ? i : nt - 1);
    if constexpr (LEAN) {
      auto at = [](const float* from, unsigned int off) __attribute__((always_inline)) { return reinterpret_cast<const char*>(from) + off; };
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        x.tk[t] = *reinterpret_cast<const f4*>(at(p, at_row) + 1024 * t);
        x.qe[t] = *reinterpret_cast<const f4*>(at(p + 16 * dkp, at_row) + 1024 * t);
        x.ke[t] = *reinterpret_cast<const f4*>(at(p + 32 * dkp, at_row) + 1024 * t);
        x.gc[t] = *reinterpret_cast<const f4*>(at(p + 48 * dkp, at_gc) + 64 * t);
      }
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        x.tv[c] = *reinterpret_cast<const f4*>(at(p + 49 * dkp, at_col) + 256 * c);
        x.ov[c] = *reinterpret_cast<const float*>(at(p + 49 * dkp + 16 * dvp + wave, at_col) + 256 * c);
      }
    } else {
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        x.tk[t] = *reinterpret_cast<const f4*>(p + (base + 16 * t) * 16 + 4 * lane);
        x.qe[t] = *reinterpret_cast<const f4*>(p + (dkp + base + 16 * t) * 16 + 4 * lane);
        x.ke[t] = *reinterpret_cast<const f4*>(p + (2 * dkp + base + 16 * t) * 16 + 4 * lane);
        x.gc[t] = *reinterpret_cast<const f4*>(p + 48 * dkp + base + 16 * t + 4 * lq);
      }
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        x.tv[c] = *reinterpret_cast<const f4*>(p + 49 * dkp + (lq * dvp + col + 16 * c) * 4);
        x.ov[c] = p[49 * dkp + ((4 + lq) * dvp + col + 16 * c) * 4 + wave];
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // the loads are issued here and not where they are used
  };
  auto run = [&](Tile& x, int i) __attribute__((always_inline)) {
    f4 xk[CT], xq[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) xk[c] = xq[c] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          xk[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.tk[t][e], s[c][t][e], xk[c], 0, 0, 0);
          xq[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.qe[t][e], s[c][t][e], xq[c], 0, 0, 0);
        }
    f4(*pb)[2 * CT][64] = part[i & 1];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      pb[wave][2 * c][lane] = xk[c];
      pb[wave][2 * c + 1][lane] = xq[c];
    }
    __syncthreads();  // (the other buffer may still be read by slower waves, this one not: they are past the last barrier)
    const int tok = 16 * i + 4 * lq + wave;
    f4 u[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      f4 sum = pb[0][2 * c][lane];
      float os = reinterpret_cast<const float*>(&pb[0][2 * c + 1][lane])[wave];
#pragma unroll
      for (int v = 1; v < 4; ++v) {
        sum += pb[v][2 * c][lane];
        os += reinterpret_cast<const float*>(&pb[v][2 * c + 1][lane])[wave];
      }
      u[c] = x.tv[c] - sum;
      if (tok < n && col_on[c]) o[((row0 + tok) * a.heads + h) * a.vdim + col + 16 * c] = x.ov[c] + os;
#pragma unroll
      for (int t = 0; t < RT; ++t) s[c][t] *= x.gc[t];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c) s[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.ke[t][e], u[c][e], s[c][t], 0, 0, 0);
  };
  fetch(ta, 0);
  fetch(tb, 1);
  int i = 0;
  for (; i + 1 < nt; i += 2) {
    run(ta, i);
    fetch(ta, i + 2);
    run(tb, i + 1);
    fetch(tb, i + 3);
  }
  if (i < nt) run(ta, i);
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = base + 16 * t + 4 * lq + r;
        if (col_on[c] && d < a.dim) sp[(long long)d * a.vdim + 16 * c] = s[c][t][r];
      }
  if (y == 0) {  // the convolution inputs the next portion needs (their readers ran in the tile kernel)
    const int rep = a.heads / a.kv_heads, g = h / rep, qk = a.kv_heads * a.dim;
    const int keep = n < a.taps ? n : a.taps;
    const int own = a.vdim + (h % rep == 0 ? 2 * a.dim : 0);
    for (int idx = tid; idx < own; idx += 256) {
      const int c = idx < a.vdim ? 2 * qk + h * a.vdim + idx : idx < a.vdim + a.dim ? g * a.dim + idx - a.vdim : qk + g * a.dim + idx - a.vdim - a.dim;
      const T* p = proj + row0 * a.ldp + chan_col(a, c);
      for (int i = n - keep; i < n; ++i) ring[((long long)slot * a.taps + (pos0 + i) % a.taps) * a.channels + c] = p[i * a.ldp];
    }
  }
}

// Sixteen lanes of a load read 256 bytes in a row: as rows of tokens the coefficients were sixteen places, and the loads took a quarter of the time (us a layer,
// rows and now: 4 x 560 tokens of 32 heads 97 and 87, all of the delta rule for 1 x 2048 218 and 201, 64 x 20 246 and 226, 16 heads of 256 channels 4 x 300 131
// and 115; without any loads the first takes 81).  The figures below are from before.
// grid (heads, dvp / 16, portions).  What bounds a tile's step is what is read of it (25 KB for 128 key channels and 16 columns, from beyond the L2) and
// the fp32 matrix instructions (0.35 us); its serial chain is about as long.  Two column tiles a workgroup read half as much and leave half the
// workgroups.  Measured for 128 x 128, us of a layer's launches for portions, one tile a workgroup and two: 32 heads, 4 x 512 tokens 225, 204; 16 x 128
// 240, 220; 64 x 20 305, 281; 16 heads, 8 x 256 123, 111; with few workgroups (1 x 2048) the chain alone 133, 202.  For key sizes up to 64 two gain nothing (8 x 256
// tokens of 32 heads of 64: 99, 104), above 128 their registers leave one workgroup on a CU (16 heads of 256 x 128, 4 x 300: 144, 159).
// How many portions there are only the device knows, how long they are in the mean the host: with up to a tile for each there might be, they may be
// many of one tile, which wait for memory and want workgroups beside them (64 x 13: 147, and 165 where the registers are left to the compiler, 142
// here).  So WGS is the workgroups a CU holds: 0, one column tile each, as the registers allow; 3, two where they are more than two workgroups per CU
// (as many as that are dealt out unevenly when three find room: 4 x 256 tokens 128 against 122 by one); 2, two where they are more than one (at 513
// to 768 of one tile that costs 3 %: 3 x 683 226, 234).  The half of the grid that has nothing to do is the upper half of the columns: with every
// other column idle, 16 heads put all live workgroups on half of an XCD's engines.
template <typename T, int RT, int WGS>
__global__ __launch_bounds__(256, WGS == 3 ? 3 : 1) void delta_chain_kernel(const float* __restrict__ ws, float* __restrict__ o, const T* __restrict__ proj, T* __restrict__ ring,
                                                                            const int* __restrict__ seg_row, const int* __restrict__ seg_n, const int* __restrict__ seg_pos,
                                                                            const int* __restrict__ seg_slot, const int* __restrict__ seg_tile, int min_n, int dkp, int dvp, DeltaArgs a) {
  __shared__ __attribute__((aligned(16))) f4 part[2 * 4 * (WGS ? 4 : 2) * 64];
  const int n = seg_n[blockIdx.z];
  if (n == 0 || n < min_n) return;
  if constexpr (WGS > 0) {
    int live = 0;
    for (int i = threadIdx.x & 63; i - (int)(threadIdx.x & 63) < (int)gridDim.z; i += 64)
      live += __builtin_popcountll(__builtin_amdgcn_ballot_w64(i < (int)gridDim.z && seg_n[i] > 0 && seg_n[i] >= min_n));
    if (live * (int)(gridDim.x * gridDim.y) > (WGS == 3 ? 1024 : 512)) {
      if (blockIdx.y >= gridDim.y / 2) return;
      delta_chain<T, RT, 2, WGS == 3>(part, blockIdx.y, n, ws, o, proj, ring, seg_row, seg_pos, seg_slot, seg_tile, dkp, dvp, a);
      return;
    }
  }
  delta_chain<T, RT, 1, WGS == 3>(part, blockIdx.y, n, ws, o, proj, ring, seg_row, seg_pos, seg_slot, seg_tile, dkp, dvp, a);
}

}  // namespace

// What every entry point below takes (a plain struct, filled by the bindings)
struct KvdArgs {
  long long ldp, ldl;
  int q_off, k_off, v_off, b_off, z_off, gate_off;
  const float *conv_w, *a_log, *dt_bias, *o_norm;
  float* state;
  const int *tok_seq, *positions, *tok_kind, *tok_off;
  int heads, kv_heads, dim, vdim, taps, channels;
  float eps, out_scale;
  long long ldo; int o_off;
};

namespace {
DeltaArgs args_of(const KvdArgs& k) {
  return DeltaArgs{k.ldp, k.ldl, k.q_off, k.k_off, k.v_off, k.b_off, k.z_off, k.gate_off, k.conv_w, k.a_log, k.dt_bias, k.o_norm, k.state, k.tok_seq, k.positions, k.tok_kind, k.tok_off,
                   k.heads, k.kv_heads, k.dim, k.vdim, k.taps, k.channels, k.eps, k.out_scale, k.ldo, k.o_off};
}
bool bad(const KvdArgs& k) {
  return k.heads <= 0 || k.kv_heads <= 0 || k.heads % k.kv_heads || k.dim <= 0 || k.vdim <= 0 || k.taps < 1 || k.channels != 2 * k.kv_heads * k.dim + k.heads * k.vdim;
}
// rows of S per thread of the one-token kernel; 0: the head does not fit it
int step_rows(int dim, int vdim) {
  if ((vdim & 3) || vdim > 1024 || vdim < 4) return 0;
  const int nrg = 256 / (vdim >> 2), rows = (dim + nrg - 1) / nrg;
  if ((3 * dim + vdim + 2 * nrg * vdim) * 4 > 60000) return 0;
  return rows <= 4 ? 4 : rows <= 8 ? 8 : rows <= 16 ? 16 : rows <= 32 ? 32 : 0;
}
}  // namespace

extern "C" {

int kvd_step_rows(int dim, int vdim) { return step_rows(dim, vdim); }

// row_list: [n_rows] token rows that are alone in their sequence (-1 = unused)
int kvd_step(const KvdArgs* k, const void* proj, const void* low, void* ring, void* out, int f32, const int* row_list, int n_rows, hipStream_t s) {
  const int rows = bad(*k) ? 0 : step_rows(k->dim, k->vdim);
  if (n_rows <= 0 || rows == 0) return -1;
  const DeltaArgs a = args_of(*k);
  const size_t lds = (size_t)(3 * a.dim + a.vdim + 2 * (256 / (a.vdim >> 2)) * a.vdim) * 4;
  const dim3 grid(n_rows, a.heads);
  // Heads of up to 64 x 64 are one item a thread: asking for a second one, for nothing, made 61 rows of 16 such heads 10.4 us (9.95 without)
  const bool one_item = a.dim <= 64 && a.vdim <= 64;
#define KV_ST1(Tt, R, TP, E) hipLaunchKernelGGL((delta_step_kernel<Tt, R, TP, E>), grid, dim3(256), lds, s, row_list, (const Tt*)proj, (const Tt*)low, (Tt*)ring, (Tt*)out, a)
#define KV_STE(Tt, R, TP) do { if (R == 4 && one_item) KV_ST1(Tt, 4, TP, 1); else KV_ST1(Tt, R, TP, 2); } while (0)
#define KV_ST(Tt, R) do { if (a.taps == 4) KV_STE(Tt, R, 4); else if (a.taps == 3) KV_STE(Tt, R, 3); else if (a.taps == 2) KV_STE(Tt, R, 2); else KV_ST1(Tt, R, 0, 0); } while (0)
#define KV_ST2(R) do { if (f32) KV_ST(float, R); else KV_ST(bf16raw, R); } while (0)
  switch (rows) {
    case 4: KV_ST2(4); break;
    case 8: KV_ST2(8); break;
    case 16: KV_ST2(16); break;
    default: KV_ST2(32); break;
  }
#undef KV_ST2
#undef KV_ST
#undef KV_STE
#undef KV_ST1
  return (int)hipGetLastError();
}

int kvd_prep(const KvdArgs* k, const void* proj, const void* low, const void* ring, int f32, float* qn, float* kn, float* vv, float* dec, float* beta, int dimp, int min_kind, int T,
             hipStream_t s) {
  if (T <= 0 || bad(*k) || dimp < k->dim || (dimp & 7)) return -1;
  const DeltaArgs a = args_of(*k);
  const dim3 grid(T, (2 * a.kv_heads + 2 * a.heads + 3) / 4);
  if (f32) hipLaunchKernelGGL((delta_prep_kernel<float>), grid, dim3(256), 0, s, (const float*)proj, (const float*)low, (const float*)ring, qn, kn, vv, dec, beta, dimp, min_kind, a);
  else hipLaunchKernelGGL((delta_prep_kernel<bf16raw>), grid, dim3(256), 0, s, (const bf16raw*)proj, (const bf16raw*)low, (const bf16raw*)ring, qn, kn, vv, dec, beta, dimp, min_kind, a);
  return (int)hipGetLastError();
}

int kvd_scan(const float* qn, const float* kn, const float* vv, const float* dec, const float* beta, float* o, const int* segs, int n_segs, int min_n, int dimp, float* state, int heads,
             int kv_heads, int dim, int vdim, hipStream_t s) {
  if (n_segs <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || dim > 512 || dimp < dim || (dimp & 7) || vdim <= 0) return -1;
  const int *row = segs, *n = segs + n_segs, *pos = segs + 2 * n_segs, *slot = segs + 3 * n_segs;
#define KV_SC(RG)                                                                                                                                                      \
  hipLaunchKernelGGL((delta_scan_kernel<RG>), dim3((vdim + 4 * (64 / RG) - 1) / (4 * (64 / RG)), heads, n_segs), dim3(256), 0, s, qn, kn, vv, dec, beta, o, row, n, pos, slot, min_n, \
                     dimp, state, heads, kv_heads, dim, vdim)
  if (dim <= 32) KV_SC(4);
  else if (dim <= 64) KV_SC(8);
  else if (dim <= 128) KV_SC(16);
  else if (dim <= 256) KV_SC(32);
  else KV_SC(64);
#undef KV_SC
  return (int)hipGetLastError();
}

// padded sizes of the tile form (0: the key size is beyond it)
int kvd_tile_dkp(int dim) { return dim <= 64 ? 64 : dim <= 128 ? 128 : dim <= 256 ? 256 : 0; }
long long kvd_tile_floats(int dkp, int dvp) { return tile_floats(dkp, dvp); }

// tiles: int32 [4, tile_stride]: first row, tokens (0 = unused), first position, slot of up to 16 tokens, the first n_tiles in use;
// segs: int32 [5, n_segs]: ... and the portion's first tile; T: rows of the step.  ws: n_tiles * heads * kvd_tile_floats floats.
int kvd_tiles(const KvdArgs* k, const void* proj, const void* low, void* ring, int f32, const int* tiles, int tile_stride, int n_tiles, const int* segs, int n_segs, int min_n, int T, float* ws,
              float* o, hipStream_t s) {
  const int dkp = bad(*k) ? 0 : kvd_tile_dkp(k->dim);
  if (dkp == 0 || n_tiles <= 0 || n_tiles > tile_stride || n_segs <= 0) return -1;
  const DeltaArgs a = args_of(*k);
  const int dvp = (a.vdim + 15) / 16 * 16;
  const size_t lds = (size_t)(3 * 16 * (dkp + 4) + 16 * dvp + 8 * PAIRS + 640) * 4;
  if (lds > 160 * 1024 - 256) return -1;
  const int *tr = tiles, *tn = tiles + tile_stride, *tp = tiles + 2 * tile_stride, *ts = tiles + 3 * tile_stride;
  const int *row = segs, *n = segs + n_segs, *pos = segs + 2 * n_segs, *slot = segs + 3 * n_segs, *first = segs + 4 * n_segs;
  auto tiles_of = [&](auto of, auto taps, auto keys) {
    using Row = decltype(of);
    constexpr auto kernel = delta_tile_kernel<Row, decltype(taps)::value, decltype(keys)::value>;
    if (lds > 65536 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return -1;
    hipLaunchKernelGGL(kernel, dim3(a.heads, n_tiles), dim3(256), lds, s, (const Row*)proj, (const Row*)low, (const Row*)ring, ws, tr, tn, tp, ts, dvp, a);
    return (int)hipGetLastError();
  };
  auto of_keys = [&](auto of, auto taps) {
    return dkp == 64 ? tiles_of(of, taps, std::integral_constant<int, 64>{}) : dkp == 128 ? tiles_of(of, taps, std::integral_constant<int, 128>{}) : tiles_of(of, taps, std::integral_constant<int, 256>{});
  };
  auto of_taps = [&](auto of) {
    switch (a.taps) {
      case 4: return of_keys(of, std::integral_constant<int, 4>{});
      case 3: return of_keys(of, std::integral_constant<int, 3>{});
      case 2: return of_keys(of, std::integral_constant<int, 2>{});
      default: return of_keys(of, std::integral_constant<int, 0>{});
    }
  };
  const int rc = f32 ? of_taps(float{}) : of_taps(bf16raw{});
  if (rc) return rc;
  const dim3 grid(a.heads, dvp / 16, n_segs);
#define KV_CH(Tt, RT, WGS) hipLaunchKernelGGL((delta_chain_kernel<Tt, RT, WGS>), grid, dim3(256), 0, s, ws, o, (const Tt*)proj, (Tt*)ring, row, n, pos, slot, first, min_n, dkp, dvp, a)
#define KV_CH2(RT, WGS) do { if (f32) KV_CH(float, RT, WGS); else KV_CH(bf16raw, RT, WGS); } while (0)
  if (dkp == 64) KV_CH2(1, 0);
  else if (dkp == 256) KV_CH2(4, 0);
  else if (dvp % 32) KV_CH2(2, 0);
  else if (T <= 16 * (long long)n_segs) KV_CH2(2, 3);
  else KV_CH2(2, 2);
#undef KV_CH2
#undef KV_CH
  return (int)hipGetLastError();
}

int kvd_out(const KvdArgs* k, const float* o, const void* low, void* out, int f32, int min_kind, int T, hipStream_t s) {
  if (T <= 0 || bad(*k)) return -1;
  const DeltaArgs a = args_of(*k);
#define KV_OUT(LPR)                                                                                                                                        \
  do {                                                                                                                                                      \
    const dim3 grid(T, (a.heads + 256 / LPR - 1) / (256 / LPR));                                                                                            \
    if (f32) hipLaunchKernelGGL((delta_out_kernel<float, LPR>), grid, dim3(256), 0, s, o, (const float*)low, (float*)out, min_kind, a);                      \
    else hipLaunchKernelGGL((delta_out_kernel<bf16raw, LPR>), grid, dim3(256), 0, s, o, (const bf16raw*)low, (bf16raw*)out, min_kind, a);                    \
  } while (0)
  if (a.vdim <= 32) KV_OUT(8);
  else if (a.vdim <= 64) KV_OUT(16);
  else KV_OUT(32);
#undef KV_OUT
  return (int)hipGetLastError();
}

int kvd_conv_tail(const KvdArgs* k, const void* proj, void* ring, int f32, const int* segs, int n_segs, int min_n, hipStream_t s) {
  if (n_segs <= 0 || bad(*k)) return -1;
  const DeltaArgs a = args_of(*k);
  const int *row = segs, *n = segs + n_segs, *pos = segs + 2 * n_segs, *slot = segs + 3 * n_segs;
  const dim3 grid((a.channels + 255) / 256, n_segs);
  if (f32) hipLaunchKernelGGL((conv_tail_kernel<float>), grid, dim3(256), 0, s, (const float*)proj, (float*)ring, row, n, pos, slot, min_n, a);
  else hipLaunchKernelGGL((conv_tail_kernel<bf16raw>), grid, dim3(256), 0, s, (const bf16raw*)proj, (bf16raw*)ring, row, n, pos, slot, min_n, a);
  return (int)hipGetLastError();
}

}  // extern "C"
