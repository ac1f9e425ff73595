// What paged_attention_kernel and the rows of prompt_attention_64_kernel do for row t and kv head g: included into both.  Which products are fused with sums is
// stated (those of one expression): left to the compiler it was another choice in each kernel, 43 outputs of a million one rounding apart, which in rows
// that are rounded to e4m3 moves codes, and a step's results by 4 % of their norm.  Included, since as an inlined function the kernels of heads of 128 with a bf16
// cache hold 20 registers more and take longer (40 rows of 3000 tokens, groups of four: 52.9 and 58.7 us; of eight: 77.0 and 84.7).
{
#pragma clang fp contract(on)
  constexpr int BS = 16, NT = 64 * NWAVE;
  constexpr int DQ = HD / 4;   // dims of the QK dot owned by a lane
  constexpr int NV = DQ / 8;   // 16-byte K loads per lane
  constexpr int DP = HD / 16;  // output dims owned by a lane in PV
  constexpr bool RAWV = KV8 && HD == 128;
  static_assert(HD == 64 || HD == 128, "head_dim 64 or 128");
  __shared__ float p_lds[NWAVE][REP][BS];    // per-wave probabilities of the current block
  __shared__ float m_lds[NWAVE][REP], l_lds[NWAVE][REP];
  __shared__ float o_lds[NWAVE][REP][HD];
  // wave index in a scalar register: the block-table reads below become scalar loads, which do
  // not queue behind (and so do not drain) the K/V loads in flight
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int ctx = ctx_lens[t];
  float v_scale = 1.f;
  if constexpr (KV8) {  // stored K / V are x / scale: the K scale folds into the score scale, the V scale into the output
    scale_log2e *= kv_scale[g];
    v_scale = kv_scale[nkv + g];
  }
  unsigned short* orow = out + (long long)t * nh * HD + (long long)g * REP * HD;
  if (ctx <= 0) {  // 0: padding token, zero output; negative: a prompt-chunk row that the tiled kernel writes
    if (ctx == 0)
      for (int i = tid; i < REP * HD; i += NT) orow[i] = 0;
    return;
  }
  const int* bt = block_tables + (long long)tok_seq[t] * max_blocks_per_seq;
  const int n_blocks = (ctx + BS - 1) / BS;

  // Each wave keeps two K/V blocks in flight beyond the one it computes on, in three register stages whose roles
  // rotate through a loop unrolled by three (no register copies, and no copy that would wait for the newest loads).
  // The loads are unconditional — past the sequence's end the last block is read again and never used — so the
  // number of loads in flight is the same on every path and a stage is waited for by count (two stages stay in
  // flight), not by draining the queue.
  // MF (e4m3 cache, head width 128): the scores come from the matrix cores — a K fragment lane is (key = lane & 15,
  // dims 32 (lane >> 4) ..), the A operand of v_mfma_f32_16x16x32_bf16 as it is loaded, against q as the B operand
  // (column = head); the vector ALU keeps the softmax and P V
  constexpr bool MF = HD == 128;
  const int qk_tok = MF ? (lane & 15) : (lane >> 2), qk_c = MF ? (lane >> 4) : (lane & 3);
  const int pv_tg = lane >> 4, pv_dv = lane & 15;
  typedef __attribute__((ext_vector_type(DP))) unsigned short vrow_t;  // 16 B (HD 128) or 8 B (HD 64)
  typedef PAStage<HD, KV8> stage_t;
  const int last_b = n_blocks - 1;
  auto entry = [&](int b) __attribute__((always_inline)) {
    return bt[b < last_b ? b : last_b];
  };
  // block bases in scalar registers (the block id is wave-uniform), per-lane offsets fixed for the whole walk: the
  // loads need no vector address arithmetic, whose temporaries would otherwise share registers with a stage in flight
  // and wait for it
  const unsigned koff = stage_t::k_off(qk_tok, qk_c), voff = stage_t::v_off(pv_tg, pv_dv);
  constexpr int ESZ = KV8 ? 1 : 2;
  auto issue = [&](stage_t& st, int blk) __attribute__((always_inline)) {
    const long long base = ((long long)__builtin_amdgcn_readfirstlane(blk) * nkv + g) * (BS * HD * ESZ);
    st.load_at(reinterpret_cast<const char*>(k_cache) + base, reinterpret_cast<const char*>(v_cache) + base, koff, voff);
  };
  stage_t s0, s1, s2;
  issue(s0, entry(wave));
  issue(s1, entry(wave + NWAVE));
  // this lane's DQ-dim slice of the REP query heads, kept as packed bf16 pairs for
  // v_dot2_f32_bf16 (half the registers and multiplies of an fp32 copy, no unpacking of K)
  bf16x2 qp[MF ? 1 : REP][DQ / 2];
  typedef __attribute__((ext_vector_type(8))) __bf16 mf_ab;
  typedef __attribute__((ext_vector_type(4))) float mf_cd;
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  mf_ab qb[4];             // MF: q of head (lane & 15), dims 32 qk_c + 8 v .. + 8 (zero for columns past the group's heads)
  const int col = lane & 15;
  if constexpr (MF) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      bf16x8 raw = (bf16x8){0, 0, 0, 0, 0, 0, 0, 0};
      if (col < REP) raw = *reinterpret_cast<const bf16x8*>(q + (long long)t * q_row_stride + (long long)(g * REP + col) * HD + qk_c * 32 + v * 8);
      qb[v] = __builtin_bit_cast(mf_ab, raw);
    }
  } else {
    const unsigned short* qrow = q + (long long)t * q_row_stride + (long long)g * REP * HD + qk_c * DQ;
#pragma unroll
    for (int h = 0; h < REP; ++h)
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const bf16x2x4 a = __builtin_bit_cast(bf16x2x4, *reinterpret_cast<const bf16x8*>(qrow + h * HD + v * 8));
#pragma unroll
        for (int j = 0; j < 4; ++j) qp[h][v * 4 + j] = a.p[j];
      }
  }
  float m_own = -1e30f;    // MF: running maximum of this lane's own head (equals m_run[col])
  float acc[REP][DP];
  float m_run[REP], l_run[REP];
#pragma unroll
  for (int h = 0; h < REP; ++h) {
    m_run[h] = -1e30f; l_run[h] = 0.f;
#pragma unroll
    for (int j = 0; j < DP; ++j) acc[h][j] = 0.f;
  }

  // one block: scores, online softmax, P V on the stage that holds block b
  auto block = [&](const stage_t& st, int b) __attribute__((always_inline)) {
    bf16x8 kv[NV];
    vrow_t vv[4];
    float vf[RAWV ? 4 : 1][8];  // e4m3 cache, head width 128: V as fp32, in the lane's own token order (KVStage<true>::unpack_f32)
    if constexpr (RAWV) st.unpack_f32(kv, vf, pv_dv);
    else st.unpack(kv, vv, pv_dv);
    if constexpr (MF) {
      mf_cd sc = (mf_cd){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int v = 0; v < 4; ++v) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mf_ab, kv[v]), qb[v], sc, 0, 0, 0);
      // lane (head col, quarter qk_c): sc[e] = q_col . k of key 4 qk_c + e of the block
      float mx = -1e30f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sc[e] = (col < REP && b * BS + 4 * qk_c + e < ctx) ? sc[e] * scale_log2e : -1e30f;
        mx = fmaxf(mx, sc[e]);
      }
      mx = quad_rows_max(mx);  // over the four quarters: the block's maximum for head col
      const float m_own_new = fmaxf(m_own, mx);
      mf_cd pe;
      float ps = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pe[e] = __builtin_amdgcn_exp2f(sc[e] - m_own_new);
        ps += pe[e];
      }
      m_own = m_own_new;
      ps = quad_rows_sum(ps);
      if (col < REP) *reinterpret_cast<mf_cd*>(&p_lds[wave][col][4 * qk_c]) = pe;
#pragma unroll
      for (int h = 0; h < REP; ++h) {  // (head h's maximum and sum sit in lane h: scalar reads)
        const float m_new = fmaxf(m_run[h], lane_value(mx, h));
        const float corr = __builtin_amdgcn_exp2f(m_run[h] - m_new);
        l_run[h] = l_run[h] * corr + lane_value(ps, h);
        m_run[h] = m_new;
#pragma unroll
        for (int j = 0; j < DP; ++j) acc[h][j] *= corr;
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): p_lds visible to the wave
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tok = RAWV ? pv_tg + 4 * (i ^ (pv_dv & 1)) : pv_tg + 4 * i;
#pragma unroll
        for (int h = 0; h < REP; ++h) {
          const float p = p_lds[wave][h][tok];
#pragma unroll
          for (int j = 0; j < DP; ++j) {
            if constexpr (RAWV) acc[h][j] += p * vf[i][j];
            else acc[h][j] += p * bf2f(vv[i][j]);
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
      return;
    }
    // ---- QK^T
    float s[REP];
#pragma unroll
    for (int h = 0; h < REP; ++h) {
      float d = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const bf16x2x4 kw = __builtin_bit_cast(bf16x2x4, kv[v]);
#pragma unroll
        for (int j = 0; j < 4; ++j) d = __builtin_amdgcn_fdot2_f32_bf16(qp[h][v * 4 + j], kw.p[j], d, false);
      }
      d += dpp_f32<0xB1>(d);  // the 4 dim chunks of a key sit in one quad: quad swaps in registers
      d += dpp_f32<0x4E>(d);
      s[h] = (b * BS + qk_tok < ctx) ? d * scale_log2e : -1e30f;
    }
    // ---- online softmax over the block's 16 tokens (token index lives in lane bits 2..5)
#pragma unroll
    for (int h = 0; h < REP; ++h) {
      // quads hold equal values: half-row and row mirror fold the 4 quads of a row in
      // registers, only the two cross-row steps go through the LDS crossbar
      float mx = s[h];
      mx = fmaxf(mx, dpp_f32<0x141>(mx));
      mx = fmaxf(mx, dpp_f32<0x140>(mx));
      mx = quad_rows_max(mx);
      const float m_new = fmaxf(m_run[h], mx);
      const float p = __builtin_amdgcn_exp2f(s[h] - m_new);
      float ps = p;
      ps += dpp_f32<0x141>(ps);
      ps += dpp_f32<0x140>(ps);
      ps = quad_rows_sum(ps);
      const float corr = __builtin_amdgcn_exp2f(m_run[h] - m_new);
      l_run[h] = l_run[h] * corr + ps;
      m_run[h] = m_new;
#pragma unroll
      for (int j = 0; j < DP; ++j) acc[h][j] *= corr;
      if (qk_c == 0) p_lds[wave][h][qk_tok] = p;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): p_lds visible to the wave (single wave: no barrier needed)
    __builtin_amdgcn_wave_barrier();
    // ---- PV
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tok = RAWV ? pv_tg + 4 * (i ^ (pv_dv & 1)) : pv_tg + 4 * i;
#pragma unroll
      for (int h = 0; h < REP; ++h) {
        const float p = p_lds[wave][h][tok];
#pragma unroll
        for (int j = 0; j < DP; ++j) {
          if constexpr (RAWV) acc[h][j] += p * vf[i][j];
          else acc[h][j] += p * bf2f(vv[i][j]);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  };

  for (int b = wave; b < n_blocks; b += 3 * NWAVE) {
    // the round's three block-table entries: scalar loads issued together (nothing about them is carried around the
    // loop — a carried id ends up in a vector register that doubles as a load destination, and waiting for it drains the queue)
    const int e2 = entry(b + 2 * NWAVE), e3 = entry(b + 3 * NWAVE), e4 = entry(b + 4 * NWAVE);
    issue(s2, e2);
    block(s0, b);
    if (b + NWAVE >= n_blocks) break;
    issue(s0, e3);
    block(s1, b + NWAVE);
    if (b + 2 * NWAVE >= n_blocks) break;
    issue(s1, e4);
    block(s2, b + 2 * NWAVE);
  }
  // ---- sum the 4 token groups inside the wave (lanes l, l^16, l^32, ...)
#pragma unroll
  for (int h = 0; h < REP; ++h)
#pragma unroll
    for (int j = 0; j < DP; ++j) {
      float v = acc[h][j];
      v = lanes::meet<16>(v, lanes::Sum{});
      v = lanes::meet<32>(v, lanes::Sum{});
      acc[h][j] = v;
    }
  if (pv_tg == 0) {
#pragma unroll
    for (int h = 0; h < REP; ++h)
#pragma unroll
      for (int j = 0; j < DP; ++j) o_lds[wave][h][pv_dv * DP + j] = acc[h][j];
  }
  if (lane == 0) {
#pragma unroll
    for (int h = 0; h < REP; ++h) { m_lds[wave][h] = m_run[h]; l_lds[wave][h] = l_run[h]; }
  }
  __syncthreads();
  // ---- merge the waves; thread i handles output element i (REP*HD elements)
  for (int i = tid; i < REP * HD; i += NT) {
    const int h = i / HD, d = i % HD;
    float m = m_lds[0][h];
#pragma unroll
    for (int w = 1; w < NWAVE; ++w) m = fmaxf(m, m_lds[w][h]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < NWAVE; ++w) {
      const float c = __builtin_amdgcn_exp2f(m_lds[w][h] - m);
      num += o_lds[w][h][d] * c;
      den += l_lds[w][h] * c;
    }
    orow[i] = f2bf(den > 0.f ? num / den * v_scale : 0.f);
  }
}
