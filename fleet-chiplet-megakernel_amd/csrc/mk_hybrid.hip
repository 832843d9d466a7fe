// Selective scan and expert feed-forwards (part of the persistent kernel, included by mk_kernel.hip behind mk_flex.hip and
// mk_mix.hip, whose conventions it keeps: sizes and constants are descriptor fields, E is the type of activations and weights,
// everything named in 32 bits is 32-bit in both builds).
//   * stage_hy_conv     causal convolution per channel and silu, the inputs before the portion come from the request's slot;
//   * stage_hy_scan     S' = exp(dt A) S + dt x B, y = (S' C + D x) silu(z), state and convolution tail per request;
//   * stage_hy_route    softmax over experts, the largest few, their shares;
//   * stage_hy_experts  gated or plain linears of the chosen experts over their tokens, and of a shared expert over all tokens.
// (The step sizes dt and the router logits are forms of stage_mx_head_linear, the weighted sum over a token's experts is part of
// the norm behind it.)

__device__ __forceinline__ float hy_silu(uint16_t, float z) { return z * mx_sigmoid((uint16_t)0, z); }
__device__ __forceinline__ float hy_silu(float, float z) { return z / (1.f + expf(-z)); }

// ----------------------------------------------------------------------------- convolution
// out[t, c] = silu(b[c] + sum_j w[j][c] x[t - (taps - 1) + j, c]); st.n channels (a multiple of 4), x = in[t, cols[0] + c], w fp32
// [taps][n].  Tail of a slot: [taps - 1][n], row r the input at position p0 - (taps - 1) + r; positions before the first count as
// zero whatever the slot holds.  The scan stage writes the new tail, so that every token of a portion is independent here.
template <typename E>
__device__ __forceinline__ void stage_hy_conv(CStage &st, Ctx &c, const MkRuntime &rt, int M) {
  barrier_wait(c);
  const int n = st.n, n4 = n / 4, taps = st.taps, per = (n4 + MK_THREADS - 1) / MK_THREADS;
  const float *w = (const float *)st.norm_w;
  for (int i = mx_spread(c); i < M * per; i += c.G) {
    const int t = i / per, q = (i - t * per) * MK_THREADS + c.tid;
    if (q >= n4) continue;
    const int t0 = __builtin_amdgcn_readfirstlane(c.sh_tok[2 * MK_MAX_TOKENS + t]), pos = __builtin_amdgcn_readfirstlane(c.sh_tok[t]);
    const int slot = __builtin_amdgcn_readfirstlane(rt.state_ids[__builtin_amdgcn_readfirstlane(c.sh_tok[MK_MAX_TOKENS + t])]);
    const E *x = (const E *)st.in + st.cols[0] + 4 * q, *tail = (const E *)st.tail + (size_t)slot * (taps - 1) * n + 4 * q;
    f32x4 acc = *(const f32x4 *)(st.in_bias + 4 * q);
    for (int j0 = 0; j0 < taps; j0 += 4) {
      f32x4 v[4], g[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int tap = min(j0 + j, taps - 1), back = taps - 1 - tap, k = back - (t - t0);  // k > 0: k positions before the portion
        const E *src = k > 0 ? tail + (size_t)(taps - 1 - k) * n : x + (size_t)(t - back) * st.ld_in;
        v[j] = fx_ldc_quad(src);
        g[j] = *(const f32x4 *)(w + (size_t)tap * n + 4 * q);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const bool on = j0 + j < taps && taps - 1 - (j0 + j) <= pos;
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] = on ? fmaf(v[j][e], g[j][e], acc[e]) : acc[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; e++) acc[e] = hy_silu(E(), acc[e]);
    fx_stc_quad((E *)st.out + (size_t)t * st.ld_out + 4 * q, acc);
  }
  c.wrote_through = true;
}

// ----------------------------------------------------------------------------- selective scan
// L = 4, 8 or 16 lanes hold the states of a channel, Q quads each: lane j of them states 4 (i L + j) .. + 3, i < Q, so the sum over states stays
// among L neighbours.  A lane works on CH channels at a time.  A workgroup takes 256 CH / L channels of one request and walks its
// tokens, TB at a time; the rows of the next TB (or of the next unit, with its state) are in flight meanwhile.  A lane finishes (gate,
// store) every L-th output.  State: fp32 [slot][channel][states rounded up to 4], zero where a request begins.  dt: fp32
// rows (in2), x: conv output rows (q_ws), B and C: columns cols[1], cols[2] of in3, z: column cols[3] of in.
__device__ __forceinline__ float hy_lanes_sum(float v, int L) {
  v += dpp_f32<0xB1>(v);  // quad_perm [1,0,3,2]
  v += dpp_f32<0x4E>(v);  // quad_perm [2,3,0,1]
  v += L >= 8 ? dpp_f32<0x141>(v) : 0.f;   // row_half_mirror
  v += L >= 16 ? dpp_f32<0x140>(v) : 0.f;  // row_mirror
  return v;
}
template <typename E, int Q, int TB, int CH>
__device__ __forceinline__ void stage_hy_scan_t(CStage &st, Ctx &c, const MkRuntime &rt, int M, int lg2) {
  constexpr int KK = (TB * CH + 3) / 4;  // (outputs a lane finishes, with the fewest lanes per channel)
  const int L = 1 << lg2, GW = 64 >> lg2, CW = MK_WAVES * GW * CH;
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & (L - 1);
  const int n = st.n, Np = (st.states + 3) / 4 * 4, nblk = (n + CW - 1) / CW;
  const MxDeltaUnits us = mx_delta_units(c, M);
  const int n_units = us.nreq * nblk;
  const E *in = (const E *)st.in, *xc = (const E *)st.q_ws, *bc = (const E *)st.in3;
  const float *dtr = (const float *)st.in2;
  struct Unit {
    int ch0, t0, n, p0, slot;
  };
  auto unit = [&](int u) {
    Unit a;
    const int ri = u / nblk;
    a.ch0 = (u - ri * nblk) * CW + wave * GW * CH + (lane >> lg2);
    a.t0 = (int)__ffsll(__ballot(us.first && us.rank_of == ri)) - 1;
    a.n = wave_bcast(us.my_n, a.t0);
    a.p0 = __builtin_amdgcn_readfirstlane(c.sh_tok[a.t0]);
    a.slot = __builtin_amdgcn_readfirstlane(rt.state_ids[__builtin_amdgcn_readfirstlane(c.sh_tok[MK_MAX_TOKENS + a.t0])]);
    return a;
  };
  auto channel = [&](const Unit &a, int h) { return min(a.ch0 + h * GW, n - 1); };  // (behind the last: computed, not stored)
  auto real = [&](const Unit &a, int h) { return a.ch0 + h * GW < n; };
  int at[Q];
  bool on[Q];
#pragma unroll
  for (int i = 0; i < Q; i++) {
    on[i] = 4 * (i * L + j) < Np;
    at[i] = min(4 * (i * L + j), Np - 4);
  }
  auto state_of = [&](const Unit &a, int h) { return (float *)st.k_cache + ((size_t)a.slot * n + channel(a, h)) * Np; };
  auto load_state = [&](const Unit &a, f32x4 (&S)[CH][Q]) {
#pragma unroll
    for (int h = 0; h < CH; h++)
#pragma unroll
      for (int i = 0; i < Q; i++) S[h][i] = __builtin_nontemporal_load((const f32x4 *)(state_of(a, h) + at[i]));
  };
  struct Rows {
    f32x4 B[TB][Q], C[TB][Q];
    float dt[TB][CH], x[TB][CH], z[KK];
  };
  auto load_rows = [&](const Unit &a, int tb, Rows &r) {
#pragma unroll
    for (int t = 0; t < TB; t++) {
      const size_t tok = a.t0 + min(tb + t, a.n - 1);
#pragma unroll
      for (int i = 0; i < Q; i++) {
        r.B[t][i] = fx_ldc_quad(bc + tok * st.ld_in3 + st.cols[1] + at[i]);
        r.C[t][i] = fx_ldc_quad(bc + tok * st.ld_in3 + st.cols[2] + at[i]);
      }
#pragma unroll
      for (int h = 0; h < CH; h++) {
        r.dt[t][h] = ldc_f32(dtr + tok * st.ld_in2 + channel(a, h));
        r.x[t][h] = fx_ldc(xc + tok * st.ld_qws + channel(a, h));
      }
    }
#pragma unroll
    for (int k = 0; k < KK; k++)
      if (k == 0 || L == 4) r.z[k] = fx_ldc(in + (size_t)(a.t0 + min(tb + (k * L + j) / CH, a.n - 1)) * st.ld_in + st.cols[3] + channel(a, (k * L + j) % CH));
  };
  // The convolution's last inputs: the portion's, and before them what is left of the old ones.  Few taps: a lane per row, read with
  // the unit's rows and written at its end; more: in ascending order by one thread (a row is read before it is written).
  const int keep = st.taps - 1;
  auto load_tail = [&](const Unit &a, E (&v)[CH]) {
    const int i = a.n - keep + j;
#pragma unroll
    for (int h = 0; h < CH; h++) {
      const E *old = (const E *)st.tail + ((size_t)a.slot * max(keep, 1) + min(j + a.n, max(keep, 1) - 1)) * n + channel(a, h);
      v[h] = fx_round<E>(fx_ldc(i >= 0 ? in + (size_t)(a.t0 + min(i, a.n - 1)) * st.ld_in + st.cols[0] + channel(a, h) : old));
    }
  };
  f32x4 A[CH][Q];
  float D[CH];
  auto load_rates = [&](const Unit &a) {
#pragma unroll
    for (int h = 0; h < CH; h++) {
#pragma unroll
      for (int i = 0; i < Q; i++) A[h][i] = *(const f32x4 *)(st.a_tab + (size_t)channel(a, h) * Np + at[i]);
      D[h] = st.d_tab[channel(a, h)];
    }
  };
  const int u0 = mx_spread(c);
  f32x4 S[CH][Q];
  Unit a{};
  // earlier iterations wrote the state: the first unit's is requested before the barrier is awaited
  const bool early = u0 < n_units && wave != 0;
  if (u0 < n_units) a = unit(u0);
  if (early) {
    load_state(a, S);
    load_rates(a);
  }
  barrier_wait(c);
  if (u0 < n_units && !early) {
    load_state(a, S);
    load_rates(a);
  }
  Rows r;
  E tail[CH];
  if (u0 < n_units) {
    load_rows(a, 0, r);
    load_tail(a, tail);
  }
  for (int u = u0; u < n_units; u += c.G) {
    const Unit nx = u + c.G < n_units ? unit(u + c.G) : a;
    f32x4 Sn[CH][Q];
    E tail_n[CH];
    load_state(nx, Sn);
    load_tail(nx, tail_n);
#pragma unroll
    for (int h = 0; h < CH; h++)
#pragma unroll
      for (int i = 0; i < Q; i++)
        if (!on[i] || a.p0 == 0) S[h][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int tb = 0; tb < a.n; tb += TB) {
      Rows rn;
      const bool more = tb + TB < a.n;
      load_rows(more ? a : nx, more ? tb + TB : 0, rn);
      float y[KK];
      static_assert(TB * CH <= 8, "with more than four lanes per channel a lane finishes one output");
#pragma unroll
      for (int t = 0; t < TB; t++) {
        if (TB > 1 && tb + t >= a.n) break;
#pragma unroll
        for (int h = 0; h < CH; h++) {
          const float dx = r.dt[t][h] * r.x[t][h];
          float s = 0.f;
#pragma unroll
          for (int i = 0; i < Q; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
              S[h][i][e] = fmaf(fx_exp2(E(), r.dt[t][h] * A[h][i][e]), S[h][i][e], on[i] ? dx * r.B[t][i][e] : 0.f);
              s = fmaf(S[h][i][e], on[i] ? r.C[t][i][e] : 0.f, s);
            }
          s = hy_lanes_sum(s, L) + D[h] * r.x[t][h];
          const int e = t * CH + h;
          if ((e & (L - 1)) == j) {
            if (e >= 4 && L == 4) y[e / 4] = s;
            else y[0] = s;
          }
        }
      }
#pragma unroll
      for (int k = 0; k < KK; k++) {
        const int t = (k * L + j) / CH, h = (k * L + j) % CH;
        if ((k == 0 || L == 4) && t < TB && tb + t < a.n && real(a, h)) fx_stc((E *)st.out + (size_t)(a.t0 + tb + t) * st.ld_out + channel(a, h), fx_round<E>(y[k] * hy_silu(E(), r.z[k])));
      }
      r = rn;
    }
#pragma unroll
    for (int h = 0; h < CH; h++) {
      if (!real(a, h)) continue;
#pragma unroll
      for (int i = 0; i < Q; i++)
        if (on[i]) fx_stc_quad(state_of(a, h) + at[i], S[h][i]);
    }
    if (keep <= L) {
#pragma unroll
      for (int h = 0; h < CH; h++)
        if (j < keep && real(a, h)) fx_stc((E *)st.tail + ((size_t)a.slot * keep + j) * n + channel(a, h), tail[h]);
    } else if (j == 0) {
      for (int h = 0; h < CH; h++) {
        if (!real(a, h)) continue;
        E *rows = (E *)st.tail + (size_t)a.slot * keep * n + channel(a, h);
        for (int k = 0; k < keep; k++) {
          const int i = a.n - keep + k;
          fx_stc(rows + (size_t)k * n, fx_round<E>(i >= 0 ? fx_ldc(in + (size_t)(a.t0 + i) * st.ld_in + st.cols[0] + channel(a, h)) : fx_ldc(rows + (size_t)(k + a.n) * n)));
        }
      }
    }
    if (nx.ch0 != a.ch0) load_rates(nx);
    a = nx;
#pragma unroll
    for (int h = 0; h < CH; h++) {
#pragma unroll
      for (int i = 0; i < Q; i++) S[h][i] = Sn[h][i];
      tail[h] = tail_n[h];
    }
  }
  c.wrote_through = true;
}
template <typename E>
__device__ __forceinline__ void stage_hy_scan(CStage &st, Ctx &c, const MkRuntime &rt, int M, bool single) {
  const int lg2 = st.states <= 16 ? 2 : st.states <= 32 ? 3 : 4;
  // single tokens of many requests: eight channels per lane, so that a workgroup has enough in flight
  const bool many = single && (((long long)M * st.n) << lg2) >= 4ll * c.G * MK_THREADS;
  if (st.states <= 64) {
    if (many) stage_hy_scan_t<E, 1, 1, 8>(st, c, rt, M, lg2);
    else if (single) stage_hy_scan_t<E, 1, 1, 1>(st, c, rt, M, lg2);
    else stage_hy_scan_t<E, 1, 8, 1>(st, c, rt, M, lg2);
  } else {
    if (single) stage_hy_scan_t<E, 4, 1, 1>(st, c, rt, M, lg2);
    else stage_hy_scan_t<E, 4, 2, 1>(st, c, rt, M, lg2);
  }
}

// ----------------------------------------------------------------------------- routing
// One wavefront, one token: z fp32 [experts (+ 1: the shared expert's gate)].  Lane s < topk ends up with the s-th choice (ties: the
// lower index) and its share, lane topk with sigmoid of the gate.
// With MK_F_GROUPS (dual kernels): scores are sigmoids, choices are made on score + correction among the experts of the best groups, a
// group's worth being the sum of its two largest; the shares are choice_scale times the scores, the shared expert's is 1.  `scr`: 2 KB
// of LDS of the wavefront.
#if MK_HAVE_DUAL
__device__ __forceinline__ void hy_route_groups(CStage &st, const float *z, int lane, float &w, int &id, float *scr) {
  const int E = st.num_experts, count = st.groups, size = E / count;
  float s[4], p[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int e = q * 64 + lane, ec = min(e, E - 1);
    const float zv = ldc_f32(z + ec), b = st.choice_bias[ec];
    s[q] = 1.f / (1.f + expf(-zv));
    p[q] = e < E ? s[q] + b : -3.0e38f;
    scr[e] = p[q];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (count > 1) {
    for (int g = lane; g < count; g += 64) {
      float a = -3.0e38f, b = -3.0e38f;
      for (int i = 0; i < size; i++) {
        const float v = scr[g * size + i];
        b = fmaxf(b, fminf(a, v));
        a = fmaxf(a, v);
      }
      scr[256 + g] = size > 1 ? a + b : a;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (q * 64 >= E) continue;
      const int g = min(q * 64 + lane, E - 1) / size;
      const float mine = scr[256 + g];
      int better = 0;
      for (int i = 0; i < count; i++) {
        const float v = scr[256 + i];
        better += v > mine || (v == mine && i < g);
      }
      if (better >= st.groups_keep) p[q] = -3.0e38f;
    }
  }
  w = 0.f;
  id = 0;
  for (int k = 0; k < st.topk; k++) {
    float bv;
    int be;
    wave_pick(p, k, bv, be);
    const float sv = lane_f32(be < 64 ? s[0] : be < 128 ? s[1] : be < 192 ? s[2] : s[3], be & 63);
    if (lane == k) {
      w = sv * st.choice_scale;
      id = be;
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (q * 64 + lane == be) p[q] = -3.4e38f;
  }
  if (lane == st.topk) w = 1.f;
}
#endif
__device__ __forceinline__ void hy_route_wave(CStage &st, const float *z, int lane, float &w, int &id, float *scr) {
#if MK_HAVE_DUAL
  if (st.flags & MK_F_GROUPS) {
    hy_route_groups(st, z, lane, w, id, scr);
    return;
  }
#endif
  const int E = st.num_experts;
  float p[4], mx = -3.0e38f;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    p[q] = q * 64 + lane < E ? ldc_f32(z + q * 64 + lane) : -3.0e38f;
    mx = fmaxf(mx, p[q]);
  }
  const float g = st.w_shared ? ldc_f32(z + E) : 0.f;
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    p[q] = q * 64 + lane < E ? expf(p[q] - mx) : 0.f;
    sum += p[q];
  }
  sum = wave_sum(sum);
#pragma unroll
  for (int q = 0; q < 4; q++) p[q] = q * 64 + lane < E ? p[q] / sum : -1.f;
  float tot = 0.f;
  w = 0.f;
  id = 0;
  for (int s = 0; s < st.topk; s++) {
    float bv;
    int be;
    wave_pick(p, s, bv, be);
    tot += bv;
    if (lane == s) {
      w = bv;
      id = be;
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (q * 64 + lane == be) p[q] = -1.f;
  }
  w /= tot + 1e-20f;
  if (lane == st.topk) w = 1.f / (1.f + expf(-g));
}
__device__ __forceinline__ void hy_route_store(CStage &st, int t, int lane, float w, int id) {
  if (lane < st.topk) stc_i32(st.ids + (size_t)t * st.topk + lane, id);
  if (lane < st.topk + (st.w_shared ? 1 : 0)) stc_f32((float *)st.slot_w + (size_t)t * st.ld_slot_w + lane, w);
}
// (iterations of several tokens; a single token is routed by the expert stage itself)
__device__ __forceinline__ void stage_hy_route(CStage &st, Ctx &c, int M, char *smem) {
  barrier_wait(c);
  const int lane = c.tid & 63, wave = __builtin_amdgcn_readfirstlane(c.tid >> 6);
  for (int t = mx_wave_item(c, wave); t < M; t += c.G * MK_WAVES) {
    float w;
    int id;
    hy_route_wave(st, (const float *)st.moe_logits + (size_t)t * st.ld_logits, lane, w, id, (float *)smem + wave * 512);
    hy_route_store(st, t, lane, w, id);
  }
  c.wrote_through = true;
}

// ----------------------------------------------------------------------------- experts
// Weights of an expert are operand tiles (see stage_mx_head_linear); a unit is a pair of 16-row tiles of one expert over at most 16 of
// the tokens that visit it.  MK_F_SILU: the pair is gate and up of the same 16 outputs, out = silu(gate) up.  Expert e < num_experts
// takes row (token, s) of `in` where s is its place among the token's choices (ld_in_slot 0: the token's one row) and writes row
// (token, s) of `out`; the shared expert has its own sizes and place topk.  st.n / n_shared: rows of a matrix (gate and up together),
// st.k / k_shared: reduction length (whole operand rows).
//
// The stage is bound by streaming the weights.  Units are numbered expert by expert (the shared one first) and a workgroup takes a
// contiguous range, so that a wavefront reads one contiguous stream per tile and share of the reduction, and the token rows of an
// expert are staged in LDS once for all the units of it: between two units of a range the wavefronts issue nothing but weight
// requests, a ring of D steps x 2 tiles that never drains (64 KB per CU at D = 8; 128 KB gained nothing).  The wavefronts split
// the reduction, so a workgroup's share is balanced to one unit; sums meet in LDS, double-buffered, one workgroup barrier per unit.
// Token rows read from L2 inside the loop had tied every step to a round trip behind the weights.  Before -> now, gate/up and down: 64
// experts of 1536 on rows of 4096, 64 tokens 371 -> 268 and 175 -> 150 us (1.6 GB at 6.1 TB/s, 0.8 GB at 5.5), one token 64.7 -> 45.2
// and 35.1 -> 26.4 us; 128 experts of 768 on rows of 2048, 16 tokens 91 -> 68 and 50 -> 42 us.
struct HyLists {
  unsigned long long tok[MK_MOE_MAX_EXPERTS];   // tokens that visit the expert
  unsigned short entry[896];                    // expert | group of tokens << 8: one entry per `rows that fit` tokens of an expert
  int n_entries, pad[15];
  unsigned place[MK_MOE_MAX_EXPERTS][MK_MAX_TOKENS / 8];  // place of the expert among a token's choices, 4 bits each
};
constexpr int HY_X = (sizeof(HyLists) + 63) / 64 * 64;            // staged token rows [16-byte word of the row][row]
constexpr int HY_RED = MK_LDS_BYTES - 2 * MK_WAVES * 2 * 64 * 16; // partial sums of two units
static_assert(HY_X <= MK_OUT_OFFSET && HY_RED - HY_X >= 128 * 1024, "16 rows of 8 KB fit; the routing's scratch is free by then");
static_assert(MK_MOE_MAX_EXPERTS + MK_MAX_TOKENS * MK_MOE_MAX_TOPK / 2 <= 896 && MK_MOE_MAX_TOPK <= 16 && MK_MOE_MAX_EXPERTS <= 256, "entries with at least two rows each");
template <typename E>
__device__ __forceinline__ float hy_glu(E, CStage &st, bool shared, float a, float b) {
#if MK_HAVE_DUAL
  if (st.flags & MK_F_CLAMP_GLU) {
    const float lim = shared ? st.glu_limit_shared : st.glu_limit, g = fminf(a, lim), u = fminf(fmaxf(b, -lim), lim);
    return g * mx_sigmoid(E(), st.glu_beta * g) * (u + st.glu_bias);
  }
#endif
  return hy_silu(E(), a) * b;
}
// rows that LDS holds of one entry (at most 16: the columns of a matrix instruction); fewer than two: rows are read from memory
template <typename E>
__device__ __forceinline__ int hy_rows(int K) { return min(16, (HY_RED - HY_X) / (K * (int)sizeof(E))); }

// What a workgroup walks: units [s0, s1) of the shared expert (gs groups of tokens, units_s each), then units [r0, r1) of the entries
// (`units` each).  2^ksl_s, 2^ksl wavefronts split the reduction of a pair of tiles of the one and the others.
struct HyRange {
  int s0, s1, r0, r1, gs, units_s, units, ksl_s, ksl;
};
// The u-th unit of a range: D steps of the reduction are a block.
struct HyUnit {
  const u32x4 *w0, *w1;  // this lane's operands of the two tiles
  int nks, kb, ke, nb;   // steps of the reduction, this wavefront's share of them, blocks it takes (alike for all wavefronts)
  int i, pair, n, ksl;   // entry (negative: a group of the shared expert), pair of tiles (may lie behind the last one), outputs, split
};
template <typename E, int D>
__device__ __forceinline__ HyUnit hy_unit(CStage &st, const HyLists *ls, const HyRange &rg, int u, int wave, int lane) {
  HyUnit a;
  const int ns = rg.s1 - rg.s0;
  const bool shared = u < ns;
  const int ksl = shared ? rg.ksl_s : rg.ksl, ks = 1 << ksl;
  const int v = shared ? rg.s0 + u : rg.r0 + u - ns, per = shared ? rg.units_s : rg.units, q = v / per;
  a.pair = ((v - q * per) << (2 - ksl)) + (wave >> ksl);
  a.i = shared ? q - rg.gs : q;
  a.n = shared ? st.n_shared : st.n;
  a.ksl = ksl;
  a.nks = (shared ? st.k_shared : st.k) / FxType<E>::KW;
  const int kq = (a.nks + ks - 1) >> ksl, p = (a.n + 31) / 32;
  a.kb = min(a.nks, (wave & (ks - 1)) * kq);
  a.ke = min(a.nks, a.kb + kq);
  a.nb = (kq + D - 1) / D;
  const int e = shared ? 0 : __builtin_amdgcn_readfirstlane(ls->entry[q]) & 255;
  a.w0 = (shared ? (const u32x4 *)st.w_shared : (const u32x4 *)st.w.seg[0]) + ((size_t)e * p + min(a.pair, p - 1)) * 2 * a.nks * 64 + lane;
  a.w1 = a.w0 + (size_t)a.nks * 64;
  return a;
}
constexpr int HY_FIRST = 8;  // steps of the ring that may have been requested in advance

// Walk the units of `rg`.  w: the ring, its first steps requested if `early`.  row_words: 16-byte words per row where all rows of a single token
// lie in LDS (row of place p at p * row_words; 0: one row).
// XLDS: rows are staged in LDS.  ONCE: the range is one unit, so what would be staged is read once as well: its rows come straight from memory
// beside the weights, and nothing is requested behind its last step.  us, before ranges -> staged -> ONCE: 64 x 64 of 16, 5 tokens 6.8 -> 8.4 ->
// 7.1; 512 x 1024 of 16, 5 tokens 8.9 -> 9.1 -> 8.6; 512 x 2048 of 8, 64 tokens 14.1 -> 13.6 -> 11.1.
template <typename E, int D, bool XLDS, bool ONCE>
__device__ __forceinline__ void hy_expert_walk(CStage &st, const Ctx &c, const HyLists *ls, int M, const HyRange rg, bool early, u32x4 (&w)[2][12], bool rows_in, int row_words, char *smem) {
  constexpr int EPC = FxType<E>::EPC, KW = FxType<E>::KW;
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
  const bool glu = st.flags & MK_F_SILU;
  u32x4 *xl = (u32x4 *)(smem + HY_X);
  f32x4 *red = (f32x4 *)(smem + HY_RED);
  const int ns = rg.s1 - rg.s0, n_all = ns + rg.r1 - rg.r0;
  HyUnit a = hy_unit<E, D>(st, ls, rg, 0, wave, lane);
#pragma unroll
  for (int j = 0; j < D; j++)
    if ((j >= HY_FIRST || !early) && (!ONCE || a.kb + j < a.ke)) {
      w[0][j] = ldg_stream(a.w0 + (size_t)min(a.kb + j, a.nks - 1) * 64);
      w[1][j] = ldg_stream(a.w1 + (size_t)min(a.kb + j, a.nks - 1) * 64);
    }
  int staged = 0x7fffffff, cnt = 1, tok = 0, place = 0;  // rows in LDS belong to this entry; token and place of column lane & 15
  const auto x_rows = dev_rows(st.in);
  int xr = 0;  // row of column lane & 15 in memory, in bytes
  const u32x4 *xb = xl + lg;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  for (int u = 0; u < n_all; u++) {
    if (a.i != staged) {
      // ---- the unit's token rows
      staged = a.i;
      const bool shared = a.i < 0;
      if (rows_in) {
        place = shared ? st.topk : a.i;
        xb = xl + place * row_words + lg;
      } else {
        const int en = shared ? (a.i + rg.gs) << 8 : __builtin_amdgcn_readfirstlane(ls->entry[a.i]), e = en & 255, K = a.nks * KW;
        unsigned long long toks = M >= 64 ? ~0ull : (1ull << M) - 1ull;
        if (!shared) {
          const unsigned long long t = ls->tok[e];
          toks = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)t) | ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(t >> 32)) << 32);
        }
        const int per = XLDS ? hy_rows<E>(K) : 16, r0 = (en >> 8) * per;
        cnt = min(per, __popcll(toks) - r0);
        // lane r gets the r-th token of the group (lane 63 what is left over)
        const int rank = (toks >> lane) & 1 ? __popcll(toks & ((1ull << lane) - 1ull)) - r0 : -1;
        const int nth = __builtin_amdgcn_ds_permute((rank >= 0 && rank < cnt ? rank : 63) << 2, lane);
        auto token = [&](int r) { return __builtin_amdgcn_ds_bpermute(r << 2, nth); };
        auto place_of = [&](int t) { return shared ? st.topk : (int)(ls->place[e][t >> 3] >> ((t & 7) * 4) & 15u); };
        tok = token(min(lr, cnt - 1));
        place = place_of(tok);
        xr = (tok * st.ld_in + place * st.ld_in_slot + lg * EPC) * (int)sizeof(E);
        xb = xl + lg * cnt + min(lr, cnt - 1);
        if constexpr (XLDS) {
          __syncthreads();  // (everybody is done with the rows of the entry before)
          // word q: 16 bytes 4 b + (q & 3) of row r, (b, r) = q / 4 in steps of the grid: four lanes read 64 bytes of a row, and what a wavefront
          // stores is one contiguous piece of LDS
          const int total = cnt * (a.nks << 2), dr = (MK_THREADS / 4) % cnt, db = (MK_THREADS / 4) / cnt;
          int r = (tid >> 2) % cnt, b = (tid >> 2) / cnt;
          for (int q0 = 0; q0 < total; q0 += 8 * MK_THREADS) {
            u32x4 v[8];
            int at[8];
#pragma unroll
            for (int z = 0; z < 8; z++) {
              const bool in = q0 + z * MK_THREADS + tid < total;
              const int t = token(in ? r : 0), j = in ? 4 * b + (tid & 3) : 0;
              at[z] = in ? j * cnt + r : -1;
              v[z] = ldc_16B(x_rows, (t * st.ld_in + place_of(t) * st.ld_in_slot + j * EPC) * (int)sizeof(E));
              r += dr;
              b += db;
              if (r >= cnt) {
                r -= cnt;
                b++;
              }
            }
#pragma unroll
            for (int z = 0; z < 8; z++)
              if (at[z] >= 0) xl[at[z]] = v[z];
          }
          __syncthreads();
        }
      }
    }
    const bool more = u + 1 < n_all;
    const HyUnit nx = more ? hy_unit<E, D>(st, ls, rg, u + 1, wave, lane) : a;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    auto block = [&](int blk, auto refill) {
      constexpr bool REFILL = decltype(refill)::value;
      const bool last = blk + 1 == a.nb;
      const int k0 = a.kb + blk * D;
      u32x4 b[D];
#pragma unroll
      for (int j = 0; j < D; j++) {
        if (ONCE && !REFILL && k0 + j >= a.ke) continue;
        const int s = min(k0 + j, a.nks - 1);
        if constexpr (XLDS) b[j] = xb[s * 4 * cnt];
        else b[j] = ldc_16B(x_rows, xr + s * KW * (int)sizeof(E));
      }
      // what the ring takes next: this unit's block or the first one of the unit behind (behind the range: one line again and again)
      const u32x4 *p0 = last ? nx.w0 : a.w0, *p1 = last ? nx.w1 : a.w1;
      const int kn = last ? nx.kb : k0 + D, end = (last ? nx.nks : a.nks) - 1, kl = last && !more ? min(kn, end) : end;
#pragma unroll
      for (int j = 0; j < D; j++) {
        const bool real = k0 + j < a.ke;
        if (ONCE && !REFILL && !real) continue;
        const u32x4 x = real ? b[j] : zero;  // (both operands: steps behind the share hold values of others, which need not be finite)
#pragma unroll
        for (int h = 0; h < 2; h++) acc[h] = fx_mma_k(E(), real ? w[h][j] : zero, x, acc[h]);
        if constexpr (REFILL) {
          w[0][j] = ldg_stream(p0 + (size_t)min(kn + j, kl) * 64);
          w[1][j] = ldg_stream(p1 + (size_t)min(kn + j, kl) * 64);
        }
      }
    };
    for (int blk = 0; blk < (ONCE ? a.nb - 1 : a.nb); blk++) block(blk, std::true_type{});
    if constexpr (ONCE) block(a.nb - 1, std::false_type{});
    // ---- the wavefronts' sums
    f32x4 *rb = red + (u & 1) * (MK_WAVES * 2 * 64);
#pragma unroll
    for (int h = 0; h < 2; h++) rb[(wave * 2 + h) * 64 + lane] = acc[h];
    __syncthreads();
    const int ks = 1 << a.ksl;
    const f32x4 *rw = rb + (wave >> a.ksl << a.ksl) * 2 * 64 + lane;
    auto total = [&](int h) {
      f32x4 v = rw[h * 64];
      for (int q = 1; q < ks; q++) v += rw[(2 * q + h) * 64];
      return v;
    };
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if (((2 * u + h) & (ks - 1)) != (wave & (ks - 1)) || lr >= cnt || (glu && h) || a.pair * 32 >= a.n) continue;
      const f32x4 v = total(h);
      float r[4] = {v[0], v[1], v[2], v[3]};
      if (glu) {
        const f32x4 g = total(1);
#pragma unroll
        for (int q = 0; q < 4; q++) r[q] = hy_glu(E(), st, a.i < 0, r[q], g[q]);
      }
      fx_stc4((E *)st.out + (size_t)tok * st.ld_out + (size_t)place * st.ld_out_slot, (glu ? a.pair : 2 * a.pair + h) * 16 + lg * 4, glu ? a.n / 2 : a.n, r);
    }
    a = nx;
  }
}
template <typename E, int MAXM>
__device__ __forceinline__ void stage_hy_experts(CStage &st, Ctx &c, int M, char *smem) {
  constexpr int EPC = FxType<E>::EPC, KW = FxType<E>::KW;
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int Ex = st.num_experts, topk = st.topk;
  HyLists *ls = (HyLists *)smem;
  const int fit = hy_rows<E>(st.k), fit_s = st.w_shared ? hy_rows<E>(st.k_shared) : 16;
  // Rows in LDS for fewer tokens than an expert has make its weights pass again, which costs where the units fill the chip as it is: rows are
  // read from memory then, 16 tokens at a time.  2048 x 16384 of 4 (4 rows fit), 33 / 64 tokens, us: before ranges 67 / 91, staged 112 / 193, from
  // memory 46 / 80; 2048 x 8192 (8 rows) 43 / 52, 42 / 63, 26 / 43; a shared 512 x 8192 beside few units, 33 tokens: staged 21, from memory 35.
  const int pairs = (st.n + 31) / 32, pairs_s = st.w_shared ? (st.n_shared + 31) / 32 : 0;
  const bool again = (fit < 16 && M * topk > Ex * fit) || (fit_s < 16 && M > fit_s);
  const bool xlds = fit >= 2 && fit_s >= 2 && !(again && min(Ex, M * topk) * pairs + (M + 15) / 16 * pairs_s >= c.G);
  const int per = xlds ? fit : 16, per_s = xlds ? fit_s : 16;
  HyRange rg;
  rg.gs = st.w_shared ? (M + per_s - 1) / per_s : 0;
  // A wavefront takes a whole reduction where that is not much longer than its ring, or half of it.  64 experts of 1024, 16 tokens, us, whole /
  // halves / quarters: 512 values 16.4 / - / 22.5, 768: 19.6 / 22.1 / 22.9, 1024: 24.1 / 25.9 / 24.8, 1536: - / 33.1 / 34.9, 2048: - / 40.7 / 39.8.
  // The shared expert goes by its own length (512 x 8192 beside 1024 x 1024, one token: 23.4 -> 15.6, eight workgroups had streamed it), and where
  // there are not even as many pairs of tiles as workgroups, all four wavefronts share one.
  const bool few = min(Ex, M * topk) * pairs + rg.gs * pairs_s <= c.G;
  auto split = [&](int nks) { return few || nks >= 48 ? 2 : nks >= 24 ? 1 : 0; };
  const int nks = st.k / KW;
  rg.ksl = split(nks);
  rg.ksl_s = split(st.k_shared / KW);
  auto units = [&](int p, int ksl) { return (p + (MK_WAVES >> ksl) - 1) / (MK_WAVES >> ksl); };
  rg.units = units(pairs, rg.ksl);
  rg.units_s = units(pairs_s, rg.ksl_s);
  const int n_s = rg.gs * rg.units_s;
  auto share = [](int n, int v, int of) {  // n v / of, without the product
    const unsigned q = (unsigned)n / (unsigned)of;
    return (int)(q * v + ((unsigned)n - q * of) * v / (unsigned)of);
  };
  auto part = [&](int n, int v) { return share(n, v, c.G); };
  // A few tokens: a share of the shared expert first, whose weights are known before the routing is (3072 x 4096 of 64, 2 tokens: 51.1 us, as
  // one range with the others 53.0; 4 and 8 tokens alike within 1 %), ...
  const bool deal = M <= 4;
  rg.s0 = deal ? part(n_s, c.vid) : 0;
  rg.s1 = deal ? part(n_s, c.vid + 1) : 0;
  // ... and then of the other units so many that all workgroups have alike; fewer units than workgroups: those that have none take them (a
  // share of each by itself met in the same workgroups: 512 x 1024 of 16 and a shared 1024 x 1024, 2 tokens 13.7 -> 10.1 us).
  auto deal_routed = [&](int n_r) {
    const int all = n_s + n_r, fr = c.G - n_s;
    if (n_s >= c.G) {
      rg.r0 = part(n_r, c.vid);
      rg.r1 = part(n_r, c.vid + 1);
    } else if (all >= c.G) {
      rg.r0 = part(all, c.vid) - rg.s0;
      rg.r1 = part(all, c.vid + 1) - rg.s1;
    } else {
      rg.r0 = share(n_r, c.vid - rg.s0, fr);
      rg.r1 = share(n_r, c.vid + 1 - rg.s1, fr);
    }
  };
  // rows of a single token: all of them in LDS at once
  const int one_words = max(st.k, st.w_shared ? st.k_shared : 0) / EPC, one_rows = st.ld_in_slot ? topk + (st.w_shared ? 1 : 0) : 1;
  const bool inline_route = M == 1 && (st.flags & MK_F_MOE_INLINE_TOPK);
  const bool rows_in = M == 1 && one_rows * one_words * 16 <= (inline_route ? MK_OUT_OFFSET : HY_RED) - HY_X;
  u32x4 w[2][12];
  const bool early = rg.s0 < rg.s1 && wave != 0;  // (wavefront 0 polls and routes)
  if (early) {
    const HyUnit a = hy_unit<E, HY_FIRST>(st, ls, rg, 0, wave, lane);
#pragma unroll
    for (int j = 0; j < HY_FIRST; j++) {
      w[0][j] = ldg_stream(a.w0 + (size_t)min(a.kb + j, a.nks - 1) * 64);
      w[1][j] = ldg_stream(a.w1 + (size_t)min(a.kb + j, a.nks - 1) * 64);
    }
  }
  if (rows_in) deal_routed(topk * rg.units);
  if (M > 1 || !rows_in) {
    for (int i = tid; i < Ex; i += MK_THREADS) ls->tok[i] = 0ull;
    for (int i = tid; i < Ex * (MK_MAX_TOKENS / 8); i += MK_THREADS) ls->place[0][i] = 0u;
  }
  if (!c.pending) __syncthreads();  // (an iteration's first stage has no barrier to wait for: everybody is done clearing)
  barrier_wait(c);
  // ---- which experts have which tokens
  if (rows_in) {
    if (wave == 0) {
      float f = 0.f;
      int id = 0;
      if (inline_route) {
        hy_route_wave(st, (const float *)st.moe_logits, lane, f, id, (float *)(smem + MK_OUT_OFFSET));
        if (c.vid == 0) hy_route_store(st, 0, lane, f, id);
      } else if (lane < topk) {
        id = ldc_i32(st.ids + lane);
      }
      if (lane < topk) ls->entry[lane] = (unsigned short)id;
    } else {
      u32x4 *xl = (u32x4 *)(smem + HY_X);
      const int total = one_rows * one_words;
      const auto x_rows = dev_rows(st.in);
      for (int q0 = tid - 64; q0 < total; q0 += 4 * (MK_THREADS - 64)) {
        u32x4 v[4];
#pragma unroll
        for (int z = 0; z < 4; z++) {
          const int q = min(q0 + z * (MK_THREADS - 64), total - 1), p = q / one_words, j = q - p * one_words;
          v[z] = ldc_16B(x_rows, p * st.ld_in_slot * (int)sizeof(E) + 16 * min(j, (p == topk ? st.k_shared : one_rows == 1 ? one_words * EPC : st.k) / EPC - 1));
        }
#pragma unroll
        for (int z = 0; z < 4; z++)
          if (q0 + z * (MK_THREADS - 64) < total) xl[q0 + z * (MK_THREADS - 64)] = v[z];
      }
    }
    __syncthreads();
  } else {
    if (inline_route) {
      if (wave == 0) {
        float f;
        int id;
        hy_route_wave(st, (const float *)st.moe_logits, lane, f, id, (float *)(smem + MK_OUT_OFFSET));
        if (lane < topk) {
          ls->tok[id] = 1ull;
          ls->place[id][0] = (unsigned)lane;
        }
        if (c.vid == 0) hy_route_store(st, 0, lane, f, id);
      }
    } else {
      for (int i = tid; i < M * topk; i += MK_THREADS) {
        // (an expert that a token names twice -- the caller's ids may, and so may a routing over NaN -- has the place that came first: places
        // put together would lie outside the token's row)
        const int t = i / topk, id = ldc_i32(st.ids + i);
        if (!(atomicOr(&ls->tok[id], 1ull << t) >> t & 1)) atomicOr(&ls->place[id][t >> 3], (unsigned)(i - t * topk) << ((t & 7) * 4));
      }
    }
    __syncthreads();
    if (wave == 0) {
      int base = 0;
      for (int q = 0; q < Ex; q += 64) {
        const int g = q + lane < Ex ? (__popcll(ls->tok[q + lane]) + per - 1) / per : 0;
        const int end = base + wave_incl_scan(g, lane);
        for (int i = 0; i < g; i++) ls->entry[end - g + i] = (unsigned short)(q + lane | i << 8);
        base = wave_bcast(end, 63);
      }
      if (lane == 0) ls->n_entries = base;
    }
    __syncthreads();
    const int n_r = __builtin_amdgcn_readfirstlane(ls->n_entries) * rg.units;
    if (deal) {
      deal_routed(n_r);
    } else {  // one range over the shared expert's units and the entries'
      const int u0 = part(n_s + n_r, c.vid), u1 = part(n_s + n_r, c.vid + 1);
      rg.s0 = min(u0, n_s);
      rg.s1 = min(u1, n_s);
      rg.r0 = max(u0 - n_s, 0);
      rg.r1 = max(u1 - n_s, 0);
    }
  }
  if (rg.s0 < rg.s1 || rg.r0 < rg.r1) {
    // a ring of 8 steps per tile, or of 12 where a wavefront's share of the reduction is then walked with fewer empty steps
    const int kq = (nks + (1 << rg.ksl) - 1) >> rg.ksl;
    const bool once = per == 16 && per_s == 16 && rg.s1 - rg.s0 + rg.r1 - rg.r0 == 1;
    if (once && !rows_in) hy_expert_walk<E, 8, false, true>(st, c, ls, M, rg, early, w, false, 0, smem);
    else if (!xlds && !rows_in) hy_expert_walk<E, 8, false, false>(st, c, ls, M, rg, early, w, false, 0, smem);
    else if ((kq + 7) / 8 * 8 <= (kq + 11) / 12 * 12) hy_expert_walk<E, 8, true, false>(st, c, ls, M, rg, early, w, rows_in, one_rows > 1 ? one_words : 0, smem);
    else hy_expert_walk<E, 12, true, false>(st, c, ls, M, rg, early, w, rows_in, one_rows > 1 ? one_words : 0, smem);
  }
  c.wrote_through = true;
}
