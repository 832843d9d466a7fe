// Stages whose sizes and constants are all data (part of the persistent kernel, included by mk_kernel.hip).
//
// The stages above this file are written for one family of shapes (heads of 128 values, a bf16 residual stream, a norm
// in front of each sub-layer).  The ones here take any head size, separate value size and head grouping, keep the
// residual stream in 32 bits, and get every constant from their descriptor, so that a model of another design is another
// list of descriptors:
//   * stage_fx_embed    rows of a table times a constant, as 32-bit residual rows and as rows for the next linear;
//   * stage_fx_addnorm  alpha * x + y, RMS norm with weight (offset + w), written in both forms (y is optional);
//   * stage_fx_prep /   rotary positions on part of a head, heads divided by their root mean square, paged K/V append,
//     stage_fx_attn     softcapped scores, softmax with an extra per-head logit in the denominator, split-KV on the matrix
//                       cores for prompt portions and for single tokens alike;
//   * stage_fx_linear_f32  the 32-bit form of the linear.
// The stages are instantiated for bf16 (E = uint16_t) and for 32-bit (E = float) activations, weights and caches; scores,
// softmax, norms, angles and the residual stream are 32-bit in both.

template <typename E> struct FxType;
// EPC: elements per 16-byte operand; KW: head dims one matrix-core operand row covers (4 lane groups x EPC);
// TP: cached positions per tile; SUB: 16-position sub-tiles of a tile
template <> struct FxType<uint16_t> {
  static constexpr int EPC = 8, KW = 32, TP = 32, SUB = 2;
};
template <> struct FxType<float> {
  static constexpr int EPC = 4, KW = 16, TP = 16, SUB = 1;
};
__device__ __forceinline__ float fx_ldc(const uint16_t *p) { return bf2f(ldc_u16(p)); }
__device__ __forceinline__ float fx_ldc(const float *p) { return ldc_f32(p); }
__device__ __forceinline__ float fx_val(uint16_t v) { return bf2f(v); }
__device__ __forceinline__ float fx_val(float v) { return v; }
template <typename E> __device__ __forceinline__ E fx_round(float v) {
  if constexpr (sizeof(E) == 2) return (E)f2bf(v);
  else return v;
}
__device__ __forceinline__ void fx_stc(uint16_t *p, uint16_t v) { stc_u16(p, v); }
__device__ __forceinline__ void fx_stc(float *p, float v) { stc_f32(p, v); }
__device__ __forceinline__ void fx_stc4(uint16_t *row, int n0, int n_out, const float (&r)[4]) { stc_bf16x4(row, n0, n_out, r); }
__device__ __forceinline__ void fx_stc4(float *row, int n0, int n_out, const float (&r)[4]) {
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (n0 + i < n_out) stc_f32(row + n0 + i, r[i]);
}
// four consecutive row elements, 16-byte (32-bit) or 8-byte (bf16) aligned
__device__ __forceinline__ f32x4 fx_ldc_quad(const uint16_t *p) {
  const unsigned long long u = ldc_u64(p);
  const uint32_t a = (uint32_t)u, b = (uint32_t)(u >> 32);
  return (f32x4){bf_lo(a), bf_hi(a), bf_lo(b), bf_hi(b)};
}
__device__ __forceinline__ f32x4 fx_ldc_quad(const float *p) { return __builtin_bit_cast(f32x4, ldc_16B((const u32x4 *)p)); }
// ... of a table nobody writes during a launch
__device__ __forceinline__ f32x4 fx_ld_quad(const uint16_t *p) {
  const unsigned long long u = *(const unsigned long long *)p;
  const uint32_t a = (uint32_t)u, b = (uint32_t)(u >> 32);
  return (f32x4){bf_lo(a), bf_hi(a), bf_lo(b), bf_hi(b)};
}
__device__ __forceinline__ f32x4 fx_ld_quad(const float *p) { return *(const f32x4 *)p; }
__device__ __forceinline__ void fx_stc_quad(uint16_t *p, f32x4 v) {
  stc_u64(p, (unsigned long long)pack2(v[0], v[1]) | ((unsigned long long)pack2(v[2], v[3]) << 32));
}
__device__ __forceinline__ void fx_stc_quad(float *p, f32x4 v) { stc_16B((u32x4 *)p, __builtin_bit_cast(u32x4, v)); }

// Maximum / sum over the four 16-lane groups of a wavefront (every lane gets the result of its column lane & 15).
__device__ __forceinline__ float groups_max(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const unsigned w = __float_as_uint(v);
  const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float groups_sum(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const unsigned w = __float_as_uint(v);
  const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// ----------------------------------------------------------------------------- embedding
// out2[t, :] = table[id] * alpha in 32 bits, out[t, :] = the same rounded to E.  A negative id gives a row of zeros.
template <typename E>
__device__ __forceinline__ void stage_fx_embed(CStage &st, Ctx &c, const MkRuntime &rt, int M) {
  barrier_wait(c);
  const int k = st.k;
  for (int t = row_item(c, c.vid); t < M; t += c.G) {
    long long id;
    if (st.flags & MK_F_EMBED_FROM_TOKENS) {
      const int req = ldc_i32(&rt.request_ids[c.sh_tok[MK_MAX_TOKENS + t]]);
      id = (long long)ldc_u64(&rt.tokens[(long long)req * rt.max_seq + c.sh_tok[t]]);
    } else {
      id = (long long)ldc_u64((const long long *)st.in + t);
    }
    const float scale = id < 0 ? 0.f : st.alpha;
    const E *src = (const E *)st.w.seg[0] + (size_t)(id < 0 ? 0 : id) * k;
    E *out = (E *)st.out + (size_t)t * st.ld_out;
    float *out32 = st.out2 ? (float *)st.out2 + (size_t)t * st.ld_out2 : nullptr;
#if MK_HAVE_DUAL
    if (st.pos_tab) {  // (the caller keeps positions inside the table)
      const E *pos = (const E *)st.pos_tab + (size_t)min(c.sh_tok[t], st.pos_rows - 1) * k;
      if ((k & 3) == 0) {
        for (int i = c.tid * 4; i < k; i += MK_THREADS * 4) {
          const f32x4 v = fx_ld_quad(src + i) * scale + fx_ld_quad(pos + i);
          if (out32) fx_stc_quad(out32 + i, v);
          fx_stc_quad(out + i, v);
        }
      } else {
        for (int i = c.tid; i < k; i += MK_THREADS) {
          const float v = fmaf(fx_val(src[i]), scale, fx_val(pos[i]));
          if (out32) stc_f32(out32 + i, v);
          fx_stc(out + i, fx_round<E>(v));
        }
      }
      continue;
    }
#endif
    if ((k & 3) == 0) {
      for (int i = c.tid * 4; i < k; i += MK_THREADS * 4) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = fx_val(src[i + e]) * scale;
        if (out32) fx_stc_quad(out32 + i, v);
        fx_stc_quad(out + i, v);
      }
    } else {
      for (int i = c.tid; i < k; i += MK_THREADS) {
        const float v = fx_val(src[i]) * scale;
        if (out32) stc_f32(out32 + i, v);
        fx_stc(out + i, fx_round<E>(v));
      }
    }
  }
  c.wrote_through = true;
}

// ----------------------------------------------------------------------------- residual sum + RMS norm
// v = alpha * x + y;  out2 = v / sqrt(mean(v^2) + eps) * (w_offset + w) in 32 bits, out = the same rounded to E.  Rows are
// st.n long with st.k of them real (the rest is zero in every operand).  x (st.res) is 32-bit, y (st.in, null: none) is the
// preceding linear's output, or its K-slice partials when that linear left its sum to this stage.  A workgroup per row.
// Bound by the barrier and one round trip for the row: weights and residual are requested ahead of the barrier and all quads of a thread (four,
// eight or twelve) before the first value is waited for, the slices of four quads at a time; a branch around each quad had made a round trip
// per quad of it, and rows of more than 4096 values that waited in LDS for their factor a round trip per 4096.  As a stage, us, 4 / 64 rows:
// 4096 values from four slices 8.9 -> 3.6 / 9.5 -> 4.2; of a 32-bit summand 8192 values 5.1 (by LDS 5.7) -> 3.5 / 5.6 (6.6) -> 4.3, 12,288 values
// 6.1 (7.7) -> 4.2 / 8.0 (9.2) -> 5.6; of a bf16 one 8192 values 8.0 (7.1) -> 5.3 / 8.8 (8.0) -> 6.0.
__device__ __forceinline__ int fx_quad_at(const Ctx &c, int c0, int j, int n4) { return min(c0 + c.tid + j * MK_THREADS, n4 - 1); }
// slices of four quads of a row that the linear in front left unsummed, in slice order
__device__ __forceinline__ void fx_addnorm_slices(const Ctx &c, int dS, int t, int c0, int n4, f32x4 *v) {
  const float *p = c.defer_part + (size_t)t * c.defer_n;
  const size_t slice = (size_t)c.defer_rows * c.defer_n;
  auto sum = [&](auto ns) {
    constexpr int Q = decltype(ns)::value;
    f32x4 q[4][Q];
#pragma unroll
    for (int b = 0; b < Q; b++) {
      const auto rows = dev_rows(p + b * slice);
#pragma unroll
      for (int j = 0; j < 4; j++) q[j][b] = __builtin_bit_cast(f32x4, ldc_16B(rows, 16 * fx_quad_at(c, c0, j, n4)));
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      v[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < Q; b++) v[j] += q[j][b];
    }
  };
  if (dS == 2) sum(std::integral_constant<int, 2>{});
  else if (dS == 4) sum(std::integral_constant<int, 4>{});
  else sum(std::integral_constant<int, 8>{});
}
// NS quads per thread
template <typename E, int NS>
__device__ __forceinline__ void stage_fx_addnorm_t(CStage &st, Ctx &c, int M, char *smem) {
  const int tid = c.tid, n4 = st.n / 4;
  float *red = (float *)smem;
  const f32x4 *w4 = (const f32x4 *)st.norm_w;
  const float *xr = (const float *)st.res;
  const int t0 = row_item(c);
  f32x4 g[NS], x[NS], v[NS];
  auto load_x = [&](int t) {
    const auto row = dev_rows(xr + (size_t)t * st.ld_res);
#pragma unroll
    for (int j = 0; j < NS; j++) x[j] = __builtin_bit_cast(f32x4, ldc_16B(row, 16 * fx_quad_at(c, 0, j, n4)));
  };
#pragma unroll
  for (int j = 0; j < NS; j++) g[j] = w4[fx_quad_at(c, 0, j, n4)];
  // the residual row was written at least one barrier earlier than y: requested before the barrier is awaited (not by the
  // wavefront that polls it)
  const bool pre = (st.flags & MK_F_RES_EARLY) && t0 < M && tid >= 64;
  if (pre) load_x(t0);
  barrier_wait(c);
  const int dS = c.defer_S;
  c.defer_S = 0;
  for (int t = t0; t < M; t += c.G) {
    if (!(pre && t == t0)) load_x(t);
    if (dS) {
#pragma unroll
      for (int j = 0; j < NS; j += 4) fx_addnorm_slices(c, dS, t, j * MK_THREADS, n4, v + j);
    } else {
#pragma unroll
      for (int j = 0; j < NS; j++) v[j] = st.in ? fx_ldc_quad((const E *)st.in + (size_t)t * st.ld_in + 4 * fx_quad_at(c, 0, j, n4)) : (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NS; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        v[j][e] = fmaf(st.alpha, x[j][e], v[j][e]);
        ss += tid + j * MK_THREADS < n4 ? v[j][e] * v[j][e] : 0.f;
      }
    const float r = 1.f / sqrtf(block_sum(ss, red) / (float)st.k + st.eps);
#pragma unroll
    for (int j = 0; j < NS; j++)
      if (tid + j * MK_THREADS < n4) {
        const int s = tid + j * MK_THREADS;
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (v[j][e] * r) * (st.w_offset + g[j][e]);
        if (st.out2) fx_stc_quad((float *)st.out2 + (size_t)t * st.ld_out2 + 4 * s, o);
        fx_stc_quad((E *)st.out + (size_t)t * st.ld_out + 4 * s, o);
      }
    __syncthreads();
  }
  c.wrote_through = true;
}
template <typename E>
__device__ __forceinline__ void stage_fx_addnorm(CStage &st, Ctx &c, int M, char *smem) {
  if (st.n <= 4 * 4 * MK_THREADS) stage_fx_addnorm_t<E, 4>(st, c, M, smem);
  else if (st.n <= 8 * 4 * MK_THREADS) stage_fx_addnorm_t<E, 8>(st, c, M, smem);
  else stage_fx_addnorm_t<E, 12>(st, c, M, smem);
}

#if MK_PAIR
// The rows of several portions, two of them in flight: see norm_group_rows.
template <typename E, int NS>
__device__ __forceinline__ void fx_addnorm_group(Ctx &c, const MkRuntime &rt, int s, int portions, const int *sh_rows, char *smem) {
  CStage &st = mk_portion_stages(rt, 0)[s];
  const int tid = c.tid, n4 = st.n / 4;
  float *red = (float *)smem;
  const f32x4 *w4 = (const f32x4 *)st.norm_w;
  f32x4 g[NS];
#pragma unroll
  for (int j = 0; j < NS; j++) g[j] = w4[fx_quad_at(c, 0, j, n4)];
  barrier_wait(c);
  const int dS = c.defer_S, total = group_rows(portions, sh_rows);
  c.defer_S = 0;
  for (int i = row_item(c); i < total; i += 2 * c.G) {
    GroupRow r[2];
    f32x4 x[2][NS], v[2][NS];
#pragma unroll
    for (int z = 0; z < 2; z++) {
      r[z] = group_row(i + z * c.G, portions, sh_rows);
      CStage &sp = mk_portion_stages(rt, r[z].portion)[s];
      const auto row = dev_rows((const float *)sp.res + (size_t)r[z].row * st.ld_res);
#pragma unroll
      for (int j = 0; j < NS; j++) x[z][j] = __builtin_bit_cast(f32x4, ldc_16B(row, 16 * fx_quad_at(c, 0, j, n4)));
      if (dS) {
#pragma unroll
        for (int j = 0; j < NS; j += 4) fx_addnorm_slices(c, dS, r[z].portion * MK_MAX_TOKENS + r[z].row, j * MK_THREADS, n4, v[z] + j);
      } else {
#pragma unroll
        for (int j = 0; j < NS; j++) v[z][j] = sp.in ? fx_ldc_quad((const E *)sp.in + (size_t)r[z].row * st.ld_in + 4 * fx_quad_at(c, 0, j, n4)) : (f32x4){0.f, 0.f, 0.f, 0.f};
      }
    }
    float ss[2] = {0.f, 0.f};
#pragma unroll
    for (int z = 0; z < 2; z++)
#pragma unroll
      for (int j = 0; j < NS; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          v[z][j][e] = fmaf(st.alpha, x[z][j][e], v[z][j][e]);
          ss[z] += tid + j * MK_THREADS < n4 ? v[z][j][e] * v[z][j][e] : 0.f;
        }
    block_sums(ss, red);
#pragma unroll
    for (int z = 0; z < 2; z++) {
      const float f = 1.f / sqrtf(ss[z] / (float)st.k + st.eps);
      CStage &sp = mk_portion_stages(rt, r[z].portion)[s];
#pragma unroll
      for (int j = 0; j < NS; j++)
        if (r[z].valid && tid + j * MK_THREADS < n4) {
          const int q = tid + j * MK_THREADS;
          f32x4 o;
#pragma unroll
          for (int e = 0; e < 4; e++) o[e] = (v[z][j][e] * f) * (st.w_offset + g[j][e]);
          if (sp.out2) fx_stc_quad((float *)sp.out2 + (size_t)r[z].row * st.ld_out2 + 4 * q, o);
          fx_stc_quad((E *)sp.out + (size_t)r[z].row * st.ld_out + 4 * q, o);
        }
    }
    __syncthreads();
  }
  c.wrote_through = true;
}
template <typename E>
__device__ __forceinline__ void stage_fx_addnorm_group(CStage &st, Ctx &c, const MkRuntime &rt, int s, int portions, const int *sh_rows, char *smem) {
  if (st.n <= 4 * 4 * MK_THREADS) fx_addnorm_group<E, 4>(c, rt, s, portions, sh_rows, smem);
  else if (st.n <= 8 * 4 * MK_THREADS) fx_addnorm_group<E, 8>(c, rt, s, portions, sh_rows, smem);
  else fx_addnorm_group<E, 12>(c, rt, s, portions, sh_rows, smem);
}
#endif

// ----------------------------------------------------------------------------- head rows
// Where the q/k/v rows of an attention stage come from: the linear's output, or its unsummed K-slice partials.
template <typename E> struct FxRows {
  const E *in;
  int ld;
  int S;
  const float *part;
  size_t slice, ldp;
  const float *bias;  // (hybrid kernels) added to every row where it is used, null: none
  // what one element is made of: the linear's output, or its slices ...
  template <int NS> __device__ __forceinline__ void request(int tok, int col, float (&q)[NS ? NS : 1]) const {
    if constexpr (NS == 0) {
      q[0] = fx_ldc(in + (size_t)tok * ld + col);
    } else {
      const float *p = part + (size_t)tok * ldp + col;
#pragma unroll
      for (int b = 0; b < NS; b++) q[b] = ldc_f32(p + b * slice);
    }
  }
  // ... and its value, rounded as the linear would have
  template <int NS> static __device__ __forceinline__ float value(const float (&q)[NS ? NS : 1]) {
    if constexpr (NS == 0) {
      return q[0];
    } else {
      float s = 0.f;
#pragma unroll
      for (int b = 0; b < NS; b++) s += q[b];
      return fx_val(fx_round<E>(s));
    }
  }
  // f(slices) with the slice count as a compile-time constant: one branch per row instead of one per element
  template <typename F> __device__ __forceinline__ void with_slices(F f) const {
    if (S == 0) f(std::integral_constant<int, 0>{});
    else if (S == 2) f(std::integral_constant<int, 2>{});
    else if (S == 4) f(std::integral_constant<int, 4>{});
    else f(std::integral_constant<int, 8>{});
  }
};
template <typename E> __device__ __forceinline__ FxRows<E> fx_rows(CStage &st, Ctx &c) {
  FxRows<E> r{(const E *)st.in, st.ld_in, c.defer_S, c.defer_part, (size_t)c.defer_rows * c.defer_n, (size_t)c.defer_n, MK_HAVE_HYB ? st.in_bias : nullptr};
  c.defer_S = 0;
  return r;
}
// f(registers a head row takes per lane)
template <typename F> __device__ __forceinline__ void fx_head_regs(int D, int DV, F f) {
  if (max(D, DV) <= 128) f(std::integral_constant<int, 2>{});
  else f(std::integral_constant<int, MK_FX_MAX_HEAD_DIM / 64>{});
}
// One query or key head row by one wavefront, lane l holding every 64th column: dims [0, rot) are rotated (dim i < rot / 2 pairs with
// i + rot / 2), then the row is divided by sqrt(mean(x^2) + eps) when the stage asks for it; put(d, value) for every d < D.  A value
// row is copied as it is.
//
// Bound by round trips: a wavefront requests two rows with all their slices at once, and partners of the rotation change lanes in the
// wavefront's own LDS.  (A branch around every 64 columns, and a second request for the partners, had made four to eight trips of a row.)
// Heads of up to 128 columns have their own form (R = 2 registers a row): branches past six more blocks of every loop had each been a fetch
// of instructions.  Rows ready after the barrier of the attention stage, 32 q / 8 kv heads of 128, four streams: 9.5 -> 5.0 us; prep stage
// of 64 tokens 7.3 -> 4.0 us.
//
// Dual kernels, MK_F_ROW_NORM: the row's query heads (its key heads) are together divided by their root mean square and multiplied
// by a weight per column instead; `r` is that factor, `w` the weights.
template <int R> struct FxHead {
  float x[R], cs[R], sn[R];
#if MK_HAVE_HYB
  float b[R];  // bias of x
#endif
#if MK_HAVE_DUAL
  float r, w[R];
#endif
};
#if MK_HAVE_DUAL
// Weights of the row norm for the head whose columns begin at `col`.
template <int R>
__device__ __forceinline__ void fx_row_weights(CStage &st, int col, int lane, FxHead<R> &h) {
  if (!(st.flags & MK_F_ROW_NORM)) return;
  const int nq = st.num_q_heads * st.head_dim;
  const float *w = col < nq ? (const float *)st.q_norm_w + col : (const float *)st.k_norm_w + (col - nq);
#pragma unroll
  for (int j = 0; j < R; j++)
    if (R == 2 || j * 64 < st.head_dim) h.w[j] = w[min(j * 64 + lane, st.head_dim - 1)];
}
// This lane's part of the sum of squares over columns [c0, c1) of a row, lane `id` of `n`.
template <typename E>
__device__ __forceinline__ float fx_row_squares(const E *row, int c0, int c1, int id, int n) {
  float ss = 0.f;
  for (int q0 = c0 / 4 + id; q0 * 4 < c1; q0 += 4 * n) {
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = fx_ldc_quad(row + 4 * min(q0 + j * n, (c1 - 1) / 4));
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int at = 4 * (q0 + j * n) + e;
        ss += at >= c0 && at < c1 ? v[j][e] * v[j][e] : 0.f;
      }
  }
  return ss;
}
#endif
// Columns [col, col + n) of row `tok`, by one wavefront.
struct FxSpan {
  int tok, col, n;
};
#if MK_PAIR
template <typename E, int R, int N>
__device__ __forceinline__ void fx_span_loads(const FxRows<E> &rows, const FxSpan (&s)[N], int lane, FxHead<R> (&h)[N]) {
  rows.with_slices([&](auto ns) {
    constexpr int NS = decltype(ns)::value;
    int most = 0;
#pragma unroll
    for (int z = 0; z < N; z++) most = max(most, s[z].n);
#pragma unroll
    for (int j = 0; j < R; j += 2)
      if (R == 2 || j * 64 < most) {
        float q[N][2][NS ? NS : 1];
#pragma unroll
        for (int z = 0; z < N; z++)
#pragma unroll
          for (int i = 0; i < 2; i++) rows.template request<NS>(s[z].tok, s[z].col + min((j + i) * 64 + lane, s[z].n - 1), q[z][i]);
#pragma unroll
        for (int z = 0; z < N; z++)
#pragma unroll
          for (int i = 0; i < 2; i++) h[z].x[j + i] = rows.template value<NS>(q[z][i]);
      }
  });
}
#endif
template <typename E, int R>
__device__ __forceinline__ void fx_span_load2(const FxRows<E> &rows, const FxSpan &s0, const FxSpan &s1, int lane, FxHead<R> &h0, FxHead<R> &h1) {
  rows.with_slices([&](auto ns) {
    constexpr int NS = decltype(ns)::value;
#pragma unroll
    for (int j = 0; j < R; j += 2)
      if (R == 2 || j * 64 < max(s0.n, s1.n)) {
        float q[2][2][NS ? NS : 1];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const int d = (j + i) * 64 + lane;
          rows.template request<NS>(s0.tok, s0.col + min(d, s0.n - 1), q[0][i]);
          rows.template request<NS>(s1.tok, s1.col + min(d, s1.n - 1), q[1][i]);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
          h0.x[j + i] = rows.template value<NS>(q[0][i]);
          h1.x[j + i] = rows.template value<NS>(q[1][i]);
        }
      }
  });
}
// What is requested beside a row: its bias (hybrid kernels; added when it is used), and a head's rotation at position `pos`.
template <typename E, int R>
__device__ __forceinline__ void fx_head_tables(CStage &st, const FxRows<E> &rows, const FxSpan &s, bool rotated, int pos, int lane, FxHead<R> &h) {
#if MK_HAVE_HYB
#pragma unroll
  for (int j = 0; j < R; j++) h.b[j] = 0.f;
  if (rows.bias) {
#pragma unroll
    for (int j = 0; j < R; j++)
      if (R == 2 || j * 64 < s.n) h.b[j] = rows.bias[s.col + min(j * 64 + lane, s.n - 1)];
  }
#endif
  const int rot = rotated && (st.flags & MK_F_ROPE) ? st.rot_dims : 0, half = rot >> 1;
  const float *ct = (const float *)st.cos_tab + (size_t)pos * st.ld_cos, *sn = (const float *)st.sin_tab + (size_t)pos * st.ld_cos;
#pragma unroll
  for (int j = 0; j < R; j++)
    if (j * 64 < rot) {
      const int d = j * 64 + lane, ci = d < rot ? (d < half ? d : d - half) : 0;
      h.cs[j] = ct[ci];
      h.sn[j] = sn[ci];
    }
}
// element j of a value row
template <int R>
__device__ __forceinline__ float fx_value(const FxHead<R> &h, int j) {
#if MK_HAVE_HYB
  return h.x[j] + h.b[j];
#else
  return h.x[j];
#endif
}
// `xs`: MK_FX_MAX_HEAD_DIM floats of LDS of this wavefront
template <int R, typename Put>
__device__ __forceinline__ void fx_head_finish(CStage &st, int lane, FxHead<R> &h, float *xs, Put put) {
  const int D = st.head_dim, rot = (st.flags & MK_F_ROPE) ? st.rot_dims : 0, half = rot >> 1;
  float ss = 0.f;
#if MK_HAVE_HYB
#pragma unroll
  for (int j = 0; j < R; j++) h.x[j] += h.b[j];
#endif
#pragma unroll
  for (int j = 0; j < R; j++)
    if (j * 64 < rot) xs[j * 64 + lane] = h.x[j];
#pragma unroll
  for (int j = 0; j < R; j++)
    if (R == 2 || j * 64 < D) {
      const int d = j * 64 + lane;
      if (j * 64 < rot) {
        const float xp = xs[d < rot ? (d < half ? d + half : d - half) : 0];
        if (d < rot) h.x[j] = d < half ? h.x[j] * h.cs[j] - xp * h.sn[j] : h.x[j] * h.cs[j] + xp * h.sn[j];
      }
      ss += d < D ? h.x[j] * h.x[j] : 0.f;
    }
  if (st.flags & MK_F_QK_NORM) {
    const float r = 1.f / sqrtf(wave_sum(ss) / (float)D + st.eps);
#pragma unroll
    for (int j = 0; j < R; j++)
      if (R == 2 || j * 64 < D) h.x[j] *= r;
  }
#if MK_HAVE_DUAL
  if (st.flags & MK_F_ROW_NORM) {
#pragma unroll
    for (int j = 0; j < R; j++)
      if (R == 2 || j * 64 < D) h.x[j] = (h.x[j] * h.r) * h.w[j];
  }
#endif
#pragma unroll
  for (int j = 0; j < R; j++)
    if (j * 64 + lane < D) put(j * 64 + lane, h.x[j]);
}

// Cache layout, chosen for the matrix cores (a page is page_size positions of all kv heads):
//   K  [position / 16][kv head][dim / KW][64 lanes][EPC]: lane l holds position l % 16, dims (l / 16) * EPC .. of the KW;
//   V  [position / TP][kv head][dim / 16][64 lanes][EPC]: lane l holds dim l % 16, positions 4 (l / 16) .. + 3 of each
//      16-position sub-tile (sub-tile u in elements 4 u .. 4 u + 3).
// Every operand of a tile is then one contiguous 1 KB request, with no transpose on the way.  Dims are padded with zeros.
template <typename E>
__device__ __forceinline__ size_t fx_k_at(int page, int pp, int ps, int nkv, int g, int nkc, int d) {
  constexpr int EPC = FxType<E>::EPC, KW = FxType<E>::KW;
  return ((((((size_t)page * ps + pp) / 16) * nkv + g) * nkc + d / KW) * 64 + ((d % KW) / EPC) * 16 + (pp & 15)) * EPC + (d % EPC);
}
template <typename E>
__device__ __forceinline__ size_t fx_v_at(int page, int pp, int ps, int nkv, int g, int nvb, int d) {
  constexpr int EPC = FxType<E>::EPC, TP = FxType<E>::TP;
  return ((((((size_t)page * ps + pp) / TP) * nkv + g) * nvb + d / 16) * 64 + ((pp & 15) >> 2) * 16 + (d & 15)) * EPC + ((pp % TP) / 16) * 4 + (pp & 3);
}

// Column the value heads begin at (hybrid kernels: the keys' where a model's values are its keys before rotation).
__device__ __forceinline__ int fx_value_col(CStage &st) {
#if MK_HAVE_HYB
  return st.v_col;
#else
  return (st.num_q_heads + st.num_kv_heads) * st.head_dim;
#endif
}

// Query, key and value rows of an iteration in which some request brings several tokens: a wavefront per (token, head)
// row.  Queries go to the workspace, keys and values to their pages.  (When every request brings one token the attention
// stage does this itself and the stage is skipped.)
template <typename E>
__device__ __forceinline__ void stage_fx_prep(CStage &st, Ctx &c, const MkRuntime &rt, int M, char *smem) {
  barrier_wait(c);
  constexpr int KW = FxType<E>::KW;
  const FxRows<E> rows = fx_rows<E>(st, c);
  const int lane = c.tid & 63, wave = __builtin_amdgcn_readfirstlane(c.tid >> 6);
  const int H = st.num_q_heads, nkv = st.num_kv_heads, D = st.head_dim, DV = st.v_dim;
  const int nkc = (D + KW - 1) / KW, nvb = (DV + 15) / 16, ps = rt.page_size;
  const int per = H + 2 * nkv, total = M * per;
  E *kc = (E *)st.k_cache, *vc = (E *)st.v_cache;
  const int stride = c.G * MK_WAVES;
  float *xs = (float *)smem + wave * MK_FX_MAX_HEAD_DIM;
  fx_head_regs(D, DV, [&](auto regs) {
    constexpr int R = decltype(regs)::value;
    auto span = [&](int i, FxHead<R> &h, int &page) -> FxSpan {
      const int t = i / per, s = i - t * per;
      const int pos = __builtin_amdgcn_readfirstlane(c.sh_tok[t]);
      page = s < H ? 0 : rt.kv_indices[__builtin_amdgcn_readfirstlane(c.sh_tok[3 * MK_MAX_TOKENS + t]) + pos / ps];
      const bool head = s < H + nkv;
      const FxSpan sp = {t, head ? s * D : fx_value_col(st) + (s - H - nkv) * DV, head ? D : DV};
      fx_head_tables(st, rows, sp, head, pos, lane, h);
#if MK_HAVE_DUAL
      if (head && (st.flags & MK_F_ROW_NORM)) {
        const int c0 = s < H ? 0 : H * D, c1 = s < H ? H * D : (H + nkv) * D;
        fx_row_weights(st, s * D, lane, h);
        h.r = 1.f / sqrtf(wave_sum(fx_row_squares<E>((const E *)st.in + (size_t)t * st.ld_in, c0, c1, lane, 64)) / (float)(c1 - c0) + st.eps);
      }
#endif
      return sp;
    };
    auto finish = [&](int i, FxHead<R> &h, int page) {
      const int t = i / per, s = i - t * per;
      const int pp = __builtin_amdgcn_readfirstlane(c.sh_tok[t]) % ps;
      if (s < H) {
        E *q = (E *)st.q_ws + (size_t)t * st.ld_qws + (size_t)s * nkc * KW;
        fx_head_finish(st, lane, h, xs, [&](int d, float v) { fx_stc(q + d, fx_round<E>(v)); });
        for (int d = D + lane; d < nkc * KW; d += 64) fx_stc(q + d, (E)0);
      } else if (s < H + nkv) {
        fx_head_finish(st, lane, h, xs, [&](int d, float v) { fx_stc(kc + fx_k_at<E>(page, pp, ps, nkv, s - H, nkc, d), fx_round<E>(v)); });
      } else {
        const int g = s - H - nkv;
#pragma unroll
        for (int j = 0; j < R; j++)
          if (j * 64 + lane < DV) fx_stc(vc + fx_v_at<E>(page, pp, ps, nkv, g, nvb, j * 64 + lane), fx_round<E>(fx_value(h, j)));
      }
    };
    for (int i = c.vid * MK_WAVES + wave; i < total; i += 2 * stride) {
      FxHead<R> h0, h1;
      int p0, p1;
      const int i1 = i + stride < total ? i + stride : i;
      const FxSpan s0 = span(i, h0, p0), s1 = span(i1, h1, p1);
      fx_span_load2(rows, s0, s1, lane, h0, h1);
      finish(i, h0, p0);
      if (i1 != i) finish(i1, h1, p1);
    }
  });
  c.wrote_through = true;
}

#if MK_PAIR
// The rows of several portions, none of which leaves its rows to the attention: a wavefront stays with one portion, whose tokens are a lane each, and has as
// many rows in flight as registers allow (two at a time, portion by portion: six portions of 64 rows of 32 q / 8 kv heads of 128, from four slices, 30 us, now 19).
template <typename E>
__device__ __forceinline__ void stage_fx_prep_group(Ctx &c, const MkRuntime &rt, int s, int portions, const int *sh_rows, char *smem) {
  constexpr int KW = FxType<E>::KW;
  const int lane = c.tid & 63, wave = __builtin_amdgcn_readfirstlane(c.tid >> 6), W = c.vid * MK_WAVES + wave, n_waves = c.G * MK_WAVES;
  const int p = W % portions, first = W / portions, step = (n_waves - p + portions - 1) / portions, M = __builtin_amdgcn_readfirstlane(sh_rows[p]);
  CStage &st = mk_portion_stages(rt, p)[s];
  const int H = st.num_q_heads, nkv = st.num_kv_heads, D = st.head_dim, DV = st.v_dim;
  const int nkc = (D + KW - 1) / KW, nvb = (DV + 15) / 16, ps = rt.page_size, per = H + 2 * nkv, total = M * per;
  const int row = p * MK_MAX_TOKENS + min(lane, M - 1), my_pos = ldc_i32(&rt.tok_pos[row]);
  const int my_page = rt.kv_indices[(rt.batch_n ? rt.batch_at[p] : 0) + ldc_i32(&rt.kv_indptr[ldc_i32(&rt.tok_slot[row])]) + my_pos / ps];
  E *kc = (E *)st.k_cache, *vc = (E *)st.v_cache;
  float *xs = (float *)smem + wave * MK_FX_MAX_HEAD_DIM;
  barrier_wait(c);
  FxRows<E> rows = fx_rows<E>(st, c);
  if (rows.S) rows.part += (size_t)p * MK_MAX_TOKENS * rows.ldp;
  fx_head_regs(D, DV, [&](auto regs) {
    constexpr int R = decltype(regs)::value, N = R == 2 ? 6 : 2;
    for (int i0 = first; i0 < total; i0 += N * step) {
      FxHead<R> h[N];
      FxSpan sp[N];
#pragma unroll
      for (int z = 0; z < N; z++) {
        const int i = min(i0 + z * step, total - 1), t = i / per, q = i - t * per;
        const bool head = q < H + nkv;
        sp[z] = {t, head ? q * D : fx_value_col(st) + (q - H - nkv) * DV, head ? D : DV};
        fx_head_tables(st, rows, sp[z], head, __builtin_amdgcn_readlane(my_pos, t), lane, h[z]);
#if MK_HAVE_DUAL
        if (head && (st.flags & MK_F_ROW_NORM)) {
          const int c0 = q < H ? 0 : H * D, c1 = q < H ? H * D : (H + nkv) * D;
          fx_row_weights(st, q * D, lane, h[z]);
          h[z].r = 1.f / sqrtf(wave_sum(fx_row_squares<E>((const E *)st.in + (size_t)t * st.ld_in, c0, c1, lane, 64)) / (float)(c1 - c0) + st.eps);
        }
#endif
      }
      fx_span_loads<E, R, N>(rows, sp, lane, h);
#pragma unroll
      for (int z = 0; z < N; z++) {
        const int i = i0 + z * step, t = sp[z].tok, q = i - t * per;
        if (i >= total) break;
        const int page = __builtin_amdgcn_readlane(my_page, t), pp = __builtin_amdgcn_readlane(my_pos, t) % ps;
        if (q < H) {
          E *to = (E *)st.q_ws + (size_t)t * st.ld_qws + (size_t)q * nkc * KW;
          fx_head_finish(st, lane, h[z], xs, [&](int d, float v) { fx_stc(to + d, fx_round<E>(v)); });
          for (int d = D + lane; d < nkc * KW; d += 64) fx_stc(to + d, (E)0);
        } else if (q < H + nkv) {
          fx_head_finish(st, lane, h[z], xs, [&](int d, float v) { fx_stc(kc + fx_k_at<E>(page, pp, ps, nkv, q - H, nkc, d), fx_round<E>(v)); });
        } else {
#pragma unroll
          for (int j = 0; j < R; j++)
            if (j * 64 + lane < DV) fx_stc(vc + fx_v_at<E>(page, pp, ps, nkv, q - H - nkv, nvb, j * 64 + lane), fx_round<E>(fx_value(h[z], j)));
        }
      }
    }
  });
  c.wrote_through = true;
}
#endif

// ----------------------------------------------------------------------------- attention
__device__ __forceinline__ f32x4 fx_mma_k(uint16_t, u32x4 a, u32x4 b, f32x4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}
__device__ __forceinline__ f32x4 fx_mma_k(float, u32x4 a, u32x4 b, f32x4 acc) {
#pragma unroll
  for (int j = 0; j < 4; j++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[j]), __uint_as_float(b[j]), acc, 0, 0, 0);
  return acc;
}
__device__ __forceinline__ float fx_exp2(uint16_t, float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fx_exp2(float, float x) { return exp2f(x); }

// Work unit = (16 query rows of one request and kv head, slice of VB * 16 value dims, chunk of the cached positions).  A
// query row is a (token, query head of the group) pair, tokens outermost.  The wavefronts of a workgroup take every fourth
// tile of TP positions: scores = K tile x query rows (positions in the rows of the result), so a lane's four results per
// sub-tile are exactly its operand of the product with V (bf16: as value + rounding remainder, which keeps about 16
// mantissa bits of the weights).  Running maximum and sum per query row and wavefront; wavefronts are merged through LDS,
// chunks through the partial buffer by the last workgroup to arrive.  The sink enters once, in the final division.
//
// `single`: every request of the iteration brings one token.  The stage then rotates, normalises and appends the new rows
// itself (the chunk that owns the new position takes its key and value from LDS, nothing of the iteration is read back
// from memory), and the first tiles' rows, which earlier iterations wrote, are requested before the barrier is awaited.
// Otherwise the prep stage has written queries, keys and values.
#define MK_FX_NEG (-1e30f)
// Chunks a unit of NT tiles is split into: none while every wavefront has at most two tiles (a hand-over costs about as
// much), else one tile per wavefront, and two once that would make more than 16 chunks to combine.
__device__ __forceinline__ int fx_chunks(int NT, int cmax) {
  const int rounds = (NT + MK_WAVES - 1) / MK_WAVES;  // tiles of the busiest wavefront without a split
  return rounds <= 2 ? 1 : min(cmax, rounds <= 16 ? rounds : max(16, (rounds + 1) / 2));
}
template <typename E, int KC, int VB>
__device__ __forceinline__ void stage_fx_attn_t(CStage &st, Ctx &c, const MkRuntime &rt, int M, bool single, char *smem) {
  using X = FxType<E>;
  constexpr int EPC = X::EPC, KW = X::KW, TP = X::TP, SUB = X::SUB;
  constexpr int PSTR = VB * 16 + 4, PST = VB * 16 + 32;
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int nkv = st.num_kv_heads, qpk = st.num_q_heads / nkv, D = st.head_dim, DV = st.v_dim;
  const int nkc = (D + KW - 1) / KW, nkg = (nkc + KC - 1) / KC, nvb = (DV + 15) / 16, nvs = (nvb + VB - 1) / VB;
  const int ps = rt.page_size;
  const u32x4 *kc = (const u32x4 *)st.k_cache, *vc = (const u32x4 *)st.v_cache;
#if MK_PAIR
  // (portions follow each other without a barrier: each has scratch of its own)
  float *const part_base = rt.group_attn_part + (size_t)c.portion * rt.group_attn;
  unsigned *const cnt_base = rt.group_attn_cnt + (size_t)c.portion * rt.group_cnt * 32;
#else
  float *const part_base = (float *)rt.attn_part;
  unsigned *const cnt_base = rt.attn_cnt;
#endif
  // LDS
  u32x4 *qs = (u32x4 *)smem;                                   // [nkg * KC][64] query operands
  E *kn = (E *)(smem + nkg * KC * 1024);                       // new key, padded with zeros to nkc * KW
  E *vn = kn + nkc * KW;                                       // new value, padded with zeros to nvb * 16
  float *part = (float *)(smem + (nkg * KC * 1024 + (nkc * KW + nvb * 16) * (int)sizeof(E) + 15) / 16 * 16);  // [4][16][PSTR]
  float *ml = part + MK_WAVES * 16 * PSTR;                     // [4][16] maxima, [4][16] sums
  float *fin = ml + 128;                                       // [4][16] weights
  int *sflag = (int *)(fin + 96);
  int *spg = sflag + 4;                                        // page-table entries of the chunk
  // rows of the requests, in row tiles of 16
  int my_n, my_tiles;
  {
    const bool first = lane < M && c.sh_tok[2 * MK_MAX_TOKENS + lane] == lane;
    const unsigned long long fm = __ballot(first), later = lane < 63 ? fm >> (lane + 1) : 0ull;
    my_n = first ? (later ? (int)__ffsll(later) : M - lane) : 0;
    my_tiles = (my_n * qpk + 15) / 16;
  }
  const int tiles_incl = wave_incl_scan(my_tiles, lane);
  const int RT = wave_bcast(tiles_incl, 63);
  const int n_items = RT * nkv * nvs;
  const int cmax = max(1, min(c.G / n_items, MK_ATTN_MAX_CHUNKS));
  const int n_units = n_items * cmax;
  struct Unit {
    int item, cidx, C, g, vs, t0, r0, nrows, p0, p, tb, te, pages, kept, gap;
  };
  // Tiles of a unit are counted without those that none of its rows sees: with a window, `kept` first ones, then `gap` left out.
  const int win = MK_HAVE_HYB ? st.window : 0, keep = MK_HAVE_HYB ? st.keep_first : 0;
  auto phys = [](const Unit &a, int tile) { return MK_HAVE_HYB && tile >= a.kept ? tile + a.gap : tile; };
  auto decode = [&](int u, Unit &a) -> bool {
    a.item = u / cmax;
    a.cidx = u - a.item * cmax;
    a.g = a.item / (RT * nvs);  // kv head outermost: its units sit on adjacent workgroups, i.e. on one die
    const int rem = a.item - a.g * RT * nvs;
    a.vs = rem / RT;
    const int tile = rem - a.vs * RT;
    a.t0 = (int)__ffsll(__ballot(tiles_incl > tile)) - 1;
    const int n = wave_bcast(my_n, a.t0);
    a.r0 = (tile - (wave_bcast(tiles_incl, a.t0) - wave_bcast(my_tiles, a.t0))) * 16;
    a.nrows = min(16, n * qpk - a.r0);
    a.p0 = __builtin_amdgcn_readfirstlane(c.sh_tok[a.t0]);
    a.p = a.p0 + (a.r0 + a.nrows - 1) / qpk;  // newest position any of the rows sees
    int NT = a.p / TP + 1;
    if (MK_HAVE_HYB) {
      const int first = a.p0 + a.r0 / qpk;  // position of the unit's first row
      int oldest = win ? max(0, first - win + 1) : 0;  // oldest position inside its window
#if MK_HAVE_DUAL
      if (st.chunk) oldest = max(oldest, first - first % st.chunk);  // ... and inside its chunk
      a.kept = win || st.chunk ? min((keep + TP - 1) / TP, NT) : NT;
#else
      a.kept = win ? min((keep + TP - 1) / TP, NT) : NT;
#endif
      a.gap = max(0, oldest / TP - a.kept);
      NT -= a.gap;
    }
    a.C = fx_chunks(NT, cmax);
    if (a.cidx >= a.C) return false;
    a.tb = (int)(((long long)NT * a.cidx) / a.C);
    a.te = (int)(((long long)NT * (a.cidx + 1)) / a.C);
    a.pages = __builtin_amdgcn_readfirstlane(c.sh_tok[3 * MK_MAX_TOKENS + a.t0]);
    return true;
  };
  // operands of tile `tile`, dim group kg (page: its page-table entry).  !ok: the same number of loads from one spot.
  auto load_tile = [&](const Unit &a, int tile, int kg, int page, bool ok, u32x4 (&k)[SUB][KC], u32x4 (&v)[VB]) {
    const int pp = (tile * TP) % ps;
    const size_t pt = (size_t)page * ps + pp;
    const u32x4 *kp = kc + (ok ? ((pt / 16) * nkv + a.g) * nkc * 64 : 0) + lane;
    const u32x4 *vp = vc + (ok ? ((pt / TP) * nkv + a.g) * nvb * 64 : 0) + lane;
    const int on = ok ? 64 : 0, su = ok ? nkv * nkc * 64 : 0;
#pragma unroll
    for (int u = 0; u < SUB; u++)
#pragma unroll
      for (int s = 0; s < KC; s++) k[u][s] = kp[u * su + min(kg * KC + s, nkc - 1) * on];
#pragma unroll
    for (int b = 0; b < VB; b++) v[b] = vp[min(a.vs * VB + b, nvb - 1) * on];
  };
  u32x4 kA[SUB][KC], vA[VB], kB[SUB][KC], vB[VB];
  Unit a0;
  const bool have0 = c.vid < n_units && decode(c.vid, a0);
  auto load_first = [&](const Unit &a) {
    const int tile = a.tb + wave;
    const bool ok = tile < a.te;
    const int page = rt.kv_indices[a.pages + phys(a, ok ? tile : a.tb) * TP / ps];
    load_tile(a, phys(a, tile), 0, page, ok, kA, vA);
  };
  const bool early = single && have0 && wave != 0;  // (the polling wavefront keeps its memory queue empty)
  if (early) load_first(a0);
  // (Keys and values are read with cached loads.  Where some request brings several tokens, nothing of this layer's cache is requested before the
  // barrier behind the stage that writes the new positions.  Where every request brings one, tiles are requested early, and a line with the
  // new position may be cached as it was before: that position always comes from LDS, and the next iteration opens with an invalidate.)
  barrier_wait(c);
  c.wrote_through = true;
  FxRows<E> rows{};
  if (single) rows = fx_rows<E>(st, c);
  const float cap = st.softcap, sc1 = cap > 0.f ? st.sm_scale / cap : st.sm_scale;
  const float LOG2E = 1.4426950408889634f;

  for (int uu = c.vid; uu < n_units; uu += c.G) {
    Unit a;
    const bool first = uu == c.vid;
    int u = uu;
    if (cmax == 1 && ((uu / c.G) & 1)) {  // every other round deals the units in reverse order (contexts differ)
      const int b0 = (uu / c.G) * c.G, bn = min(c.G, n_units - b0);
      u = b0 + bn - 1 - (uu - b0);
    }
    if (first) {
      if (!have0) continue;
      a = a0;
    } else if (!decode(u, a)) {
      continue;
    }
    if (!(first && early)) load_first(a);
    __syncthreads();  // LDS reuse across units
    const int pg_lo = phys(a, a.tb) * TP / ps, npg = min((phys(a, a.te - 1) * TP + TP - 1) / ps, a.p / ps) - pg_lo + 1;
    for (int i = tid; i < npg; i += MK_THREADS) spg[i] = rt.kv_indices[a.pages + pg_lo + i];
    const bool newest = single && a.cidx == a.C - 1;
    // ---- query rows into operand order (and the new key and value)
    if (single) {
#if MK_HAVE_DUAL
      float rq = 0.f, rk = 0.f;
      if (st.flags & MK_F_ROW_NORM) {
        const int nq = st.num_q_heads * D, nk = nkv * D;
        const E *row = (const E *)st.in + (size_t)a.t0 * st.ld_in;
        rq = fx_row_squares<E>(row, 0, nq, tid, MK_THREADS);
        if (newest) rk = fx_row_squares<E>(row, nq, nq + nk, tid, MK_THREADS);
        rq = wave_sum(rq);
        rk = wave_sum(rk);
        if (lane == 0) {
          part[wave] = rq;
          part[4 + wave] = rk;
        }
        __syncthreads();
        rq = 1.f / sqrtf(((part[0] + part[1]) + (part[2] + part[3])) / (float)nq + st.eps);
        rk = 1.f / sqrtf(((part[4] + part[5]) + (part[6] + part[7])) / (float)nk + st.eps);
      }
#endif
      // (everything the row writers below leave out is zeroed: unused query columns, padding dims)
      const u32x4 z = {0u, 0u, 0u, 0u};
      for (int i = tid; i < nkg * KC * 64; i += MK_THREADS)
        if ((i & 15) >= a.nrows || (i >> 6) >= nkc) qs[i] = z;
      E *q = (E *)qs;
      for (int i = tid; i < 16 * (nkc * KW - D); i += MK_THREADS) {
        const int d = D + i / 16;
        if ((i & 15) < a.nrows) q[((d / KW) * 64 + ((d % KW) / EPC) * 16 + (i & 15)) * EPC + d % EPC] = (E)0;
      }
      for (int i = D + tid; i < nkc * KW; i += MK_THREADS) kn[i] = (E)0;
      for (int i = DV + tid; i < nvb * 16; i += MK_THREADS) vn[i] = (E)0;
      // rows 0 .. nrows - 1 are queries, the next two (the chunk that owns the new position) the new key and value.  The first
      // wavefront takes some only where that saves the others a round: its tile was requested last, and loads arrive in order.
      const int n_rows = a.nrows + (newest ? 2 : 0);
      const int RW = (n_rows + 2 * MK_WAVES - 3) / (2 * MK_WAVES - 2) > (n_rows + 2 * MK_WAVES - 1) / (2 * MK_WAVES) ? MK_WAVES : MK_WAVES - 1;
      float *xs = part + 16 + wave * MK_FX_MAX_HEAD_DIM;
      fx_head_regs(D, DV, [&](auto regs) {
        constexpr int R = decltype(regs)::value;
        auto span = [&](int r, FxHead<R> &h) -> FxSpan {
          const bool head = r <= a.nrows;
          const FxSpan sp = {a.t0, head ? (r < a.nrows ? a.g * qpk + a.r0 + r : st.num_q_heads + a.g) * D : fx_value_col(st) + a.g * DV, head ? D : DV};
          fx_head_tables(st, rows, sp, head, a.p, lane, h);
#if MK_HAVE_DUAL
          if (head) fx_row_weights(st, sp.col, lane, h);
          h.r = r < a.nrows ? rq : rk;
#endif
          return sp;
        };
        auto put_row = [&](int r, FxHead<R> &h) {
          if (r < a.nrows) {
            fx_head_finish(st, lane, h, xs, [&](int d, float v) { q[((d / KW) * 64 + ((d % KW) / EPC) * 16 + r) * EPC + d % EPC] = fx_round<E>(v); });
          } else if (r == a.nrows) {
            fx_head_finish(st, lane, h, xs, [&](int d, float v) { kn[d] = fx_round<E>(v); });
          } else {
#pragma unroll
            for (int j = 0; j < R; j++)
              if (j * 64 + lane < DV) vn[j * 64 + lane] = fx_round<E>(fx_value(h, j));
          }
        };
        if (wave != 0 || RW == MK_WAVES)
          for (int r = MK_WAVES - 1 - wave; r < n_rows; r += 2 * RW) {
            FxHead<R> h0, h1;
            const int r1 = r + RW < n_rows ? r + RW : r;
            const FxSpan s0 = span(r, h0), s1 = span(r1, h1);
            fx_span_load2(rows, s0, s1, lane, h0, h1);
            put_row(r, h0);
            if (r1 != r) put_row(r1, h1);
          }
      });
    } else {
      for (int i = tid; i < nkg * KC * 64; i += MK_THREADS) {
        const int s = i >> 6, r = i & 15, R = a.r0 + r;
        u32x4 v = {0u, 0u, 0u, 0u};
        if (r < a.nrows && s < nkc)
          v = ldc_16B((const u32x4 *)((const E *)st.q_ws + (size_t)(a.t0 + R / qpk) * st.ld_qws + (size_t)(a.g * qpk + R % qpk) * nkc * KW + s * KW +
                                      ((i & 63) >> 4) * EPC));
        qs[i] = v;
      }
    }
    __syncthreads();
    if (newest && a.r0 == 0 && a.vs == 0) {  // append the new rows to their page
      const int pp = a.p % ps, page = spg[a.p / ps - pg_lo];
      for (int i = tid; i < nkc * 4; i += MK_THREADS)
        stc_16B((u32x4 *)st.k_cache + (((((size_t)page * ps + pp) / 16) * nkv + a.g) * nkc + (i >> 2)) * 64 + (i & 3) * 16 + (pp & 15), ((const u32x4 *)kn)[i]);
      for (int d = tid; d < DV; d += MK_THREADS) fx_stc((E *)st.v_cache + fx_v_at<E>(page, pp, ps, nkv, a.g, nvb, d), vn[d]);
    }
    // ---- tiles
    const int plim = a.p0 + (a.r0 + min(lr, a.nrows - 1)) / qpk;  // newest position this lane's query row sees
#if MK_HAVE_DUAL
    const int olim = st.chunk ? plim - plim % st.chunk : 0;  // oldest one
    const float sc_row = sc1 * (st.temp ? st.temp[a.g * qpk + (a.r0 + min(lr, a.nrows - 1)) % qpk] : 1.f);
#else
    const float sc_row = sc1;
#endif
    float m = MK_FX_NEG, l = 0.f;
    f32x4 acc[VB], S[SUB];
#pragma unroll
    for (int b = 0; b < VB; b++) acc[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int n_mine = a.te - a.tb > wave ? (a.te - a.tb - wave + MK_WAVES - 1) / MK_WAVES : 0;
    auto compute = [&](int tile, int kg, u32x4 (&k)[SUB][KC], u32x4 (&v)[VB]) {
      const bool has_new = single && tile == a.p / TP;
      if (has_new) {
        const u32x4 *kn4 = (const u32x4 *)kn;
#pragma unroll
        for (int u_ = 0; u_ < SUB; u_++)
          if (u_ == (a.p % TP) / 16) {
#pragma unroll
            for (int s = 0; s < KC; s++) {
              const u32x4 x = kn4[min(kg * KC + s, nkc - 1) * 4 + lg];
              if (lr == (a.p & 15)) k[u_][s] = x;
            }
          }
      }
      if (kg == 0) {
#pragma unroll
        for (int u_ = 0; u_ < SUB; u_++) S[u_] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int s = 0; s < KC; s++) {
        const u32x4 q = qs[(kg * KC + s) * 64 + lane];
#pragma unroll
        for (int u_ = 0; u_ < SUB; u_++) S[u_] = fx_mma_k(E(), k[u_][s], q, S[u_]);
      }
      if (kg + 1 < nkg) return;
      float sc[SUB][4];
      float tm = MK_FX_NEG;
      auto each = [&](auto f) {
#pragma unroll
        for (int u_ = 0; u_ < SUB; u_++)
#pragma unroll
          for (int i = 0; i < 4; i++) f(sc[u_][i], S[u_][i] * sc_row);
      };
      // (one branch for all values: with one at every value they follow each other)
      if (cap > 0.f) {
        if constexpr (sizeof(E) == 2) {
          each([&](float &s, float x) { s = __builtin_amdgcn_exp2f(x * (2.f * LOG2E)); });
          each([&](float &s, float x) { s = (cap * LOG2E) * (1.f - 2.f * __builtin_amdgcn_rcpf(1.f + s)); });
        } else {
          each([&](float &s, float x) { s = (cap * LOG2E) * tanhf(x); });
        }
      } else {
        each([&](float &s, float x) { s = x * LOG2E; });
      }
#pragma unroll
      for (int u_ = 0; u_ < SUB; u_++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float s = sc[u_][i];
          const int at = tile * TP + u_ * 16 + lg * 4 + i;
          bool seen = at <= plim;
          if (MK_HAVE_HYB) seen = seen && (win == 0 || plim - at < win || at < keep);
#if MK_HAVE_DUAL
          seen = seen && at >= olim;
#endif
          s = seen ? s : MK_FX_NEG;
          sc[u_][i] = s;
          tm = fmaxf(tm, s);
        }
      tm = groups_max(tm);
      if (__any(tm > m)) {
        const float nm = fmaxf(m, tm), corr = fx_exp2(E(), m - nm);
        m = nm;
        l *= corr;
#pragma unroll
        for (int b = 0; b < VB; b++) acc[b] *= corr;
      }
#pragma unroll
      for (int u_ = 0; u_ < SUB; u_++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          sc[u_][i] = sc[u_][i] > 0.5f * MK_FX_NEG ? fx_exp2(E(), sc[u_][i] - m) : 0.f;
          l += sc[u_][i];
        }
      if (has_new) {
#pragma unroll
        for (int b = 0; b < VB; b++) {
          const E x = vn[min(a.vs * VB + b, nvb - 1) * 16 + lr];
          const int slot = ((a.p % TP) / 16) * 4 + (a.p & 3);
#pragma unroll
          for (int w = 0; w < 4; w++) {
            uint32_t nv;
            bool here;
            if constexpr (sizeof(E) == 2) {
              here = w == (slot >> 1);
              nv = (slot & 1) ? (v[b][w] & 0xffffu) | ((uint32_t)x << 16) : (v[b][w] & 0xffff0000u) | (uint32_t)x;
            } else {
              here = w == slot;
              nv = __float_as_uint(x);
            }
            if (here && lg == ((a.p & 15) >> 2)) v[b][w] = nv;
          }
        }
      }
      if ((tile + 1) * TP - 1 > a.p) {  // values behind the newest position belong to nobody: whatever they are, 0 x them is 0
#pragma unroll
        for (int b = 0; b < VB; b++)
#pragma unroll
          for (int w = 0; w < 4; w++) {
            if constexpr (sizeof(E) == 2) {
              const int q = tile * TP + (w >> 1) * 16 + lg * 4 + (w & 1) * 2;
              v[b][w] = q > a.p ? 0u : (q + 1 > a.p ? v[b][w] & 0xffffu : v[b][w]);
            } else {
              if (tile * TP + lg * 4 + w > a.p) v[b][w] = 0u;
            }
          }
      }
      if constexpr (sizeof(E) == 2) {
        u32x4 hi, lo;
#pragma unroll
        for (int w = 0; w < 4; w++) {
          const float x0 = sc[w >> 1][(w & 1) * 2], x1 = sc[w >> 1][(w & 1) * 2 + 1];
          hi[w] = pack2(x0, x1);
          lo[w] = pack2(x0 - bf_lo(hi[w]), x1 - bf_hi(hi[w]));
        }
#pragma unroll
        for (int b = 0; b < VB; b++) {
          acc[b] = fx_mma_k(E(), v[b], hi, acc[b]);
          acc[b] = fx_mma_k(E(), v[b], lo, acc[b]);
        }
      } else {
        u32x4 pw;
#pragma unroll
        for (int w = 0; w < 4; w++) pw[w] = __float_as_uint(sc[0][w]);
#pragma unroll
        for (int b = 0; b < VB; b++) acc[b] = fx_mma_k(E(), v[b], pw, acc[b]);
      }
    };
    const int n_it = n_mine * nkg;
    int tile = a.tb + wave, kg = 0;
    auto next = [&](int &tl, int &kk) {
      if (++kk == nkg) {
        kk = 0;
        tl += MK_WAVES;
      }
    };
    for (int it = 0; it < n_it; it += 2) {
      int tl = tile, kk = kg;
      next(tl, kk);
      bool ok = it + 1 < n_it;
      load_tile(a, phys(a, tl), kk, ok ? spg[phys(a, tl) * TP / ps - pg_lo] : 0, ok, kB, vB);
      compute(phys(a, tile), kg, kA, vA);
      if (!ok) break;
      tile = tl;
      kg = kk;
      next(tl, kk);
      ok = it + 2 < n_it;
      load_tile(a, phys(a, tl), kk, ok ? spg[phys(a, tl) * TP / ps - pg_lo] : 0, ok, kA, vA);
      compute(phys(a, tile), kg, kB, vB);
      tile = tl;
      kg = kk;
    }
    // ---- wavefronts of the workgroup
    l = groups_sum(l);
#pragma unroll
    for (int b = 0; b < VB; b++) *(f32x4 *)(part + (wave * 16 + lr) * PSTR + b * 16 + lg * 4) = acc[b];
    if (lg == 0) {
      ml[wave * 16 + lr] = m;
      ml[64 + wave * 16 + lr] = l;
    }
    __syncthreads();
    const float *sink = (const float *)st.sink;
    auto sink_of = [&](int r) -> float { return sink ? sink[a.g * qpk + (a.r0 + min(r, a.nrows - 1)) % qpk] * LOG2E : -INFINITY; };
    if (tid < 16) {
      float M_ = MK_FX_NEG, L_ = 0.f;
#pragma unroll
      for (int w = 0; w < MK_WAVES; w++) M_ = fmaxf(M_, ml[w * 16 + tid]);
#pragma unroll
      for (int w = 0; w < MK_WAVES; w++) {
        const float e = exp2f(ml[w * 16 + tid] - M_);
        fin[w * 16 + tid] = e;
        L_ += ml[64 + w * 16 + tid] * e;
      }
      if (a.C == 1) {
        const float inv = 1.f / (L_ + exp2f(sink_of(tid) - M_));
#pragma unroll
        for (int w = 0; w < MK_WAVES; w++) fin[w * 16 + tid] *= inv;
      } else {
        float *pb = part_base + ((size_t)u * 16 + tid) * PST + VB * 16;
        stc_f32(pb, M_);
        stc_f32(pb + 1, L_);
      }
    }
    __syncthreads();
    const int dv0 = a.vs * VB * 16;
    auto emit = [&](int r, int d, const f32x4 &o) {
      const int R = a.r0 + r;
      E *row = (E *)st.out + (size_t)(a.t0 + R / qpk) * st.ld_out + (size_t)(a.g * qpk + R % qpk) * DV;
      const float q[4] = {o[0], o[1], o[2], o[3]};
      fx_stc4(row, dv0 + d, DV, q);
    };
    for (int i = tid; i < 16 * VB * 4; i += MK_THREADS) {
      const int r = i / (VB * 4), d = (i - r * (VB * 4)) * 4;
      if (r >= a.nrows || dv0 + d >= DV) continue;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < MK_WAVES; w++) o += *(const f32x4 *)(part + (w * 16 + r) * PSTR + d) * fin[w * 16 + r];
      if (a.C == 1) emit(r, d, o);
      else stc_16B((u32x4 *)(part_base + ((size_t)u * 16 + r) * PST + d), __builtin_bit_cast(u32x4, o));
    }
    if (a.C == 1) continue;
    // ---- chunks: the last workgroup to arrive combines them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      unsigned *cnt = cnt_base + (size_t)a.item * 32;
      const int last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(a.C - 1);
      if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *sflag = last;
    }
    __syncthreads();
    if (!*sflag) continue;
    // Every thread weighs the chunks of its query row itself: maxima, sums and partial results of up to sixteen chunks are one round trip
    // (weights by way of LDS had made it two and three barriers).
    const float *pb = part_base + (size_t)a.item * cmax * 16 * PST;
    constexpr int CB = 16;
    static_assert(MK_ATTN_MAX_CHUNKS <= 2 * CB, "at most two blocks of chunks");
    for (int i = tid; i < 16 * VB * 4; i += MK_THREADS) {
      const int r = i / (VB * 4), d = (i - r * (VB * 4)) * 4;
      if (r >= a.nrows || dv0 + d >= DV) continue;
      float cm[CB], cl[CB];
      f32x4 x[CB];
      auto request = [&](int q0, bool data) {
#pragma unroll
        for (int q = 0; q < CB; q++)
          if (q0 + q < a.C) {
            const float *p = pb + ((size_t)(q0 + q) * 16 + r) * PST;
            const unsigned long long u = ldc_u64(p + VB * 16);
            cm[q] = __uint_as_float((uint32_t)u);
            cl[q] = __uint_as_float((uint32_t)(u >> 32));
            if (data) x[q] = fx_ldc_quad(p + d);
          }
      };
      float M_ = MK_FX_NEG, L_ = 0.f;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
      auto largest = [&](int q0) {
#pragma unroll
        for (int q = 0; q < CB; q++)
          if (q0 + q < a.C) M_ = fmaxf(M_, cm[q]);
      };
      if (a.C > CB) {
        request(CB, false);
        largest(CB);
      }
      request(0, true);
      largest(0);
      for (int q0 = 0; q0 < a.C; q0 += CB) {
        if (q0) request(q0, true);
#pragma unroll
        for (int q = 0; q < CB; q++)
          if (q0 + q < a.C) {
            const float e = exp2f(cm[q] - M_);
            L_ += cl[q] * e;
            o += x[q] * e;
          }
      }
      emit(r, d, o * (1.f / (L_ + exp2f(sink_of(r) - M_))));
    }
  }
}
#if MK_PAIR
// Four tiles of dims' sums, first with the rounded weights, then with their remainders.  In assembly, as in add_products.
__device__ __forceinline__ void fx_add_products(f32x4 &o0, f32x4 &o1, f32x4 &o2, f32x4 &o3, u32x4 v0, u32x4 v1, u32x4 v2, u32x4 v3, u32x4 hi, u32x4 lo) {
#define MK_PV(o, w) "v_mfma_f32_16x16x32_bf16 %" #o ", %[v" #o "], %[" #w "], %" #o "\n\t"
  asm volatile("s_nop 3\n\t" MK_PV(0, hi) MK_PV(1, hi) MK_PV(2, hi) MK_PV(3, hi) MK_PV(0, lo) MK_PV(1, lo) MK_PV(2, lo) MK_PV(3, lo) "s_nop 11"
               : "+v"(o0), "+v"(o1), "+v"(o2), "+v"(o3)
               : [v0] "v"(v0), [v1] "v"(v1), [v2] "v"(v2), [v3] "v"(v3), [hi] "v"(hi), [lo] "v"(lo));
#undef MK_PV
}
// Attention of several portions whose rows the prep stage has written (MK_PAIR_BOTH on a FX_ATTN stage).
//
// Bound by round trips, hand-overs and chains of dependent instructions: a unit of stage_fx_attn_t waits for its page entries, its queries and its first tile,
// for each tile's maximum, then for the other chunks' workgroups and what those have stored.  Here a task is two units, neighbouring row tiles of a
// request, whose chains cover each other over the same tiles, with all of their chunks, whose partial results stay in LDS (those behind CHUNKS in memory,
// written through: other layers' attention, with other units or portion by portion, uses the same words from other dies); pages and queries of the next task are requested while one runs, and the first tile of the next chunk or task before
// sums are merged.  (Units whose chunks end at different tiles follow each other; few units are a task each.)  Chunks, sums and merges are those of
// stage_fx_attn_t, in its order.  Six portions of 64 rows behind 1000 to 1500 positions, 32 q / 8 kv heads of 128: 96 us as a stage, portion by portion;
// a unit a task 68, now 50.
struct FxGroupRows {
  int row[MK_GROUP];     // a lane's rows as the first token of a request in a portion; row tiles up to its own << 8, tasks << 20
  int tiles, parts;      // of portion `lane`: row tiles; tasks of a kv head, and those of the portions in front
  int per_task, tasks;   // units of a task at most; of all portions, a kv head
};
// False: another form of the stage (long heads, long page lists, or too few units: a workgroup would be alone with all chunks of one), portion by portion.
__device__ __forceinline__ bool fx_attn_group_rows(CStage &st, const Ctx &c, const MkRuntime &rt, int portions, const int *sh_rows, FxGroupRows &g) {
  if ((rt.max_seq + rt.page_size - 1) / rt.page_size > MK_ATTN_PAIR_PAGES || st.head_dim > st.k_tiles * FxType<uint16_t>::KW) return false;
  const int lane = threadIdx.x & 63, qpk = st.num_q_heads / st.num_kv_heads, nvb = (st.v_dim + 15) / 16, nvs = (nvb + st.v_tiles - 1) / st.v_tiles;
  int units = 0, begins[MK_GROUP];
  g.tiles = 0;
#pragma unroll
  for (int p = 0; p < MK_GROUP; p++) begins[p] = ldc_i32(&rt.tok_first[min(p, portions - 1) * MK_MAX_TOKENS + lane]);  // (of rows that are none, looked at by nobody)
#pragma unroll
  for (int p = 0; p < MK_GROUP; p++) {
    const int M = p < portions ? __builtin_amdgcn_readfirstlane(sh_rows[p]) : 0;
    const bool first = lane < M && begins[p] == lane;
    const unsigned long long fm = __ballot(first), later = lane < 63 ? fm >> (lane + 1) : 0ull;
    const int n = first ? (later ? (int)__ffsll(later) : M - lane) : 0, incl = wave_incl_scan((n * qpk + 15) / 16, lane);
    g.row[p] = n | incl << 8;
    const int tiles = wave_bcast(incl, 63);
    if (lane == p) g.tiles = tiles;
    units += tiles * nvs * st.num_kv_heads;
  }
  g.per_task = units > c.G ? 2 : 1;
  int parts = 0;
#pragma unroll
  for (int p = 0; p < MK_GROUP; p++) {
    const int incl = wave_incl_scan((((g.row[p] & 0xff) * qpk + 15) / 16 + g.per_task - 1) / g.per_task, lane);
    g.row[p] |= incl << 20;
    if (lane == p) parts = wave_bcast(incl, 63) * nvs;
  }
  g.parts = wave_incl_scan(parts, lane);
  g.tasks = wave_bcast(g.parts, 63);
  return 2 * units >= c.G;
}
template <typename E, int KC, int VB>
__device__ __forceinline__ void fx_attn_group(Ctx &c, const MkRuntime &rt, int s, int portions, const int *sh_rows, const FxGroupRows &rows, char *smem) {
  using X = FxType<E>;
  static_assert(sizeof(E) == 2, "16-bit activations");
  constexpr int EPC = X::EPC, KW = X::KW, TP = X::TP, SUB = X::SUB, NU = 2, ROWS = MK_GROUP * MK_MAX_TOKENS;
  constexpr int PSTR = VB * 16 + 4, PST = VB * 16 + 32, QUADS = 16 * VB * 4, CHUNKS = 3, QMAX = KC * 64, PG = MK_ATTN_PAIR_PAGES / MK_THREADS;
  static_assert(QUADS % MK_THREADS == 0, "a merged chunk is whole quads of all threads");
  // LDS: query operands of this task and the next, page lists of both, the tokens' positions, first page-table entries and FxGroupRows::row, the wavefronts' sums, chunks
  u32x4 *const q_at = (u32x4 *)smem;
  int *const pages_at = (int *)(q_at + 2 * NU * QMAX), *const tab = pages_at + 2 * MK_ATTN_PAIR_PAGES;
  int *const row_at = tab + 2 * ROWS;
  float *const part = (float *)(row_at + ROWS), *const ml = part + NU * MK_WAVES * 16 * PSTR, *const chunk_ml = ml + NU * 128;
  f32x4 *const chunk_at = (f32x4 *)(chunk_ml + NU * MK_ATTN_MAX_CHUNKS * 32);
  static_assert((2 * NU * QMAX + NU * CHUNKS * QUADS) * 16 + (2 * MK_ATTN_PAIR_PAGES + 3 * ROWS + NU * (MK_WAVES * 16 * PSTR + 128 + MK_ATTN_MAX_CHUNKS * 32)) * 4 <= MK_LDS_BYTES, "attention scratch exceeds the LDS window");
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
  CStage &st = mk_portion_stages(rt, 0)[s];
  const int nkv = st.num_kv_heads, qpk = st.num_q_heads / nkv, D = st.head_dim, DV = st.v_dim;
  const int nkc = (D + KW - 1) / KW, nvb = (DV + 15) / 16, nvs = (nvb + VB - 1) / VB, ps = rt.page_size;
  const u32x4 *kc = (const u32x4 *)st.k_cache, *vc = (const u32x4 *)st.v_cache;
  const int win = MK_HAVE_HYB ? st.window : 0, keep = MK_HAVE_HYB ? st.keep_first : 0;
  if (wave == 0) {
#pragma unroll
    for (int p = 0; p < MK_GROUP; p++) row_at[p * MK_MAX_TOKENS + lane] = rows.row[p];
  }
  group_tokens(rt, portions, sh_rows, tab, tab + ROWS);
  const int n_tasks = rows.tasks * nkv;
  // Units from row r0 of a request on (its first row and position: t0, p0): query rows, none for the second where there is no such unit, and newest positions;
  // tiles NT, those behind the first `kept` ones `gap` further on, in C chunks.  split: the units follow each other.
  struct Task {
    int g, vs, portion, t0, r0, p0, item, cmax, C, NT, kept, gap, n_pages, nrows[NU], newest[NU];
    bool split;
    const int *pages;
  };
  // kv head outermost, and every other round from its end (contexts differ): see stage_fx_attn_t
  auto decode = [&](int u, int sub, Task &a) {
    const int round0 = u / c.G * c.G, turned = (u / c.G) & 1 ? round0 + min(c.G, n_tasks - round0) - 1 - (u - round0) : u;
    a.g = turned / rows.tasks;
    int k = turned - a.g * rows.tasks;
    // (looked up in a lane's registers and LDS: portions' numbers in scalar registers, and the choice among them, were spilled and fetched again for every task)
    a.portion = __builtin_amdgcn_readfirstlane((int)__ffsll(__ballot(rows.parts > k)) - 1);
    const int RT = wave_bcast(rows.tiles, a.portion), before = a.portion ? wave_bcast(rows.parts, a.portion - 1) : 0;
    const int mine = row_at[a.portion * MK_MAX_TOKENS + lane], parts = (wave_bcast(rows.parts, a.portion) - before) / nvs;
    k -= before;
    a.vs = k / parts;
    k -= a.vs * parts;
    a.cmax = max(1, min(c.G / (RT * nkv * nvs), MK_ATTN_MAX_CHUNKS));
    a.t0 = (int)__ffsll(__ballot((mine >> 20) > k)) - 1;
    const int own = wave_bcast(mine, a.t0), n_rows = (own & 0xff) * qpk, tiles = (n_rows + 15) / 16;
    const int tile = (k - ((own >> 20) - (tiles + rows.per_task - 1) / rows.per_task)) * rows.per_task;
    a.r0 = tile * 16;
    a.item = (a.g * nvs + a.vs) * RT + ((own >> 8) & 0xfff) - tiles + tile;
    a.p0 = __builtin_amdgcn_readfirstlane(tab[a.portion * MK_MAX_TOKENS + a.t0]);
    a.pages = rt.kv_indices + __builtin_amdgcn_readfirstlane(tab[ROWS + a.portion * MK_MAX_TOKENS + a.t0]);
    int NT[NU], kept[NU], gap[NU];
#pragma unroll
    for (int e = 0; e < NU; e++) {
      const int r = a.r0 + 16 * e;
      a.nrows[e] = e < rows.per_task ? max(0, min(16, n_rows - r)) : 0;
      a.newest[e] = a.p0 + (r + max(a.nrows[e], 1) - 1) / qpk;
      NT[e] = a.newest[e] / TP + 1;
      kept[e] = NT[e];
      gap[e] = 0;
      if (MK_HAVE_HYB) {
        const int first = a.p0 + r / qpk;
        int oldest = win ? max(0, first - win + 1) : 0;
#if MK_HAVE_DUAL
        if (st.chunk) oldest = max(oldest, first - first % st.chunk);
        if (win || st.chunk) kept[e] = min((keep + TP - 1) / TP, NT[e]);
#else
        if (win) kept[e] = min((keep + TP - 1) / TP, NT[e]);
#endif
        gap[e] = max(0, oldest / TP - kept[e]);
        NT[e] -= gap[e];
      }
    }
    a.split = a.nrows[1] && (NT[0] != NT[1] || kept[0] != kept[1] || gap[0] != gap[1]);
    a.NT = sub ? NT[1] : NT[0];
    a.kept = sub ? kept[1] : kept[0];
    a.gap = sub ? gap[1] : gap[0];
    if (sub) {
      a.r0 += 16;
      a.item++;
      a.nrows[0] = a.nrows[1];
      a.newest[0] = a.newest[1];
    }
    if (a.split) a.nrows[1] = 0;
    if (!a.nrows[1]) a.newest[1] = a.newest[0];
    a.C = fx_chunks(a.NT, a.cmax);
    a.n_pages = a.newest[1] / ps + 1;
  };
  auto phys = [](int tile, int kept, int gap) { return MK_HAVE_HYB && tile >= kept ? tile + gap : tile; };
  constexpr int NQ = NU * QMAX / MK_THREADS;
  static_assert(NU * QMAX % MK_THREADS == 0, "query operands of a unit, whole ones a thread");
  u32x4 q_next[NQ];
  int pg_next[PG];
  auto request = [&](const Task &a) {
    CStage &sp = mk_portion_stages(rt, a.portion)[s];
    const int r = tid & 15;
    unsigned row[NU];
    const auto queries = dev_rows(sp.q_ws);
#pragma unroll
    for (int e = 0; e < NU; e++) {
      const int R = a.nrows[e] ? a.r0 + e * 16 + min(r, a.nrows[e] - 1) : a.r0, t = R / qpk;  // (a unit that is none: the first one's first row, as none may follow)
      row[e] = 2u * ((unsigned)(a.t0 + t) * st.ld_qws + (unsigned)(a.g * qpk + R - t * qpk) * nkc * KW + ((tid & 63) >> 4) * EPC);
    }
    // Behind a wait for everything: without it the compiler, which cannot see that the registers' last loads have landed, waits in front of each of these
    // loads for all others.
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
#pragma unroll
    for (int j = 0; j < NQ; j++) {
      const int at = tid + j * MK_THREADS, i = at & (QMAX - 1);
      q_next[j] = ldc_16B(queries, (at >= QMAX ? row[1] : row[0]) + 2 * min(i >> 6, nkc - 1) * KW);
    }
#pragma unroll
    for (int i = 0; i < PG; i++) pg_next[i] = a.pages[min(tid + i * MK_THREADS, a.n_pages - 1)];
  };
  auto put = [&](const Task &a, int turn) {
#pragma unroll
    for (int j = 0; j < NQ; j++) {
      const int at = tid + j * MK_THREADS, i = at & (QMAX - 1);
      const u32x4 z = {0u, 0u, 0u, 0u};
      q_at[turn * (NU * QMAX) + at] = (tid & 15) < (at >= QMAX ? a.nrows[1] : a.nrows[0]) && (i >> 6) < nkc ? q_next[j] : z;
    }
#pragma unroll
    for (int i = 0; i < PG; i++)
      if (tid + i * MK_THREADS < a.n_pages) pages_at[turn * MK_ATTN_PAIR_PAGES + tid + i * MK_THREADS] = pg_next[i];
  };
  // Operands of a tile: keys, then values, each as soon as the registers are free (two sets of registers, and the tile's code twice, were
  // longer in the fetching of instructions than any tile).  !ok: the same number of loads from one spot.
  u32x4 k[SUB][KC], v[VB];
  size_t pt = 0;
  const int whole_shift = (ps & (ps - 1)) == 0 ? 31 - __builtin_clz(ps) : -1;
  auto load_keys = [&](int g, int turn, int tile, bool ok) {
    const int at = ok ? tile * TP : 0;
    const int page = whole_shift >= 0 ? at >> whole_shift : at / ps;  // (a division is longer than what it finds takes to arrive)
    pt = ok ? (size_t)__builtin_amdgcn_readfirstlane(pages_at[turn * MK_ATTN_PAIR_PAGES + page]) * ps + at - page * ps : 0;
    const u32x4 *kp = kc + ((pt / 16) * nkv + g) * nkc * 64 + lane;
    const int on = ok ? 64 : 0, su = ok ? nkv * nkc * 64 : 0;
#pragma unroll
    for (int u = 0; u < SUB; u++)
#pragma unroll
      for (int j = 0; j < KC; j++) k[u][j] = kp[u * su + min(j, nkc - 1) * on];
    __builtin_amdgcn_sched_barrier(0);
  };
  auto load_values = [&](int g, int vs, bool ok) {  // of the tile whose keys were requested last
    const u32x4 *vp = vc + ((pt / TP) * nkv + g) * nvb * 64 + lane;
    const int on = ok ? 64 : 0;
#pragma unroll
    for (int b = 0; b < VB; b++) v[b] = vp[min(vs * VB + b, nvb - 1) * on];
    __builtin_amdgcn_sched_barrier(0);
  };
  auto load_first = [&](int NT, int C, int kept, int gap, int g, int vs, int turn, int ci) {  // of a chunk, this wavefront's
    const int tile = NT * ci / C + wave;
    const bool ok = tile < NT * (ci + 1) / C;
    load_keys(g, turn, phys(tile, kept, gap), ok);
    load_values(g, vs, ok);
  };
  const float cap = st.softcap, sc1 = cap > 0.f ? st.sm_scale / cap : st.sm_scale, LOG2E = 1.4426950408889634f;
  const float *sink = (const float *)st.sink;
  Task next;
  if (c.vid < n_tasks) decode(c.vid, 0, next);
  barrier_wait(c);
  c.wrote_through = true;
  if (c.vid < n_tasks) {
    request(next);
    put(next, 0);
    __syncthreads();
    load_first(next.NT, next.C, next.kept, next.gap, next.g, next.vs, 0, 0);
  }
  for (int u = c.vid, sub = 0, turn = 0; u < n_tasks; turn ^= 1) {
    const Task a = next;
    if (a.split && !sub) {
      sub = 1;
    } else {
      sub = 0;
      u += c.G;
    }
    const bool goes_on = u < n_tasks;
    if (goes_on) {
      decode(u, sub, next);
      request(next);
    }
    CStage &sp = mk_portion_stages(rt, a.portion)[s];
    const u32x4 *qs = q_at + turn * (NU * QMAX);
    int plim[NU], olim[NU];
    float sc_row[NU];
#pragma unroll
    for (int e = 0; e < NU; e++) {
      const int R = a.r0 + 16 * e + min(lr, max(a.nrows[e], 1) - 1);
      plim[e] = a.p0 + R / qpk;
#if MK_HAVE_DUAL
      olim[e] = st.chunk ? plim[e] - plim[e] % st.chunk : 0;
      sc_row[e] = sc1 * (st.temp ? st.temp[a.g * qpk + R % qpk] : 1.f);
#else
      olim[e] = 0;
      sc_row[e] = sc1;
#endif
    }
    const int dv0 = a.vs * VB * 16;
    auto sink_of = [&](int e, int r) -> float { return sink ? sink[a.g * qpk + (a.r0 + 16 * e + min(r, max(e ? a.nrows[1] : a.nrows[0], 1) - 1)) % qpk] * LOG2E : -INFINITY; };
    auto emit = [&](int e, int r, int d, const f32x4 &o) {
      const int R = a.r0 + 16 * e + r;
      const float q[4] = {o[0], o[1], o[2], o[3]};
      fx_stc4((E *)sp.out + (size_t)(a.t0 + R / qpk) * st.ld_out + (size_t)(a.g * qpk + R % qpk) * DV, dv0 + d, DV, q);
    };
    float *const chunk_far = rt.group_attn_part + (size_t)a.portion * rt.group_attn + (size_t)a.item * a.cmax * 16 * PST;
    auto far = [&](int e, int ci, int r, int d) { return (f32x4 *)(chunk_far + ((size_t)(e * a.cmax + ci) * 16 + r) * PST + d); };
    for (int ci = 0; ci < a.C; ci++) {
      const int tb = a.NT * ci / a.C, te = a.NT * (ci + 1) / a.C;
      float m[NU], l[NU];
      f32x4 acc[NU][VB], S[NU][SUB];
#pragma unroll
      for (int e = 0; e < NU; e++) {
        m[e] = MK_FX_NEG;
        l[e] = 0.f;
#pragma unroll
        for (int b = 0; b < VB; b++) acc[e][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
      // (see stage_fx_attn_t for what is done with a tile; the last one is requested again behind the end)
      for (int tl = tb + wave; tl < te; tl += MK_WAVES) {
        const int tile = phys(tl, a.kept, a.gap);
        const bool more = tl + MK_WAVES < te;
#pragma unroll
        for (int e = 0; e < NU; e++)
#pragma unroll
          for (int u_ = 0; u_ < SUB; u_++) S[e][u_] = (f32x4){0.f, 0.f, 0.f, 0.f};
        u32x4 q[KC][NU];
#pragma unroll
        for (int j = 0; j < KC; j++)
#pragma unroll
          for (int e = 0; e < NU; e++) q[j][e] = qs[e * QMAX + j * 64 + lane];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < KC; j++)
#pragma unroll
          for (int u_ = 0; u_ < SUB; u_++)
#pragma unroll
            for (int e = 0; e < NU; e++) S[e][u_] = fx_mma_k(E(), k[u_][j], q[j][e], S[e][u_]);
        load_keys(a.g, turn, phys(tl + MK_WAVES, a.kept, a.gap), more);
        float sc[NU][SUB][4], tm[NU];
        auto each = [&](auto f) {
#pragma unroll
          for (int e = 0; e < NU; e++)
#pragma unroll
            for (int u_ = 0; u_ < SUB; u_++)
#pragma unroll
              for (int i = 0; i < 4; i++) f(e, u_, i);
        };
        // (one branch: at every value of its own the values follow each other, 14 us of 55 in a thousand positions)
        if (cap > 0.f) {
          each([&](int e, int u_, int i) { sc[e][u_][i] = __builtin_amdgcn_exp2f(S[e][u_][i] * sc_row[e] * (2.f * LOG2E)); });
          each([&](int e, int u_, int i) { sc[e][u_][i] = (cap * LOG2E) * (1.f - 2.f * __builtin_amdgcn_rcpf(1.f + sc[e][u_][i])); });
        } else {
          each([&](int e, int u_, int i) { sc[e][u_][i] = S[e][u_][i] * sc_row[e] * LOG2E; });
        }
        tm[0] = tm[1] = MK_FX_NEG;
        each([&](int e, int u_, int i) {
          const int at = tile * TP + u_ * 16 + lg * 4 + i;
          bool seen = at <= plim[e];
          if (MK_HAVE_HYB) seen = seen && (win == 0 || plim[e] - at < win || at < keep);
#if MK_HAVE_DUAL
          seen = seen && at >= olim[e];
#endif
          sc[e][u_][i] = seen ? sc[e][u_][i] : MK_FX_NEG;
          tm[e] = fmaxf(tm[e], sc[e][u_][i]);
        });
#pragma unroll
        for (int e = 0; e < NU; e++) tm[e] = groups_max(tm[e]);
        if (__any(tm[0] > m[0] || tm[1] > m[1])) {
#pragma unroll
          for (int e = 0; e < NU; e++) {
            const float nm = fmaxf(m[e], tm[e]), corr = fx_exp2(E(), m[e] - nm);
            m[e] = nm;
            l[e] *= corr;
#pragma unroll
            for (int b = 0; b < VB; b++) acc[e][b] *= corr;
          }
        }
        u32x4 hi[NU], lo[NU];
#pragma unroll
        for (int e = 0; e < NU; e++) {
#pragma unroll
          for (int u_ = 0; u_ < SUB; u_++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
              sc[e][u_][i] = sc[e][u_][i] > 0.5f * MK_FX_NEG ? fx_exp2(E(), sc[e][u_][i] - m[e]) : 0.f;
              l[e] += sc[e][u_][i];
            }
#pragma unroll
          for (int w = 0; w < 4; w++) {
            const float x0 = sc[e][w >> 1][(w & 1) * 2], x1 = sc[e][w >> 1][(w & 1) * 2 + 1];
            hi[e][w] = pack2(x0, x1);
            lo[e][w] = pack2(x0 - bf_lo(hi[e][w]), x1 - bf_hi(hi[e][w]));
          }
        }
        const bool edge = (tile + 1) * TP - 1 > a.newest[0];
#pragma unroll
        for (int e = NU - 1; e >= 0; e--) {
          if (edge) {  // values behind the newest position belong to nobody (the first unit's is not behind the second's)
#pragma unroll
            for (int b = 0; b < VB; b++)
#pragma unroll
              for (int w = 0; w < 4; w++) {
                const int q = tile * TP + (w >> 1) * 16 + lg * 4 + (w & 1) * 2;
                v[b][w] = q > a.newest[e] ? 0u : (q + 1 > a.newest[e] ? v[b][w] & 0xffffu : v[b][w]);
              }
          }
#pragma unroll
          for (int b = 0; b < VB; b += 4) fx_add_products(acc[e][b], acc[e][b + 1], acc[e][b + 2], acc[e][b + 3], v[b], v[b + 1], v[b + 2], v[b + 3], hi[e], lo[e]);
        }
        load_values(a.g, a.vs, more);
      }
      // ---- wavefronts of the workgroup
      const bool last = ci == a.C - 1;
      if (last && goes_on) put(next, turn ^ 1);
#pragma unroll
      for (int e = 0; e < NU; e++) l[e] = groups_sum(l[e]);
      lds_barrier();  // (sums of the chunk in front have been read, and what was put is there)
      if (!last || goes_on)
        load_first(last ? next.NT : a.NT, last ? next.C : a.C, last ? next.kept : a.kept, last ? next.gap : a.gap, last ? next.g : a.g, last ? next.vs : a.vs, last ? turn ^ 1 : turn, last ? 0 : ci + 1);
#pragma unroll
      for (int e = 0; e < NU; e++) {
#pragma unroll
        for (int b = 0; b < VB; b++) *(f32x4 *)(part + ((e * MK_WAVES + wave) * 16 + lr) * PSTR + b * 16 + lg * 4) = acc[e][b];
        if (lg == 0) {
          ml[e * 128 + wave * 16 + lr] = m[e];
          ml[e * 128 + 64 + wave * 16 + lr] = l[e];
        }
      }
      lds_barrier();
#pragma unroll 1
      for (int i = tid; i < (a.nrows[1] ? 2 : 1) * QUADS; i += MK_THREADS) {
        const int e = i >= QUADS, q = i - e * QUADS, r = q / (VB * 4), d = (q - r * (VB * 4)) * 4;
        const float *const mr = ml + e * 128 + r, *const pr = part + (e * MK_WAVES * 16 + r) * PSTR + d;
        float M_ = MK_FX_NEG, L_ = 0.f, fin[MK_WAVES];
#pragma unroll
        for (int w = 0; w < MK_WAVES; w++) M_ = fmaxf(M_, mr[w * 16]);
#pragma unroll
        for (int w = 0; w < MK_WAVES; w++) {
          fin[w] = exp2f(mr[w * 16] - M_);
          L_ += mr[64 + w * 16] * fin[w];
        }
        if (a.C == 1) {
          const float inv = 1.f / (L_ + exp2f(sink_of(e, r) - M_));
#pragma unroll
          for (int w = 0; w < MK_WAVES; w++) fin[w] *= inv;
        } else if (d == 0) {
          float *const cml = chunk_ml + (e * MK_ATTN_MAX_CHUNKS + ci) * 32 + r;
          cml[0] = M_;
          cml[16] = L_;
        }
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < MK_WAVES; w++) o += *(const f32x4 *)(pr + w * 16 * PSTR) * fin[w];
        if (a.C > 1) {  // (not one address for both: it would be a generic one)
          if (ci < CHUNKS) chunk_at[(e * CHUNKS + ci) * QUADS + q] = o;
          else stc_16B((u32x4 *)far(e, ci, r, d), __builtin_bit_cast(u32x4, o));
        } else if (r < (e ? a.nrows[1] : a.nrows[0]) && dv0 + d < DV) {
          emit(e, r, d, o);
        }
      }
    }
    if (a.C == 1) continue;
    // ---- chunks
    lds_barrier();
#pragma unroll 1
    for (int i = tid; i < (a.nrows[1] ? 2 : 1) * QUADS; i += MK_THREADS) {
      const int e = i >= QUADS, q = i - e * QUADS, r = q / (VB * 4), d = (q - r * (VB * 4)) * 4;
      if (r >= (e ? a.nrows[1] : a.nrows[0]) || dv0 + d >= DV) continue;
      const float *const cml = chunk_ml + e * MK_ATTN_MAX_CHUNKS * 32 + r;
      float M_ = MK_FX_NEG, L_ = 0.f;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int ci = 0; ci < a.C; ci++) M_ = fmaxf(M_, cml[ci * 32]);
#pragma unroll 1
      for (int ci = 0; ci < a.C; ci++) {
        const float f = exp2f(cml[ci * 32] - M_);
        f32x4 x;
        if (ci < CHUNKS) x = chunk_at[(e * CHUNKS + ci) * QUADS + q];
        else x = __builtin_bit_cast(f32x4, ldc_16B((const u32x4 *)far(e, ci, r, d)));
        L_ += cml[ci * 32 + 16] * f;
        o += x * f;
      }
      emit(e, r, d, o * (1.f / (L_ + exp2f(sink_of(e, r) - M_))));
    }
  }
}
template <typename E>
__device__ __forceinline__ void stage_fx_attn_group(CStage &st, Ctx &c, const MkRuntime &rt, int s, int portions, const int *sh_rows, const FxGroupRows &rows, char *smem) {
  if (st.v_tiles == 4) {
    if (st.k_tiles == 2) fx_attn_group<E, 2, 4>(c, rt, s, portions, sh_rows, rows, smem);
    else fx_attn_group<E, 4, 4>(c, rt, s, portions, sh_rows, rows, smem);
  } else {
    fx_attn_group<E, 4, 8>(c, rt, s, portions, sh_rows, rows, smem);
  }
}
#endif
template <typename E>
__device__ __forceinline__ void stage_fx_attn(CStage &st, Ctx &c, const MkRuntime &rt, int M, bool single, char *smem) {
  if constexpr (sizeof(E) == 2) {
    if (st.v_tiles == 4) {
      if (st.k_tiles == 2) stage_fx_attn_t<E, 2, 4>(st, c, rt, M, single, smem);
      else stage_fx_attn_t<E, 4, 4>(st, c, rt, M, single, smem);
    } else {
      stage_fx_attn_t<E, 4, 8>(st, c, rt, M, single, smem);
    }
  } else {
    stage_fx_attn_t<E, 8, 8>(st, c, rt, M, single, smem);
  }
}

// ----------------------------------------------------------------------------- 32-bit linear
__device__ __forceinline__ float fx_glu_f32(CStage &st, float g, float u) {
#if MK_HAVE_DUAL
  if (st.flags & MK_F_GELU) return 0.5f * g * (1.f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
#endif
  return g / (1.f + expf(-g)) * u;
}
// out[m, n] = sum_k x[m, k] W[n, k] in true 32-bit (v_mfma_f32_16x16x4_f32), optional SwiGLU epilogue.
//
// Bound by the weights' stream with few tokens, by the matrix cores (157 TFLOP/s) and the CU's path to L2 with many.  A unit is a 16-column
// output tile (a pair of them under SwiGLU) times MT tiles of 16 tokens; a workgroup walks a contiguous range of units, its wavefronts
// split the reduction and are reduced through LDS in a fixed order.  Operands of D steps of 32 k are in flight per wavefront and never
// drain between units; the weights of the first ones are requested before the previous stage's barrier.
// Rows are read eight lanes to a whole 128-byte line and change into operand order in a wavefront's own LDS (16-byte words of a row
// XORed with the row, so neither direction meets a bank twice): read in operand order, every lane another row, a CU takes in 16 bytes a
// clock, a quarter of what it can.
// MT is the number of token tiles that leaves the workgroup with the most units the least to multiply, the largest of them where they
// tie: a weight row is then read once for more tokens.  The token groups of a tile are neighbours in a range, so that what they read
// again comes from the die's L2.
// Before -> now, 3 / 64 tokens, us: 5120 x 2048 34 -> 14 / 60 -> 33, 2048 x 4096 34 -> 13 / 56 -> 19, gate and up 12288 x 2048 46 -> 28 / 71
// -> 48, 2048 x 6144 48 -> 17 / 80 -> 26, 32768 x 2048 129 -> 49 (5.5 TB/s) / 217 -> 120 (72 TFLOP/s; operand-order loads: 158).
template <int MT, bool SILU>
__device__ __forceinline__ void stage_fx_linear_f32_t(CStage &st, Ctx &c, int M, char *smem) {
  constexpr int NH = SILU ? 2 : 1, NT = NH + MT, D = MT == 1 ? 8 : 4;  // 16-row tiles of a step: weights, then tokens
  constexpr bool DB = NH * MT < 8;                                       // sums of two units fit beside the operands
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4, l8 = lane >> 3, c8 = lane & 7;
  const int K = st.k, n_out = SILU ? st.n / 2 : st.n, half = st.silu_half, nks = K / 16;  // (16 k of a tile are one operand)
  const int ng = (M + 16 * MT - 1) / (16 * MT), n_units = (n_out + 15) / 16 * ng;
  const int u0 = (int)(((long long)c.vid * n_units) / c.G), u1 = (int)(((long long)(c.vid + 1) * n_units) / c.G);
  const int kq = (nks + MK_WAVES - 1) / MK_WAVES, kb = min(nks, wave * kq), ke = min(nks, kb + kq), nb = (kq + 2 * D - 1) / (2 * D);
  f32x4 *red = (f32x4 *)smem;  // [DB ? 2 : 1][waves][NH][MT][64]
  f32x4 *ops = red + (DB ? 2 : 1) * MK_WAVES * NH * MT * 64 + wave * 2 * NT * 128;  // [2][tile][8-row half][8 rows][8 words]
  struct Unit {
    const f32x4 *w[NH][2];  // this lane's weight row of either half of a tile
    int x[MT][2];           // ... token row, in bytes
    int tile, m0;
  };
  auto unit = [&](int u) {
    Unit a;
    a.tile = u / ng;
    a.m0 = (u - a.tile * ng) * 16 * MT;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int o = min(a.tile * 16 + 8 * i + l8, n_out - 1);
      const int vr = SILU ? (o / half) * 2 * half + (o % half) : o;
#pragma unroll
      for (int h = 0; h < NH; h++) a.w[h][i] = (const f32x4 *)weight_row(st.w, vr + h * half, K / 4);
#pragma unroll
      for (int mt = 0; mt < MT; mt++) a.x[mt][i] = min(a.m0 + mt * 16 + 8 * i + l8, M - 1) * st.ld_in * 4;
    }
    return a;
  };
  f32x4 ring[D][NT][2];
  Unit a{};
  if (u0 < u1) a = unit(u0);
  const bool early = u0 < u1 && wave != 0;
  auto word = [&](int s) { return min(4 * s + c8, 4 * nks - 1); };  // this lane's 16-byte word of the step that begins at s (in units of 16 k)
  const auto x_rows = dev_rows(st.in);
  auto request_w = [&](f32x4 (&r)[NT][2], const Unit &p, int s) {
#pragma unroll
    for (int h = 0; h < NH; h++)
#pragma unroll
      for (int i = 0; i < 2; i++) r[h][i] = p.w[h][i][word(s)];
  };
  auto request_x = [&](f32x4 (&r)[NT][2], const Unit &p, int s) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int i = 0; i < 2; i++) r[NH + mt][i] = __builtin_bit_cast(f32x4, ldc_16B(x_rows, p.x[mt][i] + 16 * word(s)));
  };
  if (early) {
#pragma unroll
    for (int j = 0; j < D; j++) request_w(ring[j], a, kb + 2 * j);
  }
  barrier_wait(c);
  c.wrote_through = true;
  if (u0 >= u1) return;
  if (!early) {
#pragma unroll
    for (int j = 0; j < D; j++) request_w(ring[j], a, kb + 2 * j);
  }
#pragma unroll
  for (int j = 0; j < D; j++) request_x(ring[j], a, kb + 2 * j);
  f32x4 op[2][NT][2];  // operands of two steps, [tile][16 k]
  auto turn = [&](const f32x4 (&r)[NT][2], f32x4 (&o)[NT][2], int slot) {
    f32x4 *b = ops + slot * NT * 128;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int i = 0; i < 2; i++) b[t * 128 + i * 64 + l8 * 8 + (c8 ^ l8)] = r[t][i];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int h = 0; h < 2; h++) o[t][h] = b[t * 128 + lr * 8 + ((h * 4 + lg) ^ (lr & 7))];
  };
  turn(ring[0], op[0], 0);
  for (int u = u0; u < u1; u++) {
    const bool more = u + 1 < u1;
    const Unit nx = more ? unit(u + 1) : a;
    f32x4 acc[NH][MT];
#pragma unroll
    for (int h = 0; h < NH; h++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) acc[h][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int blk = 0; blk < nb; blk++) {
      const bool last = blk + 1 == nb;
      const int k0 = kb + blk * 2 * D, kn = last ? kb : k0 + 2 * D, step = last && !more ? 0 : 2;  // (behind the range: one line again and again)
      Unit p;
#pragma unroll
      for (int i = 0; i < 2; i++) {
#pragma unroll
        for (int h = 0; h < NH; h++) p.w[h][i] = last ? nx.w[h][i] : a.w[h][i];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) p.x[mt][i] = last ? nx.x[mt][i] : a.x[mt][i];
      }
#pragma unroll
      for (int j = 0; j < D; j++) {
        // operands of the step behind this one, whose place in the ring is then free (the one behind a block's last is its successor's first)
        request_w(ring[j], p, kn + step * j);
        request_x(ring[j], p, kn + step * j);
        turn(ring[(j + 1) % D], op[(j + 1) & 1], (j + 1) & 1);
        const int s = k0 + 2 * j;
#pragma unroll
        for (int e = 0; e < 2; e++)
          if (s + e < ke) {
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
              for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int h = 0; h < NH; h++) acc[h][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(op[j & 1][h][e][q], op[j & 1][NH + mt][e][q], acc[h][mt], 0, 0, 0);
          }
      }
    }
    f32x4 *rb = red + (DB ? u & 1 : 0) * (MK_WAVES * NH * MT * 64) + lane;
    if (!DB) __syncthreads();
#pragma unroll
    for (int h = 0; h < NH; h++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) rb[((wave * NH + h) * MT + mt) * 64] = acc[h][mt];
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const int m = a.m0 + mt * 16 + lr;
      if (((u * MT + mt) & (MK_WAVES - 1)) != wave || m >= M) continue;
      f32x4 v[NH];
#pragma unroll
      for (int h = 0; h < NH; h++) {
        v[h] = rb[(h * MT + mt) * 64];
#pragma unroll
        for (int q = 1; q < MK_WAVES; q++) v[h] += rb[((q * NH + h) * MT + mt) * 64];
      }
      float r[4];
#pragma unroll
      for (int i = 0; i < 4; i++) r[i] = SILU ? fx_glu_f32(st, v[0][i], v[NH - 1][i]) : linear_act(st, v[0][i]);
      fx_stc4((float *)st.out + (size_t)m * st.ld_out, a.tile * 16 + lg * 4, n_out, r);
    }
    a = nx;
  }
}
__device__ __forceinline__ void stage_fx_linear_f32(CStage &st, Ctx &c, int M, char *smem) {
  const bool silu = st.flags & MK_F_SILU;
  const int tiles = ((silu ? st.n / 2 : st.n) + 15) / 16, mt = (M + 15) / 16;
  auto rounds = [&](int per) { return (tiles * ((mt + per - 1) / per) + c.G - 1) / c.G * per; };  // token tiles of the busiest workgroup
  const int r1 = rounds(1), r2 = mt > 1 ? rounds(2) : 1 << 30, r4 = mt > 2 ? rounds(4) : 1 << 30;
  if (r4 <= r2 && r4 <= r1) {
    if (silu) stage_fx_linear_f32_t<4, true>(st, c, M, smem);
    else stage_fx_linear_f32_t<4, false>(st, c, M, smem);
  } else if (r2 <= r1) {
    if (silu) stage_fx_linear_f32_t<2, true>(st, c, M, smem);
    else stage_fx_linear_f32_t<2, false>(st, c, M, smem);
  } else if (silu) {
    stage_fx_linear_f32_t<1, true>(st, c, M, smem);
  } else {
    stage_fx_linear_f32_t<1, false>(st, c, M, smem);
  }
}
