// Iterations of several portions of prompts (part of the persistent kernel, included by mk_kernel.hip where MK_PAIR is set): what runs for all portions at
// once.  See MkPairEntry for the rest.

// The stages as they run for a portion of several in one iteration.
__device__ __forceinline__ CStage *mk_portion_stages(const MkRuntime &rt, int portion) {
  return (CStage *)(unsigned long long)(portion ? rt.stages2 + (size_t)(portion - 1) * rt.num_stages : rt.stages);
}
// Its tokens (Ctx::sh_tok), a lane each.  What is looked up by slot, page tables among it, lies batch_at words behind.
__device__ __forceinline__ void mk_portion_rows(const MkRuntime &rt, int *tok, int t, int rows, int portion) {
  if (t < 0 || t >= rows) return;
  const int at = portion * MK_MAX_TOKENS + t, slot = ldc_i32(&rt.tok_slot[at]);
  tok[t] = ldc_i32(&rt.tok_pos[at]);
  tok[MK_MAX_TOKENS + t] = slot;
  tok[2 * MK_MAX_TOKENS + t] = ldc_i32(&rt.tok_first[at]);
  tok[3 * MK_MAX_TOKENS + t] = (rt.batch_n ? rt.batch_at[portion] : 0) + ldc_i32(&rt.kv_indptr[slot]);
}

// 16 bytes of every lane, `off` bytes behind a uniform address, straight to LDS: lane l's land at byte `lds` + 16 l.  In assembly, as the compiler waits for all
// such requests of its own in front of every read of LDS, whichever buffer that reads: the ring of weights ran dry at every pass.  Whoever requests rows
// waits for them by count.
__device__ __forceinline__ void lds_request(const char *base, unsigned off, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 sc1" ::"v"(off), "s"(base), "s"(lds) : "memory", "m0");
}

// Linear over the rows of several portions (MK_PAIR_BOTH): mk_group_plan says who takes what.  Two portions, 64 rows each, are the columns of a task; each
// of the four wavefronts multiplies TW weight tiles of its own with all of them, so that a weight goes from the cache to its registers once, as a
// ring of NB steps, and LDS carries token rows only, two passes of NSP steps, each staged by all wavefronts while the other is multiplied.  Sums
// of an output are made in the order in which stage_linear_mfma_xres makes them.
//
// Bound by the matrix cores, once the rows are many: a wavefront has its SIMD to itself, so the operands of eight tiles are read while the eight in front are
// multiplied, and whatever is not covered that way (a workgroup barrier and the first operands of a pass, the first rows of a task) is lost.
// Outputs [o, o + 8) of row m of a portion (whose stage is `sp`) from sums(column): four sums from that column of the weight tiles on.
template <typename Sums>
__device__ __forceinline__ void linear_group_out(CStage &st, CStage &sp, int m, int o, int n_out, Sums sums) {
  const bool silu = st.flags & MK_F_SILU;
  float r[2][4], res[2][4];
  if (st.flags & MK_F_RES) {
#pragma unroll
    for (int h = 0; h < 2; h++) ldc_bf16x4((const uint16_t *)sp.res + (size_t)m * st.ld_res, o + h * 4, n_out, res[h]);
  }
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int col = silu ? (o >> 4) * 32 + (o & 15) + h * 4 : o + h * 4;  // (tiles of 16: gate, up, gate, up ...)
    const f32x4 g = sums(col), u = silu ? sums(col + 16) : g;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      float v = silu ? linear_glu(st, g[e], u[e]) : g[e];
      if (st.flags & MK_F_RES) v += res[h][e];
      r[h][e] = linear_act(st, v);
    }
  }
  uint16_t *row = (uint16_t *)sp.out + (size_t)m * st.ld_out;
  if (o + 8 <= n_out && ((unsigned long long)(row + o) & 15) == 0) {
    stc_16B((u32x4 *)(row + o), (u32x4){pack2(r[0][0], r[0][1]), pack2(r[0][2], r[0][3]), pack2(r[1][0], r[1][1]), pack2(r[1][2], r[1][3])});
  } else {
#pragma unroll
    for (int h = 0; h < 2; h++) stc_bf16x4(row, o + h * 4, n_out, r[h]);
  }
}
template <int TW>
__device__ __forceinline__ void linear_group_tasks(CStage &st, const MkRuntime &rt, int s, int vid, int G, int tid, int portions, const int *sh_rows, const GroupPlan plan, char *smem) {
  constexpr int MT = 8, PQ = MT / 4, NSP = 32 / MT, NB = 4, XBUF = NSP * MT * 128;  // XBUF: 16-byte operands of a buffer, [step][token tile][16 rows][8]
  static_assert(NB % NSP == 0 && NB * TW * 2 <= 63, "a ring is whole passes, and can be waited for by count");
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
  const bool silu = st.flags & MK_F_SILU;
  const int K = st.k, n_out = silu ? st.n / 2 : st.n, S = plan.S;
  const int kslice = K / S, nsuper = (kslice >> 6) / NB, all_rows = portions * MK_MAX_TOKENS;
  const bool defer = (st.flags & MK_F_DEFER_SUM) && S > 1, normed = st.flags & MK_F_NORM;
  const int ldx = normed ? st.ld_norm : st.ld_in, ld_part = defer ? st.n : plan.wt * 16;
  u32x4 *xl = (u32x4 *)smem;
  const unsigned lds = (unsigned)(unsigned long long)(__attribute__((address_space(3))) char *)smem;
  static_assert(2 * XBUF * 16 <= MK_LDS_BYTES, "rows fit");
  const int task0 = (int)(((long long)vid * plan.tasks) / G), task1 = (int)(((long long)(vid + 1) * plan.tasks) / G);
  for (int task = task0; task < task1; task++) {
    const int mb = task % plan.mb, rest = task / plan.mb, sl = rest % S, nb = rest / S;
    const int kbeg = sl * kslice, tw0 = (nb * MK_WAVES + wave) * TW;
    const char *wrow[TW];  // (uniform; a lane's words lie 16 bytes apart)
#pragma unroll
    for (int t = 0; t < TW; t++) wrow[t] = (const char *)st.wpack + ((size_t)min(tw0 + t, plan.wt - 1) * (K >> 6) + (kbeg >> 6)) * 2048;
    bf16x8 a[NB][TW][2];
    auto w_load = [&](int step, bf16x8 (&aa)[TW][2]) {
#pragma unroll
      for (int t = 0; t < TW; t++)
#pragma unroll
        for (int h = 0; h < 2; h++) aa[t][h] = *(const MK_GLOBAL bf16x8 *)((const MK_GLOBAL char *)(unsigned long long)(wrow[t] + (size_t)step * 2048) + (unsigned)lane * 16u + h * 1024);
    };
    // rows of a pass: item (step, token tile) as two requests of eight whole 128-byte lines; a wavefront takes one token tile of each portion (of the last
    // one again, where there are no more).  See stage_linear_mfma_xres for where a word lies.
    const int p0 = PQ * mb, here = min(PQ, portions - p0);
    const char *x[PQ];
    unsigned at[PQ][2];
    const int rr = wave * 16 + (lane >> 3), kw = kbeg + ((lane & 7) ^ (lane >> 3)) * 8;
#pragma unroll
    for (int q = 0; q < PQ; q++) {
      const int p = min(p0 + q, portions - 1), last = __builtin_amdgcn_readfirstlane(sh_rows[p]) - 1;
      CStage &sp = mk_portion_stages(rt, p)[s];
      x[q] = (const char *)(normed ? sp.norm_out : sp.in);
#pragma unroll
      for (int h = 0; h < 2; h++) at[q][h] = 2u * (unsigned)(min(rr + 8 * h, last) * ldx + kw);
    }
    auto stage_pass = [&](int pass) {
#pragma unroll
      for (int step = 0; step < NSP; step++)
#pragma unroll
        for (int q = 0; q < PQ; q++)
#pragma unroll
          for (int h = 0; h < 2; h++)
            lds_request(x[q] + (size_t)(pass * NSP + step) * 128, at[q][h], lds + (unsigned)((pass & 1) * XBUF + (step * MT + q * 4 + wave) * 128 + h * 64) * 16);
    };
    if (task > task0) lds_barrier();  // (everybody is through with the rows of the task in front)
    __builtin_amdgcn_sched_barrier(0);
    stage_pass(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NB; j++) w_load(j, a[j]);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc[TW][MT];
#pragma unroll
    for (int t = 0; t < TW; t++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) acc[t][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // a step is NBLK blocks of eight token tiles and 32 of its 64 values
    constexpr int NBLK = MT / 4;
    auto operands = [&](const u32x4 *xb, int blk, u32x4 (&b)[8]) {
      const int h = blk / (MT / 8), m0 = blk % (MT / 8) * 8;
#pragma unroll
      for (int m = 0; m < 8; m++) b[m] = xb[(m0 + m) * 128 + lr * 8 + ((h * 4 + lg) ^ (lr & 7))];
      __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const bf16x8 (&aa)[TW][2], int blk, const u32x4 (&b)[8]) {
      const int h = blk / (MT / 8), m0 = blk % (MT / 8) * 8;
#pragma unroll
      for (int m = 0; m < 8; m++)
#pragma unroll
        for (int t = 0; t < TW; t++) acc[t][m0 + m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aa[t][h], __builtin_bit_cast(bf16x8, b[m]), acc[t][m0 + m], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto super = [&](int sp, auto first_c, auto more_c) {  // the steps of a ring
      constexpr bool FIRST = decltype(first_c)::value, MORE = decltype(more_c)::value;
#pragma unroll
      for (int u = 0; u < NB / NSP; u++) {
        const int pass = sp * (NB / NSP) + u;
        // this pass's rows have landed: what was requested behind them is the ring, or a pass's part of it
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((FIRST && u == 0 ? NB : u == 0 || MORE ? NSP : 0) * TW * 2) : "memory");
        lds_barrier();
        if (MORE || u + 1 < NB / NSP) stage_pass(pass + 1);
        __builtin_amdgcn_sched_barrier(0);
        const u32x4 *xb = xl + (pass & 1) * XBUF;
        u32x4 b[2][8];
        operands(xb, 0, b[0]);
#pragma unroll
        for (int j = 0; j < NSP; j++) {
#pragma unroll
          for (int blk = 0; blk < NBLK; blk++) {
            const int next = j * NBLK + blk + 1;
            if (next < NSP * NBLK) operands(xb + next / NBLK * MT * 128, next % NBLK, b[next & 1]);
            multiply(a[u * NSP + j], blk, b[(next & 1) ^ 1]);
          }
          if (MORE) w_load((sp + 1) * NB + u * NSP + j, a[u * NSP + j]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    super(0, std::true_type{}, std::true_type{});  // (a slice is 512 values at least)
    for (int sp = 1; sp < nsuper - 1; sp++) super(sp, std::false_type{}, std::true_type{});
    super(nsuper - 1, std::false_type{}, std::false_type{});
    // lane l holds token m = mt * 16 + (l & 15) of the portions' four tiles each, output columns tile * 16 + (l >> 4) * 4 .. + 3
    if (S > 1) {
#pragma unroll
      for (int t = 0; t < TW; t++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
          if (tw0 + t < plan.wt && mt / 4 < here)
            stc_16B((u32x4 *)(rt.group_part + ((size_t)sl * all_rows + p0 * MK_MAX_TOKENS + mt * 16 + lr) * ld_part + (tw0 + t) * 16 + lg * 4), __builtin_bit_cast(u32x4, acc[t][mt]));
      continue;
    }
    // Outputs from the accumulators, which go through LDS a portion at a time.  (From the registers they lie in, the code of every tile's activation would
    // stand here once for every tile, and a row's outputs leave in pieces of 32 bytes.)
    constexpr int COLS = MK_WAVES * TW * 16, LDT = COLS + 4;
    static_assert(MK_MAX_TOKENS * LDT * 4 <= 2 * XBUF * 16, "a portion's sums fit the row buffers");
    float *tile = (float *)smem;
    const int per_row = (silu ? COLS / 2 : COLS) / 8, o_base = nb * (silu ? COLS / 2 : COLS);
#pragma unroll
    for (int q = 0; q < PQ; q++) {
      if (q >= here) continue;
      lds_barrier();  // (everybody is through with the rows, or with the sums of the portion in front)
#pragma unroll
      for (int t = 0; t < TW; t++)
#pragma unroll
        for (int mt = 0; mt < 4; mt++) *(f32x4 *)(tile + (mt * 16 + lr) * LDT + (wave * TW + t) * 16 + lg * 4) = acc[t][q * 4 + mt];
      lds_barrier();
      CStage &sp = mk_portion_stages(rt, p0 + q)[s];
      const int rows = __builtin_amdgcn_readfirstlane(sh_rows[p0 + q]);
      for (int i = tid; i < rows * per_row; i += MK_THREADS) {
        const int m = i / per_row, o = o_base + (i - m * per_row) * 8;
        if (o < n_out) linear_group_out(st, sp, m, o, n_out, [&](int col) { return *(const f32x4 *)(tile + m * LDT + col - nb * COLS); });
      }
    }
  }
}
__device__ __forceinline__ void stage_linear_group(CStage &st, Ctx &c, const MkRuntime &rt, int s, int portions, const int *sh_rows, char *smem) {
  barrier_wait(c);
  const GroupPlan p = mk_group_plan(st, c.G, portions);
  const int tw = __builtin_amdgcn_readfirstlane(p.tw);
  if (tw == 2) linear_group_tasks<2>(st, rt, s, c.vid, c.G, c.tid, portions, sh_rows, p, smem);
  else if (tw == 3) linear_group_tasks<3>(st, rt, s, c.vid, c.G, c.tid, portions, sh_rows, p, smem);
  else linear_group_tasks<4>(st, rt, s, c.vid, c.G, c.tid, portions, sh_rows, p, smem);
  c.wrote_through = true;  // (partial sums and outputs)
  if (p.S == 1) return;
  if (st.flags & MK_F_DEFER_SUM) {
    c.defer_S = p.S;
    c.defer_rows = portions * MK_MAX_TOKENS;
    c.defer_n = st.n;
    c.defer_part = rt.group_part;
    c.defer_res = (st.flags & MK_F_RES) ? st.res : nullptr;
    c.defer_ld_res = st.ld_res;
    c.defer_stage = s;
    return;
  }
  // Sums of the slices, in their order, by all workgroups once all are there.  (By the last workgroup of a task to arrive, as one portion's linear does it, 6144 x 4096
  // at 512 rows took 50 us longer than with its sums left to the stage behind.)
  barrier_arrive(c);
  barrier_wait(c);
  const int n_out = (st.flags & MK_F_SILU) ? st.n / 2 : st.n, per_row = (n_out + 7) / 8, ld = p.wt * 16;
  for (int q = 0; q < portions; q++) {
    CStage &sp = mk_portion_stages(rt, q)[s];
    const int rows = __builtin_amdgcn_readfirstlane(sh_rows[q]);
    for (int i = c.vid * MK_THREADS + c.tid; i < rows * per_row; i += c.G * MK_THREADS) {
      const int m = i / per_row;
      linear_group_out(st, sp, m, (i - m * per_row) * 8, n_out, [&](int col) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        const u32x4 *part = (const u32x4 *)(rt.group_part + ((size_t)q * MK_MAX_TOKENS + m) * ld + col);
#pragma unroll 4
        for (int z = 0; z < p.S; z++) v += __builtin_bit_cast(f32x4, ldc_16B(part + (size_t)z * portions * MK_MAX_TOKENS * ld / 4));
        return v;
      });
    }
  }
  c.wrote_through = true;
}

// ---- attention of several portions (MK_PAIR_BOTH on an ATTN stage), 128-wide heads
//
// First every portion's rows are prepared (q/k norm, rotation; keys and values into their pages, queries into a scratch), then, behind a barrier, all
// portions' tokens are attended at once, everything out of the pages.  Portions one after the other, each with a barrier, a write-back and an invalidate in
// between, prepared a portion's key and value rows in every unit of sixteen query rows: 512 tokens behind 1540 of 32 q / 8 kv heads 377 us as a stage, now 150.
//
// A task is up to two units of stage_attn_tiles, neighbouring token groups of one request and kv head: a cached tile, once in LDS, is scored against all
// their queries, and its values, read back transposed, are packed once.  Sums are made as that stage makes them: a unit's chunks are as many and end where
// they would for its portion alone, tile t of a chunk belongs to partial sum (t - first) mod 4, and those are merged in their order; as the chunks of the
// units begin at tiles of their own, a wavefront takes the tiles w, w + 4, ... of the request and tells each unit's sum which one it is in the end.
// (Four units a task: their queries and sums leave no registers for the tile, 180 us.)  Bound by one wavefront's chain through a tile: operands out of LDS,
// scores, weights, products.
__device__ __forceinline__ void lds_request(const void *p, unsigned lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off sc1" ::"v"((const MK_GLOBAL void *)(unsigned long long)p), "s"(lds) : "memory", "m0");
}
// Maximum over a column's four lanes, l & 15 + 16 i.
__device__ __forceinline__ float lanes_max(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const unsigned w = __float_as_uint(v);
  const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// Token groups and tasks of an iteration: bit t of a portion's word says that one begins at its row t.
struct GroupTasks {
  unsigned long long units[MK_GROUP], tasks[MK_GROUP];
  int per_task, quads;  // units of a task at most, tasks of a kv head
};
// False: some portion alone would take another form of the stage (few query rows, or units in pairs), or page lists are long: portions one after the other.
template <int QPK>
__device__ __forceinline__ bool attn_group_tasks(CStage &st, const Ctx &c, const MkRuntime &rt, int portions, const int *sh_rows, GroupTasks &g) {
  constexpr int TG = 16 / QPK;
  const int lane = threadIdx.x & 63;
  if ((rt.max_seq + rt.page_size - 1) / rt.page_size > MK_ATTN_PAIR_PAGES) return false;
  int lead[MK_GROUP], total = 0;
  bool ok = true;
#pragma unroll
  for (int p = 0; p < MK_GROUP; p++) {
    const int M = p < portions ? __builtin_amdgcn_readfirstlane(sh_rows[p]) : 0;
    lead[p] = lane < M ? lane - ldc_i32(&rt.tok_first[p * MK_MAX_TOKENS + lane]) : 1;
    ok = ok && (p >= portions || 2 * M * st.num_kv_heads >= c.G);
  }
#pragma unroll
  for (int p = 0; p < MK_GROUP; p++) {
    g.units[p] = __ballot(lead[p] % TG == 0);
    ok = ok && __popcll(g.units[p]) * st.num_kv_heads <= c.G;
    total += __popcll(g.units[p]) * st.num_kv_heads;
  }
  g.per_task = total > c.G ? 2 : 1;
  g.quads = 0;
#pragma unroll
  for (int p = 0; p < MK_GROUP; p++) {
    g.tasks[p] = __ballot(lead[p] % (TG * g.per_task) == 0);
    g.quads += __popcll(g.tasks[p]);
  }
  return ok;
}
template <int QPK>
__device__ __forceinline__ void stage_attn_group(Ctx &c, const MkRuntime &rt, int s, int portions, const int *sh_rows, const GroupTasks &g, char *smem) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  constexpr int D = 128, TG = 16 / QPK, NU = 2, RB = 3, PD = 132, GS = 1088, TS = 4 * GS, SLOT = 2 * TS;
  constexpr int PART_OFF = MK_WAVES * RB * SLOT, PAGE_OFF = PART_OFF + MK_WAVES * SLOT;  // tiles of every wavefront; new tiles, and partial sums; page list
  static_assert(PAGE_OFF + MK_ATTN_PAIR_PAGES * 4 <= MK_LDS_BYTES && MK_WAVES * 16 * PD * 4 <= MK_WAVES * SLOT, "attention scratch exceeds the LDS window");
  static_assert(MK_MAX_TOKENS == 16 * MK_WAVES, "a new tile for every wavefront");
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
  CStage &st = mk_portion_stages(rt, 0)[s];
  const int nkv = st.num_kv_heads, H = st.num_q_heads, ps = rt.page_size;
  const unsigned lds = (unsigned)(unsigned long long)(__attribute__((address_space(3))) char *)smem;
  auto base_of = [&](int p) { return rt.batch_n ? rt.batch_at[p] : 0; };
  // ---- rows: a wavefront stays with one portion, whose tokens are a lane each; eight head rows in flight
  {
    const int W = c.vid * MK_WAVES + wave, n_waves = c.G * MK_WAVES, p = W % portions, at = W / portions, step = (n_waves - p + portions - 1) / portions;
    const int M = __builtin_amdgcn_readfirstlane(sh_rows[p]), per = H + 2 * nkv, n = M * per;
    CStage &sp = mk_portion_stages(rt, p)[s];
    const int row = p * MK_MAX_TOKENS + min(lane, M - 1), pos = ldc_i32(&rt.tok_pos[row]), slot = ldc_i32(&rt.tok_slot[row]);
    const int page = rt.kv_indices[base_of(p) + ldc_i32(&rt.kv_indptr[slot]) + pos / ps];
    const size_t line = ((size_t)page * ps + pos % ps) * nkv;  // of the token's keys and values
    uint16_t w[2][2];
    if (st.flags & MK_F_QK_NORM) {
#pragma unroll
      for (int e = 0; e < 2; e++) {
        w[0][e] = ((const uint16_t *)st.q_norm_w)[lane + 64 * e];
        w[1][e] = ((const uint16_t *)st.k_norm_w)[lane + 64 * e];
      }
    }
    barrier_wait(c);
    const int S = c.defer_S;
    const float *part = c.defer_part + (size_t)p * MK_MAX_TOKENS * c.defer_n;
    const size_t slice = (size_t)c.defer_rows * c.defer_n;
    const int ld_part = c.defer_n;
    c.defer_S = 0;
    constexpr int RF = 8;
    for (int i0 = at; i0 < n; i0 += RF * step) {
      int tok[RF], head[RF];
      uint16_t cs[RF], sn[RF];
      float x[RF][2];
#pragma unroll
      for (int r = 0; r < RF; r++) {
        const int i = min(i0 + r * step, n - 1);
        tok[r] = i / per;
        head[r] = i - tok[r] * per;
        if (st.flags & MK_F_ROPE) {
          const size_t o = (size_t)__builtin_amdgcn_readlane(pos, tok[r]) * st.ld_cos;
          cs[r] = ((const uint16_t *)st.cos_tab + o)[lane];
          sn[r] = ((const uint16_t *)st.sin_tab + o)[lane];
        }
      }
      // (the heads of a kv head and, behind them, its key and value lie together)
      auto column = [&](int hd) { return hd < H ? (hd / QPK) * (QPK + 2) * D + hd % QPK * D : ((hd - H) % nkv) * (QPK + 2) * D + (QPK + (hd - H) / nkv) * D; };
      auto sum = [&](auto ns) {
        constexpr int NS = decltype(ns)::value;
        float q[RF][2][NS];
#pragma unroll
        for (int r = 0; r < RF; r++) {
          const float *pp = part + (size_t)tok[r] * ld_part + column(head[r]) + lane;
#pragma unroll
          for (int b = 0; b < NS; b++) {
            q[r][0][b] = ldc_f32(pp + b * slice);
            q[r][1][b] = ldc_f32(pp + b * slice + 64);
          }
        }
#pragma unroll
        for (int r = 0; r < RF; r++)
#pragma unroll
          for (int e = 0; e < 2; e++) {
            float v = 0.f;
#pragma unroll
            for (int b = 0; b < NS; b++) v += q[r][e][b];
            x[r][e] = bfround(v);
          }
      };
      if (S == 0) {
        uint16_t q[RF][2];
#pragma unroll
        for (int r = 0; r < RF; r++) {
          const uint16_t *pp = (const uint16_t *)sp.in + (size_t)tok[r] * sp.ld_in + column(head[r]) + lane;
          q[r][0] = ldc_u16(pp);
          q[r][1] = ldc_u16(pp + 64);
        }
#pragma unroll
        for (int r = 0; r < RF; r++) {
          x[r][0] = bf2f(q[r][0]);
          x[r][1] = bf2f(q[r][1]);
        }
      } else if (S == 2) {
        sum(std::integral_constant<int, 2>{});
      } else if (S == 4) {
        sum(std::integral_constant<int, 4>{});
      } else {
        sum(std::integral_constant<int, 8>{});
      }
#pragma unroll
      for (int r = 0; r < RF; r++) {
        if (i0 + r * step >= n) break;
        float x0 = x[r][0], x1 = x[r][1];
        const int kind = head[r] < H ? 0 : 1 + (head[r] - H) / nkv, h = (head[r] - H) % nkv;
        if (S) {  // (what the linear would have stored)
          uint16_t *d = (uint16_t *)sp.in + (size_t)tok[r] * sp.ld_in + column(head[r]);
          d[lane] = (uint16_t)f2bf(x0);
          d[lane + 64] = (uint16_t)f2bf(x1);
        }
        if (kind < 2) {
          if (st.flags & MK_F_QK_NORM) {
            const float ss = wave_sum(x0 * x0 + x1 * x1);
            const float f = rsqrtf(ss * (1.f / 128.f) + st.eps);
            x0 = bfround((x0 * f) * bf2f(kind ? w[1][0] : w[0][0]));
            x1 = bfround((x1 * f) * bf2f(kind ? w[1][1] : w[0][1]));
          }
          if (st.flags & MK_F_ROPE) {
            const float c_ = bf2f(cs[r]), s_ = bf2f(sn[r]);
            const float y0 = x0 * c_ - x1 * s_;
            const float y1 = x0 * s_ + x1 * c_;
            x0 = y0;
            x1 = y1;
          }
        }
        const size_t at_line = ((size_t)(unsigned)__builtin_amdgcn_readlane((int)line, tok[r]) | (size_t)(unsigned)__builtin_amdgcn_readlane((int)(line >> 32), tok[r]) << 32) + h;
        uint16_t *d = kind == 0 ? rt.group_q + ((size_t)(p * MK_MAX_TOKENS + tok[r]) * H + head[r]) * D : (uint16_t *)(kind == 1 ? st.k_cache : st.v_cache) + at_line * D;
        stc_u16(d + lane, (uint16_t)f2bf(x0));
        stc_u16(d + lane + 64, (uint16_t)f2bf(x1));
        if (kind == 0 && sp.q_ws) {
          uint16_t *q = (uint16_t *)sp.q_ws + (size_t)tok[r] * sp.ld_qws + (size_t)head[r] * D;
          q[lane] = (uint16_t)f2bf(x0);
          q[lane + 64] = (uint16_t)f2bf(x1);
        }
      }
    }
  }
  c.wrote_through = true;  // (what else was written nobody reads before the next iteration)
  barrier_arrive(c);
  // ---- tasks
  const int n_tasks = g.quads * nkv;
  if (c.vid >= n_tasks) barrier_wait(c);
  for (int u = c.vid; u < n_tasks; u += c.G) {
    int k = u % g.quads, p = 0;
    const int h = u / g.quads;  // (kv head outermost: its tasks sit on neighbouring workgroups, on one die where there are eight heads)
    unsigned long long begins = g.tasks[0];
    int n_units = __popcll(g.units[0]);
#pragma unroll
    for (int q = 0; q + 1 < MK_GROUP; q++)
      if (p == q && k >= __popcll(g.tasks[q])) {
        k -= __popcll(g.tasks[q]);
        p = q + 1;
        begins = g.tasks[q + 1];
        n_units = __popcll(g.units[q + 1]);
      }
    const bool mine = ((begins >> lane) & 1) && __popcll(begins & ((1ull << lane) - 1)) == k;
    const int t = (int)__ffsll(__ballot(mine)) - 1, M = __builtin_amdgcn_readfirstlane(sh_rows[p]);
    const int row = p * MK_MAX_TOKENS + min(lane, M - 1), my_first = ldc_i32(&rt.tok_first[row]), my_pos = ldc_i32(&rt.tok_pos[row]), my_slot = ldc_i32(&rt.tok_slot[row]);
    const int t0 = __builtin_amdgcn_readlane(my_first, t), p0 = __builtin_amdgcn_readlane(my_pos, t0), t_end = t0 + __popcll(__ballot(lane < M && my_first == t0));
    const int *pages = rt.kv_indices + base_of(p) + __builtin_amdgcn_readfirstlane(ldc_i32(&rt.kv_indptr[__builtin_amdgcn_readlane(my_slot, t)]));
    CStage &sp = mk_portion_stages(rt, p)[s];
    const int cmax = max(1, min(c.G / (n_units * nkv), MK_ATTN_MAX_CHUNKS)), nt = (p0 + 15) / 16, Cd = (nt + MK_WAVES - 1) / MK_WAVES + 1, C = min(Cd, cmax);
    int n_u[NU], new_u[NU];  // tokens of a unit, positions it sees that are new in its portion
#pragma unroll
    for (int e = 0; e < NU; e++) {
      const int first = t + e * TG;
      n_u[e] = e < g.per_task ? max(0, min(TG, t_end - first)) : 0;
      new_u[e] = n_u[e] ? first + n_u[e] - t0 : 0;
    }
    const int new_all = min(t + g.per_task * TG, t_end) - t0;
    // first tile of chunk `i` of unit `e` (see stage_attn_tiles)
    auto bound = [&](int e, int i) -> int {
      if (i >= C) return nt;
      if (C == Cd) return i < C - 1 ? (int)((long long)nt * i / (C - 1)) : nt;
      const int extra = 4 * MK_WAVES * ((n_u[e] * QPK + 2 * new_u[e] + 31) / 32 - 1), total = nt + (C > 1 ? min(extra, (nt + C - 2) / (C - 1)) : 0);
      return min(nt, (int)((long long)total * i / C));
    };
    int *spg = (int *)(smem + PAGE_OFF);
    lds_barrier();  // (LDS of the task in front)
    for (int i = tid; i <= (p0 + new_all - 1) / ps; i += MK_THREADS) spg[i] = pages[i];
    if (c.pending) barrier_wait(c);  // every row is where it belongs
    __syncthreads();
    const char *kc = (const char *)st.k_cache, *vc = (const char *)st.v_cache;
    const float scale = st.sm_scale_log2;
    // positions [q0, q0 + 16), none behind `last` (read again instead), as a tile at LDS byte b: values, then keys, each four groups of four rows.  Where pages are
    // powers of two and hold whole tiles, a whole tile of the cache is one address and its lanes' distances (new tiles begin anywhere).
    const int shift = 31 - __builtin_clz(ps);
    const bool plain = ps >= 16 && (ps & (ps - 1)) == 0;
    unsigned apart[4];
#pragma unroll
    for (int r = 0; r < 4; r++) apart[r] = (unsigned)((4 * r + lg) * nkv) * (2 * D) + lr * 16;
    auto load_rows = [&](int q0, int last, unsigned b) {
      if (plain && (q0 & 15) == 0 && q0 + 15 <= last) {
        const size_t at = (((size_t)__builtin_amdgcn_readfirstlane(spg[q0 >> shift]) * ps + (q0 & (ps - 1))) * nkv + h) * (2 * D);
#pragma unroll
        for (int r = 0; r < 4; r++) lds_request(kc + at, apart[r], b + TS + r * GS);
#pragma unroll
        for (int r = 0; r < 4; r++) lds_request(vc + at, apart[r], b + r * GS);
      } else {
        size_t at[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int pc = min(q0 + 4 * r + lg, last), pg = pc / ps;
          at[r] = (((size_t)spg[pg] * ps + (pc - pg * ps)) * nkv + h) * (2 * D) + lr * 16;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) lds_request(kc + at[r], b + TS + r * GS);
#pragma unroll
        for (int r = 0; r < 4; r++) lds_request(vc + at[r], b + r * GS);
      }
    };
    const unsigned buf = lds + wave * (RB * SLOT);
    bf16x8 qb[NU][4];
#pragma unroll
    for (int e = 0; e < NU; e++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int col = min(lr, max(n_u[e], 1) * QPK - 1);
        const u32x4 z = {0u, 0u, 0u, 0u};
        const u32x4 v = ldc_16B((const u32x4 *)(rt.group_q + ((size_t)(p * MK_MAX_TOKENS + min(t + e * TG, t_end - 1) + col / QPK) * H + h * QPK + col % QPK) * D + r * 32 + lg * 8));
        qb[e][r] = __builtin_bit_cast(bf16x8, lr < n_u[e] * QPK ? v : z);
      }
    f32x4 o[NU][8];
    float mrun[NU], lsum[NU], cm[NU], cl[NU], cv[NU][8];
#pragma unroll
    for (int e = 0; e < NU; e++) {
      cm[e] = -1e30f;
      cl[e] = 0.f;
#pragma unroll
      for (int d = 0; d < 8; d++) cv[e][d] = 0.f;
    }
    const int md = (tid & 15) * 8, mcol = tid >> 4;  // dims and column of a thread where sums are merged
    for (int ci = 0; ci < C; ci++) {
      int tb[NU], te[NU], lo = nt, hi = 0, all_b = 0, all_e = nt;  // a unit's tiles; those of some unit, and of all of them
#pragma unroll
      for (int e = 0; e < NU; e++) {
        tb[e] = n_u[e] ? bound(e, ci) : nt;
        te[e] = n_u[e] ? bound(e, ci + 1) : 0;
        if (n_u[e] && te[e] > tb[e]) {
          lo = min(lo, tb[e]);
          hi = max(hi, te[e]);
        }
        all_b = max(all_b, tb[e]);
        all_e = min(all_e, te[e]);
#pragma unroll
        for (int dt = 0; dt < 8; dt++) o[e][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
        mrun[e] = -INFINITY;
        lsum[e] = 0.f;
      }
      // scores of units [0, N) with the keys kf of positions [q0, q0 + 16), those up to `last` (the lane's own) seen: weights in pw, the units' maxima and sums, and
      // what has been summed, brought up to them.  (All units together: one's chain of dependent instructions, the maximum over the wavefront among them, is
      // longer than what it issues.)
      auto weigh = [&](auto first_c, auto count_c, const bf16x8 (&kf)[4], int q0, int last, float (&pw)[NU][4]) {
        constexpr int E0 = decltype(first_c)::value, E1 = E0 + decltype(count_c)::value;
        f32x4 s4[NU];
        float mx[NU], alpha[NU];
#pragma unroll
        for (int e = E0; e < E1; e++) s4[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int e = E0; e < E1; e++) s4[e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[r], qb[e][r], s4[e], 0, 0, 0);
#pragma unroll
        for (int e = E0; e < E1; e++) {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const float v = s4[e][r] * scale;
            pw[e][r] = q0 + lg * 4 + r <= last ? v : -INFINITY;
          }
          mx[e] = fmaxf(fmaxf(pw[e][0], pw[e][1]), fmaxf(pw[e][2], pw[e][3]));
        }
#pragma unroll
        for (int e = E0; e < E1; e++) mx[e] = lanes_max(mx[e]);
        bool moved = false;
#pragma unroll
        for (int e = E0; e < E1; e++) {
          const float mn = fmaxf(mrun[e], mx[e]);
          alpha[e] = __builtin_amdgcn_exp2f(mrun[e] - mn);
#pragma unroll
          for (int r = 0; r < 4; r++) pw[e][r] = __builtin_amdgcn_exp2f(pw[e][r] - mn);
          lsum[e] = lsum[e] * alpha[e] + ((pw[e][0] + pw[e][1]) + (pw[e][2] + pw[e][3]));
          mrun[e] = mn;
          moved = moved || alpha[e] != 1.f;
        }
        if (__ballot(moved)) {  // (uniform) some column's maximum moved: rescale what has been summed
#pragma unroll
          for (int e = E0; e < E1; e++) {
            float ar[4];
#pragma unroll
            for (int r = 0; r < 4; r++) ar[r] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lg * 4 + r) << 2, __builtin_bit_cast(int, alpha[e])));
#pragma unroll
            for (int dt = 0; dt < 8; dt++)
#pragma unroll
              for (int r = 0; r < 4; r++) o[e][dt][r] *= ar[r];
          }
        }
      };
      auto terms = [&](float (&pw)[4], auto &wt) {  // bf16 terms of the weights
#pragma unroll
        for (int q = 0; q < (int)(sizeof(wt) / sizeof(wt[0])); q++) {
          float ph[4];
#pragma unroll
          for (int r = 0; r < 4; r++) {
            ph[r] = bfround(pw[r]);
            pw[r] -= ph[r];  // (exact)
          }
          wt[q] = __builtin_bit_cast(s16x4, (unsigned long long)pack2(ph[0], ph[1]) | ((unsigned long long)pack2(ph[2], ph[3]) << 32));
        }
      };
      auto keys = [&](const char *b, bf16x8 (&kf)[4]) {
        const char *kl = b + TS + (lr >> 2) * GS + (lr & 3) * 256 + lg * 16;
#pragma unroll
        for (int r = 0; r < 4; r++) kf[r] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(kl + r * 64));
      };
      auto pack4 = [](unsigned v0, unsigned v1, unsigned v2, unsigned v3) { return __builtin_bit_cast(s16x4, (unsigned long long)(v0 | (v1 << 16)) | ((unsigned long long)(v2 | (v3 << 16)) << 32)); };
      auto each = [&](auto f) {
        f(std::integral_constant<int, 0>{});
        f(std::integral_constant<int, 1>{});
      };
      // ---- cached tiles of this wavefront, RB - 1 requested ahead (the last one again behind the end)
      int t_ = lo + ((wave - lo) & (MK_WAVES - 1));
      const int t_last = hi - 1 - ((hi - 1 - wave) & (MK_WAVES - 1));
      const bool some = t_ < hi;
      auto load_tile = [&](int tt, int b) { load_rows(min(tt, t_last) * 16, p0 - 1, buf + b * SLOT); };
      if (some) {
#pragma unroll
        for (int b = 0; b < RB - 1; b++) load_tile(t_ + b * MK_WAVES, b);
      }
      const bool with_new = ci == C - 1;
      if (with_new) {
        lds_barrier();  // (partial sums of the chunk in front have been read)
        if (wave * 16 < new_all) load_rows(p0 + wave * 16, p0 + new_all - 1, lds + PART_OFF + wave * SLOT);
      }
      bool more = some;
      while (more) {
#pragma unroll
        for (int b = 0; b < RB; b++) {
          load_tile(t_ + (RB - 1) * MK_WAVES, (b + RB - 1) % RB);
          static_assert(RB == 3, "the wait counts two tiles' requests");
          asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
          if (more) {
            const char *vb = smem + wave * (RB * SLOT) + b * SLOT;
            bf16x8 kf[4];
            keys(vb, kf);
            unsigned v[8][4];
            const char *vl = vb + lg * GS + lr * 2;
#pragma unroll
            for (int dt = 0; dt < 8; dt++)
#pragma unroll
              for (int r = 0; r < 4; r++) v[dt][r] = *(const uint16_t *)(vl + dt * 32 + r * 256);
            __builtin_amdgcn_sched_barrier(0);  // (all of them in flight; else the compiler reads and waits value by value)
            s16x4 bv[8];
            auto pack_values = [&]() {
#pragma unroll
              for (int dt = 0; dt < 8; dt++) bv[dt] = pack4(v[dt][0], v[dt][1], v[dt][2], v[dt][3]);
            };
            auto units = [&](auto first_c, auto count_c) {
              constexpr int E0 = decltype(first_c)::value, E1 = E0 + decltype(count_c)::value;
              float pw[NU][4];
              weigh(first_c, count_c, kf, t_ * 16, p0 - 1, pw);
              pack_values();
              s16x4 wt[NU][2];
#pragma unroll
              for (int e = E0; e < E1; e++) terms(pw[e], wt[e]);
#pragma unroll
              for (int dt = 0; dt < 8; dt++)
#pragma unroll
                for (int q = 0; q < 2; q++)
#pragma unroll
                  for (int e = E0; e < E1; e++) o[e][dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wt[e][q], bv[dt], o[e][dt], 0, 0, 0);
            };
            using std::integral_constant;
            if (t_ >= all_b && t_ < all_e && n_u[NU - 1]) {
              units(integral_constant<int, 0>{}, integral_constant<int, NU>{});
            } else {
              each([&](auto unit) {
                constexpr int e = decltype(unit)::value;
                if (t_ >= tb[e] && t_ < te[e]) units(unit, integral_constant<int, 1>{});
              });
            }
            t_ += MK_WAVES;
            more = t_ < hi;
          }
        }
      }
      // ---- new tiles: one of them, at most, belongs to a wavefront's partial sum of a unit
      if (with_new) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        each([&](auto unit) {
          constexpr int e = decltype(unit)::value;
          const int sw = (wave - tb[e]) & (MK_WAVES - 1);
          if (sw * 16 >= new_u[e]) return;
          const int q0 = p0 + sw * 16, newest = p0 + new_u[e] - 1, p_first = newest + 1 - n_u[e], n_cols = n_u[e] * QPK;
          const char *vb = smem + PART_OFF + sw * SLOT, *vl = vb + lg * GS + lr * 2;
          bf16x8 kf[4];
          keys(vb, kf);
          float pws[NU][4];
          weigh(unit, std::integral_constant<int, 1>{}, kf, q0, p_first + min(lr, n_cols - 1) / QPK, pws);
          auto &pw = pws[e];
          // (rows behind the unit's newest position count as zeros)
          s16x4 bv[8];
          unsigned top = 0;
#pragma unroll
          for (int dt = 0; dt < 8; dt++) {
            unsigned v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
              v[r] = q0 + lg * 4 + r <= newest ? *(const uint16_t *)(vl + dt * 32 + r * 256) : 0u;
              top |= (v[r] & 0x7f80u) + 0x80u;
            }
            bv[dt] = pack4(v[0], v[1], v[2], v[3]);
          }
          if (__builtin_expect(__ballot(top & 0x8000u) != 0, 0)) {  // values that are not finite: column by column, see stage_attn_tiles
            for (int g4 = 0; g4 < 4; g4++) {
#pragma unroll
              for (int r4 = 0; r4 < 4; r4++) {
                const uint16_t *v = (const uint16_t *)(vb + g4 * GS + r4 * 256) + lr;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                  const int col = lg * 4 + r;
                  const float wgt = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((g4 * 16 + col) << 2, __builtin_bit_cast(int, pw[r4])));
                  const bool seen = q0 + g4 * 4 + r4 <= p_first + min(col, n_cols - 1) / QPK;
#pragma unroll
                  for (int dt = 0; dt < 8; dt++) o[e][dt][r] = seen ? fmaf(wgt, bf2f(v[dt * 16]), o[e][dt][r]) : o[e][dt][r];
                }
              }
            }
            return;
          }
          s16x4 wt[3];
          terms(pw, wt);
#pragma unroll
          for (int dt = 0; dt < 8; dt++)
#pragma unroll
            for (int q = 0; q < 3; q++) o[e][dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wt[q], bv[dt], o[e][dt], 0, 0, 0);
        });
      }
      // ---- a unit's four partial sums, in their order, then its chunks
      float *parts = (float *)(smem + PART_OFF);
      each([&](auto unit) {
        constexpr int e = decltype(unit)::value;
        if (!n_u[e]) return;
        const int sw = (wave - tb[e]) & (MK_WAVES - 1);
        float lt = lsum[e];
        lt += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 16) << 2, __builtin_bit_cast(int, lt)));
        lt += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, lt)));
        lds_barrier();
        float *part = parts + sw * 16 * PD;
        if (lg == 0) {
          part[lr * PD + D] = mrun[e];
          part[lr * PD + D + 1] = lt;
        }
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int dt = 0; dt < 8; dt++) part[(lg * 4 + r) * PD + dt * 16 + lr] = o[e][dt][r];
        lds_barrier();
        float mx = -1e30f, ls = 0.f, os[8];
#pragma unroll
        for (int d = 0; d < 8; d++) os[d] = 0.f;
#pragma unroll
        for (int w = 0; w < MK_WAVES; w++) mx = fmaxf(mx, parts[(w * 16 + mcol) * PD + D]);
#pragma unroll
        for (int w = 0; w < MK_WAVES; w++) {
          const float *pp = parts + (w * 16 + mcol) * PD;
          const float wgt = __builtin_amdgcn_exp2f(pp[D] - mx);
          ls += pp[D + 1] * wgt;
#pragma unroll
          for (int d = 0; d < 8; d++) os[d] += pp[md + d] * wgt;
        }
        if (C == 1) {
          cl[e] = ls;
#pragma unroll
          for (int d = 0; d < 8; d++) cv[e][d] = os[d];
        } else {
          const float mn = fmaxf(cm[e], mx);
          const float sa = __builtin_amdgcn_exp2f(cm[e] - mn), sb = __builtin_amdgcn_exp2f(mx - mn);
          cl[e] = cl[e] * sa + ls * sb;
#pragma unroll
          for (int d = 0; d < 8; d++) cv[e][d] = cv[e][d] * sa + os[d] * sb;
          cm[e] = mn;
        }
      });
    }
#pragma unroll
    for (int e = 0; e < NU; e++)
      if (mcol < n_u[e] * QPK) {
        u32x4 r;
#pragma unroll
        for (int d = 0; d < 4; d++) r[d] = pack2(cv[e][2 * d] / cl[e], cv[e][2 * d + 1] / cl[e]);
        uint16_t *orow = (uint16_t *)sp.out + (size_t)(t + e * TG + mcol / QPK) * st.ld_out + (size_t)(h * QPK + mcol % QPK) * D + md;
#pragma unroll
        for (int d = 0; d < 4; d++) __hip_atomic_store((MK_GLOBAL uint32_t *)(unsigned long long)(orow + 2 * d), r[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
  }
  c.wrote_through = true;
}
