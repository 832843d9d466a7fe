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

// Positions and first page-table entries of all portions' tokens (first rows as well, if somewhere), MK_MAX_TOKENS a portion, in LDS.
__device__ __forceinline__ void group_tokens(const MkRuntime &rt, int portions, const int *sh_rows, int *pos, int *pages, int *first = nullptr) {
  constexpr int N = MK_GROUP * MK_MAX_TOKENS / MK_THREADS;
  int x[N], slot[N], f[N];
  auto there = [&](int j) {
    const int i = threadIdx.x + j * MK_THREADS;
    return i < portions * MK_MAX_TOKENS && (i & (MK_MAX_TOKENS - 1)) < sh_rows[i / MK_MAX_TOKENS];
  };
  // (each of the three together: one token behind the other is four trips to memory instead of two)
#pragma unroll
  for (int j = 0; j < N; j++) {
    const int i = there(j) ? threadIdx.x + j * MK_THREADS : 0;
    x[j] = ldc_i32(&rt.tok_pos[i]);
    slot[j] = ldc_i32(&rt.tok_slot[i]);
    f[j] = first ? ldc_i32(&rt.tok_first[i]) : 0;
  }
#pragma unroll
  for (int j = 0; j < N; j++) slot[j] = ldc_i32(&rt.kv_indptr[slot[j]]);
#pragma unroll
  for (int j = 0; j < N; j++) {
    const int i = threadIdx.x + j * MK_THREADS;
    if (!there(j)) continue;
    pos[i] = x[j];
    pages[i] = (rt.batch_n ? rt.batch_at[i / MK_MAX_TOKENS] : 0) + slot[j];
    if (first) first[i] = f[j];
  }
  __syncthreads();
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

// ---- norms of several portions' rows (MK_PAIR_BOTH on a NORM or FX_ADDNORM stage)
//
// The rows of all portions, one portion's behind the other's, are dealt round the dies as one portion's are; a workgroup has two in flight, whose sums over it
// are taken together.  Bound by the barrier and by round trips: 512 rows of 4096 values from four slices, portion by portion, a row at a time, 20 us, now 13.
struct GroupRow {
  int portion, row;
  bool valid;
};
// Row i of all (the last one, not valid, where there are fewer).
__device__ __forceinline__ GroupRow group_row(int i, int portions, const int *sh_rows) {
  int p = 0;
  while (p + 1 < portions) {
    const int M = __builtin_amdgcn_readfirstlane(sh_rows[p]);
    if (i < M) break;
    i -= M;
    p++;
  }
  const int last = __builtin_amdgcn_readfirstlane(sh_rows[p]) - 1;
  return {p, min(i, last), i <= last};
}
__device__ __forceinline__ int group_rows(int portions, const int *sh_rows) {
  int n = 0;
  for (int p = 0; p < portions; p++) n += __builtin_amdgcn_readfirstlane(sh_rows[p]);
  return n;
}
// Sums over the workgroup of one value a thread, of two rows (see block_sum).
__device__ __forceinline__ void block_sums(float (&v)[2], float *red) {
  v[0] = wave_sum(v[0]);
  v[1] = wave_sum(v[1]);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = v[0];
    red[4 + (threadIdx.x >> 6)] = v[1];
  }
  __syncthreads();
#pragma unroll
  for (int z = 0; z < 2; z++) v[z] = red[4 * z] + red[4 * z + 1] + red[4 * z + 2] + red[4 * z + 3];
}
// Residual rows of the linear that left its sum, of a portion.
__device__ __forceinline__ const void *group_residual(const Ctx &c, const MkRuntime &rt, int portion) {
  CStage &sum = mk_portion_stages(rt, portion)[c.defer_stage];
  return sum.flags & MK_F_RES ? sum.res : nullptr;
}
template <int NS>
__device__ __forceinline__ void norm_group_rows(Ctx &c, const MkRuntime &rt, int s, int portions, const int *sh_rows, char *smem) {
  CStage &st = mk_portion_stages(rt, 0)[s];
  const int tid = c.tid, k8 = st.k / 8;
  float *red = (float *)smem;
  const u32x4 *w4 = (const u32x4 *)st.norm_w;
  auto at = [&](int j) { return min(tid + j * MK_THREADS, k8 - 1); };
  auto on = [&](int j) { return NS <= 2 || j * MK_THREADS < k8; };
  u32x4 g[NS];
#pragma unroll
  for (int j = 0; j < NS; j++)
    if (on(j)) g[j] = w4[at(j)];
  barrier_wait(c);
  const int dS = c.defer_S, total = group_rows(portions, sh_rows);
  c.defer_S = 0;
  auto rows = [&](auto ns) {
    constexpr int Q = decltype(ns)::value, JB = Q && NS * Q <= 8 ? NS : 1;  // segments requested together
    for (int i = row_item(c); i < total; i += 2 * c.G) {
      GroupRow r[2];
      const u32x4 *x[2], *res[2];
      u32x4 v[2][NS];
#pragma unroll
      for (int z = 0; z < 2; z++) {
        r[z] = group_row(i + z * c.G, portions, sh_rows);
        x[z] = (const u32x4 *)((const uint16_t *)mk_portion_stages(rt, r[z].portion)[s].in + (size_t)r[z].row * st.ld_in);
        res[z] = Q ? (const u32x4 *)group_residual(c, rt, r[z].portion) : nullptr;
        if (res[z]) res[z] = (const u32x4 *)((const uint16_t *)res[z] + (size_t)r[z].row * c.defer_ld_res);
      }
      if constexpr (Q == 0) {
#pragma unroll
        for (int z = 0; z < 2; z++)
#pragma unroll
          for (int j = 0; j < NS; j++)
            if (on(j)) v[z][j] = ldc_16B(x[z] + at(j));
      } else {  // (the rows are still K-slice partials: see stage_norm_rows)
#pragma unroll
        for (int j0 = 0; j0 < NS; j0 += JB) {
          if (!on(j0)) continue;
          u32x4 pv[2][JB][Q][2], rv[2][JB];
#pragma unroll
          for (int z = 0; z < 2; z++) {
            __amdgpu_buffer_rsrc_t part[Q];
#pragma unroll
            for (int q = 0; q < Q; q++) part[q] = dev_rows(c.defer_part + ((size_t)q * c.defer_rows + r[z].portion * MK_MAX_TOKENS + r[z].row) * st.k);
#pragma unroll
            for (int j = 0; j < JB; j++) {
              const int seg = at(j0 + j);
              rv[z][j] = ldc_16B(res[z] ? res[z] + seg : (const u32x4 *)c.defer_part);
#pragma unroll
              for (int q = 0; q < Q; q++) {
                pv[z][j][q][0] = ldc_16B(part[q], seg * 32);
                pv[z][j][q][1] = ldc_16B(part[q], seg * 32 + 16);
              }
            }
          }
#pragma unroll
          for (int z = 0; z < 2; z++)
#pragma unroll
            for (int j = 0; j < JB; j++) {
              float a[8];
#pragma unroll
              for (int e = 0; e < 8; e++) a[e] = 0.f;
#pragma unroll
              for (int q = 0; q < Q; q++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                  a[e] += __uint_as_float(pv[z][j][q][0][e]);
                  a[4 + e] += __uint_as_float(pv[z][j][q][1][e]);
                }
              if (res[z]) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                  a[2 * e] += bf_lo(rv[z][j][e]);
                  a[2 * e + 1] += bf_hi(rv[z][j][e]);
                }
              }
#pragma unroll
              for (int e = 0; e < 4; e++) v[z][j0 + j][e] = pack2(a[2 * e], a[2 * e + 1]);
            }
        }
#pragma unroll
        for (int z = 0; z < 2; z++)
#pragma unroll
          for (int j = 0; j < NS; j++)
            if (r[z].valid && tid + j * MK_THREADS < k8) stc_16B((u32x4 *)x[z] + tid + j * MK_THREADS, v[z][j]);
      }
      float ss[2] = {0.f, 0.f};
#pragma unroll
      for (int z = 0; z < 2; z++)
#pragma unroll
        for (int j = 0; j < NS; j++) {
          if (!on(j)) continue;
          const bool ok = tid + j * MK_THREADS < k8;
#pragma unroll
          for (int e = 0; e < 4; e++) ss[z] += ok ? bf_lo(v[z][j][e]) * bf_lo(v[z][j][e]) + bf_hi(v[z][j][e]) * bf_hi(v[z][j][e]) : 0.f;
        }
      block_sums(ss, red);
#pragma unroll
      for (int z = 0; z < 2; z++) {
        const float f = rsqrtf(ss[z] / (float)st.k + st.eps);
        u32x4 *y = (u32x4 *)((uint16_t *)mk_portion_stages(rt, r[z].portion)[s].out + (size_t)r[z].row * st.ld_out);
#pragma unroll
        for (int j = 0; j < NS; j++)
          if (r[z].valid && tid + j * MK_THREADS < k8) {
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = pack2((bf_lo(v[z][j][e]) * f) * bf_lo(g[j][e]), (bf_hi(v[z][j][e]) * f) * bf_hi(g[j][e]));
            stc_16B(y + tid + j * MK_THREADS, o);
          }
      }
      __syncthreads();
    }
  };
  if (dS == 0) rows(std::integral_constant<int, 0>{});
  else if (dS == 2) rows(std::integral_constant<int, 2>{});
  else if (dS == 4) rows(std::integral_constant<int, 4>{});
  else rows(std::integral_constant<int, 8>{});
  c.wrote_through = true;
}
__device__ __forceinline__ void stage_norm_group(CStage &st, Ctx &c, const MkRuntime &rt, int s, int portions, const int *sh_rows, char *smem) {
  if (st.k / 8 <= MK_THREADS) norm_group_rows<1>(c, rt, s, portions, sh_rows, smem);
  else if (st.k / 8 <= 2 * MK_THREADS) norm_group_rows<2>(c, rt, s, portions, sh_rows, smem);
  else norm_group_rows<6>(c, rt, s, portions, sh_rows, smem);
}

// ---- attention of several portions (MK_PAIR_BOTH on an ATTN stage), 128-wide heads
//
// First every portion's rows are prepared (q/k norm, rotation; keys and values into their pages, queries into a scratch), then, behind a barrier, all
// portions' tokens are attended at once, everything out of the pages.  Portions one after the other, each with a barrier, a write-back and an invalidate in
// between, prepared a portion's key and value rows in every unit of sixteen query rows: 512 tokens of 32 q / 8 kv heads, as a stage, were 377 us
// behind 1540 positions; now 132 behind about 2000 (112 behind 1536, by themselves).
//
// A task is up to two units of stage_attn_tiles, neighbouring token groups of one request and kv head: a cached tile, once in LDS, is scored against all
// their queries, and its values, read back transposed, are packed once.  Sums are made as that stage makes them: a unit's chunks are as many and end where
// they would for its portion alone, tile t of a chunk belongs to partial sum (t - first) mod 4, and those are merged in their order; as the chunks of the
// units begin at tiles of their own, a wavefront takes the tiles w, w + 4, ... of the request and tells each unit's sum which one it is in the end.
// (Four units a task: their queries and sums leave no registers for the tile, 180 us.)  Bound by what a wavefront issues for a tile of sixteen positions and two units, about 1 us: scores,
// 16 exponentials, 64 sums scaled, weights in two terms, products.  (512 tokens alone, us behind 0 / 512 / 1536 / 3072 positions: 72 / 104 / 162 / 231 with the sums
// among the accumulation registers, scaled only where a maximum moved, and heads of a kv group on all dies; 62 / 80 / 114 / 168 with what add_products says, now 63 / 79 / 112 / 161.)
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void lds_request(const void *p, unsigned lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off sc1" ::"v"((const MK_GLOBAL void *)(unsigned long long)p), "s"(lds) : "memory", "m0");
}
// o[dt] += values of 16 dims by weights of 16 columns, for the eight tiles of dims of a head: lane l holds column l & 15, dims 16 dt + 4 (l >> 4) .. + 3.  In
// assembly, which keeps the sums among the vector registers: the compiler puts what matrix instructions write among the others in a kernel of this size, and
// every tile scales all of them, which is two more instructions a value there (64 of them: 0.3 us a tile).  It knows nothing of how long these instructions
// write, so the last of them is waited for.
#define MK_PV(i, w) "v_mfma_f32_16x16x16_bf16 %" #i ", %[v" #i "], %[" #w "], %" #i "\n\t"
#define MK_PV8(w) MK_PV(0, w) MK_PV(1, w) MK_PV(2, w) MK_PV(3, w) MK_PV(4, w) MK_PV(5, w) MK_PV(6, w) MK_PV(7, w)
#define MK_PV_SUMS "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]), "+v"(o[4]), "+v"(o[5]), "+v"(o[6]), "+v"(o[7])
#define MK_PV_VALUES [v0] "v"(v[0]), [v1] "v"(v[1]), [v2] "v"(v[2]), [v3] "v"(v[3]), [v4] "v"(v[4]), [v5] "v"(v[5]), [v6] "v"(v[6]), [v7] "v"(v[7])
__device__ __forceinline__ void add_products(f32x4 (&o)[8], const s16x4 (&v)[8], s16x4 w) {
  asm volatile("s_nop 3\n\t" MK_PV8(w) "s_nop 11" : MK_PV_SUMS : MK_PV_VALUES, [w] "v"(w));
}
__device__ __forceinline__ void add_products(f32x4 (&o)[8], const s16x4 (&v)[8], const s16x4 (&w)[2]) {
  asm volatile("s_nop 3\n\t" MK_PV8(w0) MK_PV8(w1) "s_nop 11" : MK_PV_SUMS : MK_PV_VALUES, [w0] "v"(w[0]), [w1] "v"(w[1]));
}
#undef MK_PV
#undef MK_PV8
#undef MK_PV_SUMS
#undef MK_PV_VALUES
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
  constexpr int D = 128, TG = 16 / QPK, NU = 2, RB = 3, PD = 132, GS = 1056, TS = 4 * GS, SLOT = 2 * TS;
  // LDS: tiles of every wavefront, and the second unit's partial sums; new tiles, and the first unit's; page lists of this task and the next; the tokens' positions,
  // first rows and first page-table entries
  constexpr int PART_OFF = MK_WAVES * RB * SLOT, PAGE_OFF = PART_OFF + MK_WAVES * SLOT, ROWS_OFF = PAGE_OFF + 2 * MK_ATTN_PAIR_PAGES * 4, ROWS = MK_GROUP * MK_MAX_TOKENS;
  static_assert(ROWS_OFF + 3 * ROWS * 4 <= MK_LDS_BYTES && 16 * PD * 4 <= SLOT && NU == 2, "attention scratch exceeds the LDS window");
  static_assert(MK_MAX_TOKENS == 16 * MK_WAVES, "a new tile for every wavefront");
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
  CStage &st = mk_portion_stages(rt, 0)[s];
  const int nkv = st.num_kv_heads, H = st.num_q_heads, ps = rt.page_size;
  const unsigned lds = (unsigned)(unsigned long long)(__attribute__((address_space(3))) char *)smem;
  int *tab = (int *)(smem + ROWS_OFF);
  group_tokens(rt, portions, sh_rows, tab, tab + 2 * ROWS, tab + ROWS);
  // ---- rows: a wavefront stays with one portion, whose tokens are a lane each; eight head rows in flight
  {
    const int W = c.vid * MK_WAVES + wave, n_waves = c.G * MK_WAVES, p = W % portions, at = W / portions, step = (n_waves - p + portions - 1) / portions;
    const int M = __builtin_amdgcn_readfirstlane(sh_rows[p]), per = H + 2 * nkv, n = M * per;
    CStage &sp = mk_portion_stages(rt, p)[s];
    const int row = p * MK_MAX_TOKENS + min(lane, M - 1), pos = tab[row], page = rt.kv_indices[tab[2 * ROWS + row] + pos / ps];
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
    // (the heads of a kv head and, behind them, its key and value lie together)
    auto column = [&](int hd) { return hd < H ? (hd / QPK) * (QPK + 2) * D + hd % QPK * D : ((hd - H) % nkv) * (QPK + 2) * D + (QPK + (hd - H) / nkv) * D; };
    // RF rows at a time, while the next RF are on their way: 24 of them a wavefront are all requested before the first is stored (a load that is waited for
    // behind a store waits for the store as well; eight at a time, one after the other, took 21 us)
    auto rows = [&](auto ns) {
      constexpr int NS = decltype(ns)::value, NQ = NS ? NS : 1, RF = NS > 4 ? 4 : 12;
      struct Rows {
        float q[RF][2][NQ];
        uint16_t cs[RF], sn[RF];
      } r0, r1;
      auto row_at = [&](int i0, int r, int &tok, int &head) {
        const int i = min(i0 + r * step, n - 1);
        tok = i / per;
        head = i - tok * per;
      };
      auto request = [&](int i0, Rows &w) {
#pragma unroll
        for (int r = 0; r < RF; r++) {
          int tok, head;
          row_at(i0, r, tok, head);
          if constexpr (NS == 0) {
            const uint16_t *pp = (const uint16_t *)sp.in + (size_t)tok * sp.ld_in + column(head) + lane;
            w.q[r][0][0] = bf2f(ldc_u16(pp));
            w.q[r][1][0] = bf2f(ldc_u16(pp + 64));
          } else {
            const float *pp = part + (size_t)tok * ld_part + column(head) + lane;
#pragma unroll
            for (int b = 0; b < NS; b++) {
              w.q[r][0][b] = ldc_f32(pp + b * slice);
              w.q[r][1][b] = ldc_f32(pp + b * slice + 64);
            }
          }
          const size_t o = st.flags & MK_F_ROPE ? (size_t)__builtin_amdgcn_readlane(pos, tok) * st.ld_cos : 0;
          if (st.flags & MK_F_ROPE) {
            w.cs[r] = ((const uint16_t *)st.cos_tab + o)[lane];
            w.sn[r] = ((const uint16_t *)st.sin_tab + o)[lane];
          }
        }
      };
      auto finish = [&](int i0, const Rows &in) {
#pragma unroll
        for (int r = 0; r < RF; r++) {
          if (i0 + r * step >= n) break;
          int tok, head;
          row_at(i0, r, tok, head);
          float x0 = in.q[r][0][0], x1 = in.q[r][1][0];
          const int kind = head < H ? 0 : 1 + (head - H) / nkv, h = (head - H) % nkv;
          if constexpr (NS > 0) {
            x0 = x1 = 0.f;
#pragma unroll
            for (int b = 0; b < NS; b++) {
              x0 += in.q[r][0][b];
              x1 += in.q[r][1][b];
            }
            x0 = bfround(x0);
            x1 = bfround(x1);
            uint16_t *d = (uint16_t *)sp.in + (size_t)tok * sp.ld_in + column(head);  // (what the linear would have stored)
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
              const float c_ = bf2f(in.cs[r]), s_ = bf2f(in.sn[r]);
              const float y0 = x0 * c_ - x1 * s_;
              const float y1 = x0 * s_ + x1 * c_;
              x0 = y0;
              x1 = y1;
            }
          }
          const size_t at_line = ((size_t)(unsigned)__builtin_amdgcn_readlane((int)line, tok) | (size_t)(unsigned)__builtin_amdgcn_readlane((int)(line >> 32), tok) << 32) + h;
          uint16_t *d = kind == 0 ? rt.group_q + ((size_t)(p * MK_MAX_TOKENS + tok) * H + head) * D : (uint16_t *)(kind == 1 ? st.k_cache : st.v_cache) + at_line * D;
          stc_u16(d + lane, (uint16_t)f2bf(x0));
          stc_u16(d + lane + 64, (uint16_t)f2bf(x1));
          if (kind == 0 && sp.q_ws) {
            uint16_t *q = (uint16_t *)sp.q_ws + (size_t)tok * sp.ld_qws + (size_t)head * D;
            q[lane] = (uint16_t)f2bf(x0);
            q[lane + 64] = (uint16_t)f2bf(x1);
          }
        }
      };
      if (at < n) request(at, r0);
      for (int i0 = at; i0 < n; i0 += 2 * RF * step) {
        if (i0 + RF * step < n) request(i0 + RF * step, r1);
        __builtin_amdgcn_sched_barrier(0);
        finish(i0, r0);
        if (i0 + 2 * RF * step < n) request(i0 + 2 * RF * step, r0);
        __builtin_amdgcn_sched_barrier(0);
        finish(i0 + RF * step, r1);
      }
    };
    if (S == 0) rows(std::integral_constant<int, 0>{});
    else if (S == 2) rows(std::integral_constant<int, 2>{});
    else if (S == 4) rows(std::integral_constant<int, 4>{});
    else rows(std::integral_constant<int, 8>{});
  }
  c.wrote_through = true;  // (what else was written nobody reads before the next iteration)
  barrier_arrive(c);
  // ---- tasks
  const int n_tasks = g.quads * nkv;
  if (c.vid >= n_tasks) barrier_wait(c);
  // The kv heads of the same tokens are neighbours, on one die: rows of one head lie two kilobytes apart, so that a die that reads no other's uses two of the
  // sixteen channels of its cache.  Every other round takes the tasks from the end, as contexts grow.
  struct Task {
    int h, p, t, t0, t_end, p0, n_units, new_all;  // kv head, portion, first row; first and last row of the request there, its first position; units of the portion
    const int *pages;
  };
  auto decode = [&](int u, Task &a) {
    const int round = u / c.G, r0 = round * c.G, rn = min(c.G, n_tasks - r0), turned = round & 1 ? r0 + rn - 1 - (u - r0) : u;
    int k = turned / nkv;
    a.h = turned - k * nkv;
    a.p = 0;
    unsigned long long begins = g.tasks[0];
    a.n_units = __popcll(g.units[0]);
#pragma unroll
    for (int q = 0; q + 1 < MK_GROUP; q++)
      if (a.p == q && k >= __popcll(g.tasks[q])) {
        k -= __popcll(g.tasks[q]);
        a.p = q + 1;
        begins = g.tasks[q + 1];
        a.n_units = __popcll(g.units[q + 1]);
      }
    const bool mine = ((begins >> lane) & 1) && __popcll(begins & ((1ull << lane) - 1)) == k;
    a.t = (int)__ffsll(__ballot(mine)) - 1;
    const int M = __builtin_amdgcn_readfirstlane(sh_rows[a.p]), *rows = tab + a.p * MK_MAX_TOKENS, my_first = rows[ROWS + min(lane, M - 1)];
    a.t0 = __builtin_amdgcn_readlane(my_first, a.t);
    a.p0 = __builtin_amdgcn_readfirstlane(rows[a.t0]);
    a.t_end = a.t0 + __popcll(__ballot(lane < M && my_first == a.t0));
    a.new_all = min(a.t + g.per_task * TG, a.t_end) - a.t0;
    a.pages = rt.kv_indices + __builtin_amdgcn_readfirstlane(rows[2 * ROWS + a.t]);
  };
  // page lists: a task's is requested while the one in front ends
  constexpr int PG = MK_ATTN_PAIR_PAGES / MK_THREADS;
  int pg_next[PG];
  auto request_pages = [&](const Task &a) {
#pragma unroll
    for (int i = 0; i < PG; i++)
      if (tid + i * MK_THREADS <= (a.p0 + a.new_all - 1) / ps) pg_next[i] = a.pages[tid + i * MK_THREADS];
  };
  auto put_pages = [&](const Task &a, int *to) {
#pragma unroll
    for (int i = 0; i < PG; i++)
      if (tid + i * MK_THREADS <= (a.p0 + a.new_all - 1) / ps) to[tid + i * MK_THREADS] = pg_next[i];
  };
  Task next;
  if (c.vid < n_tasks) {
    decode(c.vid, next);
    request_pages(next);
    put_pages(next, (int *)(smem + PAGE_OFF));
    barrier_wait(c);  // every row is where it belongs
  }
  for (int u = c.vid, turn = 0; u < n_tasks; u += c.G, turn ^= 1) {
    const Task a = next;
    const bool goes_on = u + c.G < n_tasks;
    if (goes_on) decode(u + c.G, next);
    const int h = a.h, p = a.p, t = a.t, t0 = a.t0, p0 = a.p0, t_end = a.t_end, new_all = a.new_all;
    CStage &sp = mk_portion_stages(rt, p)[s];
    const int cmax = max(1, min(c.G / (a.n_units * nkv), MK_ATTN_MAX_CHUNKS)), nt = (p0 + 15) / 16, Cd = (nt + MK_WAVES - 1) / MK_WAVES + 1, C = min(Cd, cmax);
    int n_u[NU], new_u[NU];  // tokens of a unit, positions it sees that are new in its portion
#pragma unroll
    for (int e = 0; e < NU; e++) {
      const int first = t + e * TG;
      n_u[e] = e < g.per_task ? max(0, min(TG, t_end - first)) : 0;
      new_u[e] = n_u[e] ? first + n_u[e] - t0 : 0;
    }
    // first tile of chunk `i` of unit `e` (see stage_attn_tiles)
    auto bound = [&](int e, int i) -> int {
      if (i >= C) return nt;
      if (C == Cd) return i < C - 1 ? nt * i / (C - 1) : nt;
      const int extra = 4 * MK_WAVES * ((n_u[e] * QPK + 2 * new_u[e] + 31) / 32 - 1), total = nt + (C > 1 ? min(extra, (nt + C - 2) / (C - 1)) : 0);
      return min(nt, total * i / C);
    };
    const int *spg = (const int *)(smem + PAGE_OFF) + turn * MK_ATTN_PAIR_PAGES;
    __syncthreads();  // (the page list; LDS of the task in front)
    const char *kc = (const char *)st.k_cache, *vc = (const char *)st.v_cache;
    const float scale = st.sm_scale_log2;
    // positions [q0, q0 + 16), none behind `last` (read again instead), as a tile at LDS byte b: values, then keys, each four groups of four rows.  Where pages are
    // powers of two and hold whole tiles, a whole tile of the cache is one address and its lanes' distances (new tiles begin anywhere).
    const int shift = 31 - __builtin_clz(ps);
    const bool plain = ps >= 16 && (ps & (ps - 1)) == 0;
    // (piece c of key row r lies at c ^ 4 (r & 3): the four rows of a group would meet in the same banks)
    unsigned apart[4];
    const unsigned kflip = (lr ^ (lg * 4)) * 16 - lr * 16;
#pragma unroll
    for (int r = 0; r < 4; r++) apart[r] = (unsigned)((4 * r + lg) * nkv) * (2 * D) + lr * 16;
    auto load_rows = [&](int q0, int last, unsigned b) {
      if (plain && (q0 & 15) == 0 && q0 + 15 <= last) {
        const size_t at = (((size_t)__builtin_amdgcn_readfirstlane(spg[q0 >> shift]) * ps + (q0 & (ps - 1))) * nkv + h) * (2 * D);
#pragma unroll
        for (int r = 0; r < 4; r++) lds_request(kc + at, apart[r] + kflip, b + TS + r * GS);
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
        for (int r = 0; r < 4; r++) lds_request(kc + at[r] + (int)kflip, b + TS + r * GS);
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
      auto weigh = [&](auto first_c, auto count_c, const bf16x8 (&kf)[4], int q0, int last, float (&pw)[NU][4], auto meanwhile) {
        constexpr int E0 = decltype(first_c)::value, E1 = E0 + decltype(count_c)::value;
        f32x4 s4[NU];
        float mx[NU], alpha[NU];
#pragma unroll
        for (int e = E0; e < E1; e++) s4[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int e = E0; e < E1; e++) s4[e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[r], qb[e][r], s4[e], 0, 0, 0);
        meanwhile();
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
#pragma unroll
        for (int e = E0; e < E1; e++) {
          const float mn = fmaxf(mrun[e], mx[e]);
          alpha[e] = __builtin_amdgcn_exp2f(mrun[e] - mn);
#pragma unroll
          for (int r = 0; r < 4; r++) pw[e][r] = __builtin_amdgcn_exp2f(pw[e][r] - mn);
          lsum[e] = lsum[e] * alpha[e] + ((pw[e][0] + pw[e][1]) + (pw[e][2] + pw[e][3]));
          mrun[e] = mn;
        }
        // (always: among 32 columns some maximum moves at most tiles of a context of a few thousand positions)
#pragma unroll
        for (int e = E0; e < E1; e++)
#pragma unroll
          for (int dt = 0; dt < 8; dt++)
#pragma unroll
            for (int r = 0; r < 4; r++) o[e][dt][r] *= alpha[e];
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
        for (int r = 0; r < 4; r++) kf[r] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(kl + (r ^ (lr & 3)) * 64));
      };
      // a lane's values, four positions of a dim: four rows of sixteen dims, read as eight bytes a lane, come back transposed
      auto values_of = [&](const char *b, s16x4 (&v)[8]) {
        typedef __attribute__((address_space(3))) s16x4 *Lds;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int dt = 0; dt < 8; dt++) v[dt] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds)(b + lg * GS + (lr >> 2) * 256 + (lr & 3) * 8 + dt * 32));
        __builtin_amdgcn_sched_barrier(0);
      };
      auto each = [&](auto f) {
        f(std::integral_constant<int, 0>{});
        f(std::integral_constant<int, 1>{});
      };
      // ---- cached tiles of this wavefront, RB - 1 requested ahead (the last one again behind the end)
      int t_ = lo + ((wave - lo) & (MK_WAVES - 1));
      const int t_last = hi - 1 - ((hi - 1 - wave) & (MK_WAVES - 1));
      const bool some = t_ < hi;
      auto load_tile = [&](int tt, int b) { load_rows(min(tt, t_last) * 16, p0 - 1, buf + b * SLOT); };
      if (ci > 0) lds_barrier();  // (partial sums of the chunk in front have been read)
      if (some) {
#pragma unroll
        for (int b = 0; b < RB - 1; b++) load_tile(t_ + b * MK_WAVES, b);
      }
      const bool with_new = ci == C - 1;
      if (with_new) {
        if (wave * 16 < new_all) load_rows(p0 + wave * 16, p0 + new_all - 1, lds + PART_OFF + wave * SLOT);
      }
      auto tile = [&](int b) {  // the one in buffer b
        load_tile(t_ + (RB - 1) * MK_WAVES, (b + RB - 1) % RB);
        static_assert(RB == 3, "the wait counts two tiles' requests");
        asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        const char *vb = smem + wave * (RB * SLOT) + b * SLOT;
        bf16x8 kf[4];
        keys(vb, kf);
        s16x4 v[8];
        auto values = [&]() { values_of(vb, v); };  // (requested behind the score products, all at once: the compiler would wait one by one)
        auto units = [&](auto first_c, auto count_c) {
          constexpr int E0 = decltype(first_c)::value, E1 = E0 + decltype(count_c)::value;
          float pw[NU][4];
          weigh(first_c, count_c, kf, t_ * 16, p0 - 1, pw, values);
          s16x4 wt[NU][2];
#pragma unroll
          for (int e = E0; e < E1; e++) terms(pw[e], wt[e]);
#pragma unroll
          for (int e = E0; e < E1; e++) add_products(o[e], v, wt[e]);
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
      };
      while (t_ + (RB - 1) * MK_WAVES < hi) {
#pragma unroll
        for (int b = 0; b < RB; b++) tile(b);
      }
      if (t_ < hi) tile(0);
      if (t_ < hi) tile(1);
      // ---- new tiles: one of them, at most, belongs to a wavefront's partial sum of a unit
      if (with_new) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        each([&](auto unit) {
          constexpr int e = decltype(unit)::value;
          const int sw = (wave - tb[e]) & (MK_WAVES - 1);
          if (sw * 16 >= new_u[e]) return;
          const int q0 = p0 + sw * 16, newest = p0 + new_u[e] - 1, p_first = newest + 1 - n_u[e], n_cols = n_u[e] * QPK;
          const char *vb = smem + PART_OFF + sw * SLOT;
          bf16x8 kf[4];
          keys(vb, kf);
          float pws[NU][4];
          s16x4 bv[8];
          weigh(unit, std::integral_constant<int, 1>{}, kf, q0, p_first + min(lr, n_cols - 1) / QPK, pws, [&]() { values_of(vb, bv); });
          auto &pw = pws[e];
          // (rows behind the unit's newest position count as zeros)
          unsigned top = 0;
          const int there = min(max(newest + 1 - q0 - lg * 4, 0), 4);  // of the lane's four
          const unsigned there0 = there >= 2 ? 0xffffffffu : there ? 0xffffu : 0u, there1 = there >= 4 ? 0xffffffffu : there == 3 ? 0xffffu : 0u;
#pragma unroll
          for (int dt = 0; dt < 8; dt++) {
            u32x2 v = __builtin_bit_cast(u32x2, bv[dt]);
            v[0] &= there0;
            v[1] &= there1;
#pragma unroll
            for (int r = 0; r < 2; r++) top |= ((v[r] & 0x7f80u) + 0x80u) | (((v[r] >> 16) & 0x7f80u) + 0x80u);
            bv[dt] = __builtin_bit_cast(s16x4, v);
          }
          if (__builtin_expect(__ballot(top & 0x8000u) != 0, 0)) {  // values that are not finite: column by column, see stage_attn_tiles
            const bool none = lr >= n_cols;
            for (int g4 = 0; g4 < 4; g4++) {
#pragma unroll
              for (int r4 = 0; r4 < 4; r4++) {
                const uint16_t *v = (const uint16_t *)(vb + g4 * GS + r4 * 256) + lg * 4;
                const float wgt = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((g4 * 16 + lr) << 2, __builtin_bit_cast(int, pw[r4])));
                const bool seen = q0 + g4 * 4 + r4 <= p_first + (none ? n_cols - 1 : lr) / QPK;
#pragma unroll
                for (int dt = 0; dt < 8; dt++)
#pragma unroll
                  for (int r = 0; r < 4; r++) o[e][dt][r] = seen ? fmaf(wgt, bf2f(v[dt * 16 + r]), o[e][dt][r]) : o[e][dt][r];
              }
            }
            return;
          }
          s16x4 wt[3];
          terms(pw, wt);
#pragma unroll
          for (int q = 0; q < 3; q++) add_products(o[e], bv, wt[q]);
        });
      }
      // ---- a unit's four partial sums, in their order, then its chunks.  (What the tiles requested behind the end bring has landed before sums take their place.)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (with_new && goes_on) request_pages(next);
      lds_barrier();
      auto part_of = [&](int e, int w) { return (float *)(smem + (e ? 0 : PART_OFF) + w * SLOT); };
      each([&](auto unit) {
        constexpr int e = decltype(unit)::value;
        if (!n_u[e]) return;
        float lt = lsum[e];
        lt += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 16) << 2, __builtin_bit_cast(int, lt)));
        lt += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, lt)));
        float *part = part_of(e, (wave - tb[e]) & (MK_WAVES - 1));
        if (lg == 0) {
          part[lr * PD + D] = mrun[e];
          part[lr * PD + D + 1] = lt;
        }
#pragma unroll
        for (int dt = 0; dt < 8; dt++) *(f32x4 *)(part + lr * PD + dt * 16 + lg * 4) = o[e][dt];
      });
      lds_barrier();
      each([&](auto unit) {
        constexpr int e = decltype(unit)::value;
        if (!n_u[e]) return;
        float mx = -1e30f, ls = 0.f, os[8];
#pragma unroll
        for (int d = 0; d < 8; d++) os[d] = 0.f;
#pragma unroll
        for (int w = 0; w < MK_WAVES; w++) mx = fmaxf(mx, part_of(e, w)[mcol * PD + D]);
#pragma unroll
        for (int w = 0; w < MK_WAVES; w++) {
          const float *pp = part_of(e, w) + mcol * PD;
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
    if (goes_on) put_pages(next, (int *)(smem + PAGE_OFF) + (turn ^ 1) * MK_ATTN_PAIR_PAGES);
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
