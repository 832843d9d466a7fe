// What an iteration of several portions of prompts runs (MkPairEntry).  No HIP: tests/test_pair_program.py runs the same code on the CPU.
#pragma once
#include <algorithm>
#include <vector>

#include "mk_types.h"

// Portions that run together on G workgroups at most: a wavefront prepares rows of one portion for the attention of all, so every portion needs one.
inline int mk_most_portions(int G) {
  int portions = MK_GROUP;
  while (portions > G * MK_WAVES) portions /= 2;
  return portions;
}
// As many of them as allocate(portions) finds memory for: all, a half, a quarter; 1: not even for two.
template <class Allocate>
inline int mk_portions_that_fit(int G, Allocate allocate) {
  int portions = mk_most_portions(G);
  while (portions > 1 && !allocate(portions)) portions /= 2;
  return portions;
}

// Several portions inside prompts as one iteration (MkPairEntry): linears that run for all portions at once, and between two of them the stages of
// the first portion, then those of the second, and so on, as iterations of their own would run them.  What a cache or a state gets from a portion is
// written back and read anew in front of the next one; stages that only take rows to rows run for one portion after the other without a barrier, and so do
// stages that put keys and values into pages and, behind them all, the attention over those pages, which looks at no position behind a row's own.  Norms by
// rows run for all portions at once, and so does attention with what prepares its rows, unless the portions ask for another form: then the entries
// behind, portion by portion, are the ones that run.
// stages [0, n) on G workgroups.  Empty: no linear runs that way, or a run is longer than an entry can say.
inline std::vector<unsigned> mk_pair_program(const MkStage *stages, int n, int G) {
  std::vector<unsigned> prog;
  auto keeps_nothing = [&](const MkStage &s) { return !s.k_cache && !s.v_cache && !s.tail && !s.conv_w; };
  auto row_wise = [&](const MkStage &s) {
    return keeps_nothing(s) && (s.op == MK_OP_NORM || s.op == MK_OP_FX_ADDNORM || s.op == MK_OP_MX_PRENORM || s.op == MK_OP_EMBED || s.op == MK_OP_FX_EMBED);
  };
  auto passes = [&](const MkStage &s) {  // (leaves nothing for another iteration)
    switch (s.op) {
      case MK_OP_NORM: case MK_OP_FX_ADDNORM: case MK_OP_MX_PRENORM: case MK_OP_EMBED: case MK_OP_FX_EMBED: case MK_OP_LINEAR: case MK_OP_SILU_MUL: case MK_OP_MOE_TOPK: case MK_OP_MOE_LINEAR:
      case MK_OP_MOE_COMBINE: case MK_OP_MX_HEAD_LINEAR: case MK_OP_HY_ROUTE: case MK_OP_HY_EXPERTS: case MK_OP_COPY: return keeps_nothing(s);
      default: return false;
    }
  };
  auto left_out = [&](const MkStage &s) {  // (by iterations in which nobody has several rows, or nothing was split)
    return s.op == MK_OP_FX_PREP || s.op == MK_OP_DU_CONV || s.op == MK_OP_MX_LATENT_MERGE || s.op == MK_OP_MX_DELTA_OUT;
  };
  std::vector<char> both(n, 0);
  for (int i = 0; i < n; i++) {
    MkStage s = stages[i];
    both[i] = s.op == MK_OP_LINEAR && keeps_nothing(s) && (s.k & 63) == 0 && mk_xres_plan(s, G).S >= 1;
  }
  // a convolution reads the request's last inputs, which the scan behind it writes: for a portion that must be those of the one in front, so nothing between the two
  // runs for all portions
  for (int i = 0; i < n; i++)
    for (int j = n - 1; j > i && stages[i].tail; j--)
      if (stages[j].tail == stages[i].tail) std::fill(both.begin() + i, both.begin() + j, 0);
  // what says where a sum is that was left to the stage behind says so of the last linear that left one, and is kept until all portions have read it: by a
  // stage that runs for all of them at once, or with no other linear in between
  for (int i = n - 1; i >= 0; i--) {
    if (!both[i] || !(stages[i].flags & MK_F_DEFER_SUM) || (i + 1 < n && row_wise(stages[i + 1]))) continue;
    for (int j = i + 1; j < n && !both[j]; j++)
      if (stages[j].op == MK_OP_LINEAR) both[i] = 0;
  }
  if (std::count(both.begin(), both.end(), 1) == 0) return prog;
  bool fits = true;
  auto back = [&](size_t entries) -> unsigned {  // (all that is above the other bits)
    fits = fits && entries < 1u << (32 - MK_PAIR_BACK_SHIFT);
    return (unsigned)entries << MK_PAIR_BACK_SHIFT;
  };
  for (int i = 0; i < n;) {
    if (both[i]) {
      prog.push_back(i++ | MK_PAIR_BOTH);
      continue;
    }
    int j = i;
    while (j < n && !both[j]) j++;
    // a run [q0, q1) for one portion after the other; the first stage of all may find a sum that the linear in front has left
    auto in_turn = [&](int q0, int q1, bool on) {
      bool carries = false;
      for (int q = q0; q < q1; q++) carries = carries || !(on || passes(stages[q]));
      // One write-back of the caches is enough, behind the last of these stages that no iteration leaves out, or behind later ones that may write.
      // (Each is 2 to 4 us.  Behind every stage, pairs were slower than their portions one by one where few linears run for both, us a pair: dodonex-2k
      // + 53, vizonex-8b + 50, vizonex-2k + 63, bukatar-2k + 37; now - 7, - 15, - 14, - 21, and suborax-8b - 174 -> - 184, dodonex-8b - 37 -> - 93.)
      int last = q1 - 1;
      while (last >= q0 && left_out(stages[last])) last--;
      auto entry = [&](int q) { return q | (on ? MK_PAIR_ON : 0) | (carries && (q == last || (q > last && !passes(stages[q]))) ? MK_PAIR_RELEASE : 0); };
      for (int q = q0; q < q1; q++) prog.push_back(entry(q));
      const size_t again = prog.size();
      if (carries) prog.push_back(MK_PAIR_ACQUIRE);
      for (int q = q0; q < q1; q++) prog.push_back(entry(q) | MK_PAIR_SECOND | (q == i && i > 0 ? MK_PAIR_AGAIN : 0));
      prog.back() |= MK_PAIR_LOOP | back(prog.size() - 1 - again);
    };
    // (not a stage that may find a sum which a stage of the same run has left)
    auto first = [&](int q) { return q == i || !(stages[q - 1].flags & MK_F_DEFER_SUM); };
    // attention over pages, all of whose new rows the stage in front has put there (or, of single rows, puts there itself: see mk_keeps_sum)
    auto prepared = [&](int q) {
      const MkStage &s = stages[q];
      return s.op == MK_OP_FX_ATTN && q > i && stages[q - 1].op == MK_OP_FX_PREP && stages[q - 1].k_cache == s.k_cache && stages[q - 1].v_cache == s.v_cache;
    };
    auto normed = [&](const MkStage &s) { return row_wise(s) && ((s.op == MK_OP_NORM && mk_norm_by_rows(s)) || s.op == MK_OP_FX_ADDNORM); };
    auto attends = [&](int q) {  // attention that may run for all portions at once, and what prepares its rows
      const MkStage &s = stages[q];
      if (prepared(q) || (q + 1 < j && prepared(q + 1))) return first(q);
      return s.op == MK_OP_ATTN && first(q) && (s.num_q_heads == 4 * s.num_kv_heads || s.num_q_heads == 8 * s.num_kv_heads);
    };
    auto alone = [&](int q) { return first(q) && (row_wise(stages[q]) || prepared(q) || (q + 1 < j && prepared(q + 1))); };
    for (int q = i; q < j;) {
      int e = q + 1;
      if (first(q) && normed(stages[q])) {
        prog.push_back(q | MK_PAIR_BOTH);
      } else if (attends(q)) {
        const size_t at = prog.size();
        prog.push_back(q | MK_PAIR_BOTH);
        in_turn(q, e, alone(q));
        prog[at] |= back(prog.size() - at - 1);
      } else {
        if (!alone(q))
          while (e < j && !alone(e) && !attends(e) && !(first(e) && normed(stages[e]))) e++;
        in_turn(q, e, alone(q));
      }
      q = e;
    }
    i = j;
  }
  if (!fits) prog.clear();
  return prog;
}
