"""What an iteration of several portions runs (mk_pair_program, the function the library uses), walked as the kernel walks it: every stage once for every portion, in its
order, and sums that a linear left to a later stage found where they are."""
import os
import subprocess

WALK = r'''
#include "mk_pairs.h"
#include <stdio.h>
#include <string.h>

const int G = 256;
static bool norm_op(int op) { return op == MK_OP_NORM || op == MK_OP_FX_ADDNORM || op == MK_OP_MX_PRENORM; }
static int slices(MkStage s) { return s.op == MK_OP_LINEAR && !(s.k & 63) ? mk_xres_plan(s, G).S : 0; }
// Steps of the program that go wrong.  single: portions in which every request brings one row; grouped: attention agrees to run for all portions at once.
static int walk(const std::vector<unsigned> &prog, const std::vector<MkStage> &st, int portions, unsigned single, bool grouped) {
  const int n = (int)st.size();
  int bad = 0, steps = 0, defer = 0, sum = 0, prep = 0, group = -1, again = 1;  // group: the linear whose slices lie with those of all portions
  bool together = false;                 // the last linear ran for all portions
  bool own = false;                      // what is left lies in the portion's own place ...
  int own_stage = -1, own_portion = -1;  // ... which holds this linear's
  int at = 0;                            // portion whose slices are looked at
  std::vector<int> next(portions, 0);    // stages that have run, in order
  std::vector<int> kept(portions, -1);   // the portion's own linear that has made its sum itself
  auto ran = [&](int s, int p) {
    bad += next[p] != s;
    next[p] = s + 1;
    for (int j = s + 1; j < n && p; j++) bad += st[s].tail && st[j].tail == st[s].tail && next[p - 1] <= j;  // (reads what the portion in front leaves there)
  };
  auto left_by = [&](int s) {  // the linear whose sum a stage finds, or none
    int l = s - 1;
    if (st[s].op == MK_OP_FX_ATTN && l >= 0 && st[l].op == MK_OP_FX_PREP) l--;
    return l >= 0 && st[l].op == MK_OP_LINEAR && (st[l].flags & MK_F_DEFER_SUM) && slices(st[l]) > 1 ? l : -1;
  };
  auto takes = [&](int s, int p, bool all) {
    const int l = left_by(s);
    if (l < 0 || (!all && kept[p] == l)) bad += defer != 0;
    else if (all) bad += !defer || own || group != l;
    else bad += !defer || (own ? own_stage != l || own_portion != p : group != l || at != p);
    defer = 0;
  };
  for (int e = 0; e < (int)prog.size(); e++) {
    if (++steps > 100000) return bad + 1;
    const unsigned ent = prog[e];
    if (ent & MK_PAIR_ACQUIRE) continue;
    const int s = ent & MK_PAIR_STAGE, p = ent & MK_PAIR_SECOND ? again : 0, op = st[s].op;
    if (s >= n) return bad + 1;
    const bool one = single >> p & 1, all = ent & MK_PAIR_BOTH;
    auto turn = [&]() {
      if (!(ent & MK_PAIR_LOOP)) return;
      if (again + 1 < portions) {
        again++;
        e -= 1 + (int)(ent >> MK_PAIR_BACK_SHIFT);
      } else {
        again = 1;
      }
    };
    if (ent & MK_PAIR_AGAIN) {
      defer = sum;
      own = false;
      at = p;
    }
    if (op == MK_OP_LINEAR) together = all;
    if (op == MK_OP_FX_PREP) prep = together ? defer : 0;
    if (op == MK_OP_FX_ATTN && (ent & MK_PAIR_ON) && one) {
      defer = prep;
      own = false;
      at = p;
    }
    if (op == MK_OP_FX_PREP && one) {
      if (!all) ran(s, p);  // (left out)
      turn();
      continue;
    }
    if (all && op != MK_OP_LINEAR && !norm_op(op)) {
      if (!grouped || single) continue;
      e += (int)(ent >> MK_PAIR_BACK_SHIFT);
    }
    if (all) {
      if (op == MK_OP_LINEAR) {
        bad += defer != 0;
        const int S = slices(st[s]);
        bad += S < 1;
        if (S > 1) group = s;
        if (S > 1 && (st[s].flags & MK_F_DEFER_SUM)) {
          defer = S;
          own = false;
          at = 0;
        }
        sum = defer;
      } else if (op != MK_OP_FX_ATTN) {
        takes(s, 0, true);
      }
      for (int q = 0; q < portions; q++) ran(s, q);
    } else {
      if (op == MK_OP_LINEAR) {
        bad += defer != 0;
        const int S = slices(st[s]);
        if (S > 1) own_stage = s, own_portion = p;
        if (S > 1 && (st[s].flags & MK_F_DEFER_SUM) && !mk_keeps_sum(one, s + 1 < n ? st[s + 1].op : 0)) defer = S, own = true;
        else kept[p] = s;
      } else if (norm_op(op) || op == MK_OP_ATTN || op == MK_OP_FX_PREP || (op == MK_OP_FX_ATTN && one)) {
        takes(s, p, false);
      }
      ran(s, p);
    }
    turn();
  }
  for (int q = 0; q < portions; q++) bad += next[q] != n;
  return bad;
}
static char caches[64];
static MkStage stage(int op, int n = 0, int k = 0, unsigned flags = 0) {
  MkStage s;
  memset(&s, 0, sizeof(s));
  s.op = op;
  s.n = n;
  s.k = k;
  s.flags = flags;
  if (op == MK_OP_FX_PREP || op == MK_OP_FX_ATTN || op == MK_OP_ATTN) s.k_cache = caches, s.v_cache = caches + 1, s.num_q_heads = 32, s.num_kv_heads = 8;
  return s;
}
static int walks(const std::vector<MkStage> &st, long *programs) {
  const std::vector<unsigned> prog = mk_pair_program(st.data(), (int)st.size(), G);
  if (prog.empty()) return 0;
  ++*programs;
  int bad = 0;
  for (int portions : {2, 3, 8})
    for (unsigned single : {0u, 1u, 2u, 4u, 6u, 0x55u, 0xaau, 0xffu})
      for (int grouped = 0; grouped < 2; grouped++) bad += walk(prog, st, portions, single & ((1u << portions) - 1), grouped) != 0;
  return bad;
}
'''


def _run(tmp_path, main):
    src, exe = tmp_path / "program.cpp", tmp_path / "program"
    src.write_text(WALK + main)
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fleet-chiplet-megakernel_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", csrc, str(src), "-o", str(exe)], check=True)
    return list(map(int, subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()))


def test_programs_of_any_stages(tmp_path):
    """Sequences of norms, linears (whole, in slices, none that stream; their sums left to the stage behind or not), attention with its preparation, convolutions and scans, and others."""
    bad, programs = _run(tmp_path, r'''
int main() {
  long bad = 0, programs = 0;
  unsigned seed = 1;
  auto draw = [&](int n) { return (int)((seed = seed * 1664525u + 1013904223u) >> 8) % n; };
  const int ns[] = {1024, 2048, 4096, 6144, 24576}, ks[] = {512, 2048, 2560, 4096, 12288, 1000};
  for (int it = 0; it < 4000; it++) {
    std::vector<MkStage> st;
    const bool fx = draw(2);
    for (int len = 3 + draw(14); (int)st.size() < len;) {
      switch (draw(7)) {
        case 0: st.push_back(stage(fx ? MK_OP_FX_ADDNORM : MK_OP_NORM, 2048, draw(4) ? 2048 : 2044)); break;
        case 1: if (fx) st.push_back(stage(MK_OP_MX_PRENORM, 2048)); break;
        case 2:
          if (fx) st.push_back(stage(MK_OP_FX_PREP));
          st.push_back(stage(fx ? MK_OP_FX_ATTN : MK_OP_ATTN));
          break;
        case 3: st.push_back(stage(draw(2) ? MK_OP_SILU_MUL : MK_OP_HY_STEP)); break;
        case 4:  // (a convolution reads the request's last inputs, which the scan behind it writes)
          st.push_back(stage(MK_OP_HY_CONV));
          st.back().tail = caches + st.size();
          if (draw(3)) st.push_back(stage(MK_OP_LINEAR, ns[draw(5)], ks[draw(6)]));
          if (draw(2)) st.push_back(stage(MK_OP_HY_STEP));
          st.push_back(stage(MK_OP_HY_SCAN));
          for (size_t i = st.size() - 1; st[i].op != MK_OP_HY_CONV; i--) st.back().tail = st[i - 1].tail;
          break;
        default: st.push_back(stage(MK_OP_LINEAR, ns[draw(5)], ks[draw(6)]));
      }
    }
    for (size_t i = 0; i + 1 < st.size(); i++)
      if (st[i].op == MK_OP_LINEAR && (norm_op(st[i + 1].op) || st[i + 1].op == MK_OP_ATTN || st[i + 1].op == MK_OP_FX_PREP) && draw(4)) st[i].flags |= MK_F_DEFER_SUM;
    bad += walks(st, &programs);
  }
  printf("%ld %ld\n", bad, programs);
}
''')
    assert bad == 0 and programs > 2000


def test_single_rows_behind_a_linear_of_its_own(tmp_path):
    """The projection of a layer whose output one does not stream runs portion by portion, and leaves its sum to the attention where a portion's requests bring one row each: 16
    query and 8 key heads of 160 at a width of 2048."""
    bad, programs, slices_left = _run(tmp_path, r'''
int main() {
  std::vector<MkStage> st = {stage(MK_OP_FX_ADDNORM, 2048), stage(MK_OP_LINEAR, 5120, 2048, MK_F_DEFER_SUM), stage(MK_OP_FX_PREP), stage(MK_OP_FX_ATTN), stage(MK_OP_LINEAR, 2048, 2560), stage(MK_OP_FX_ADDNORM, 2048),
                             stage(MK_OP_LINEAR, 12288, 2048), stage(MK_OP_LINEAR, 2048, 6144, MK_F_DEFER_SUM), stage(MK_OP_FX_ADDNORM, 2048)};
  long programs = 0;
  const int bad = walks(st, &programs);
  printf("%d %ld %d\n", bad, programs, slices(st[1]));
}
''')
    assert bad == 0 and programs == 1 and slices_left > 1


def test_tokens_of_a_portion_replaced_behind_a_barrier(tmp_path):
    """A left-out stage looks at its portion's tokens and has no barrier: another portion's take their place behind one, and are read behind one."""
    src, exe = tmp_path / "hold.cpp", tmp_path / "hold"
    src.write_text(r'''
#include "mk_types.h"
#include <stdio.h>
#include <vector>
int main() {
  int held = 1;
  for (int portion : {0, 1, 2, 2, 0, 2, 3, 1}) {
    printf("%d", portion);
    mk_hold_portion(portion, held, []() { printf("L"); }, []() { printf("|"); });
    printf(" ");
  }
}
''')
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fleet-chiplet-megakernel_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-I", csrc, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split() == ["0", "1", "2|L|", "2", "0", "2", "3|L|", "1|L|"]


def test_every_portion_has_a_wavefront(tmp_path):
    most = _run(tmp_path, 'int main() { for (int G : {1, 2, 3, 256}) printf("%d ", mk_most_portions(G)); }')
    assert most == [4, 8, 8, 8]


def test_as_many_portions_as_fit_the_memory(tmp_path):
    """Rows and scratch are asked for in one piece, for as many portions as a grid can have, then half of them and so on, until a piece is there."""
    tried = _run(tmp_path, r'''
int main() {
  for (int G : {256, 1})
    for (int room : {8, 7, 4, 3, 2, 1, 0}) printf("%d 0 ", mk_portions_that_fit(G, [&](int p) { printf("%d ", p); return p <= room; }));
}
''')
    wide = [[8, 8], [8, 4, 4], [8, 4, 4], [8, 4, 2, 2], [8, 4, 2, 2], [8, 4, 2, 1], [8, 4, 2, 1]]
    narrow = [[4, 4]] * 3 + [[4, 2, 2], [4, 2, 2], [4, 2, 1], [4, 2, 1]]
    assert tried == [x for t in wide + narrow for x in t + [0]]


def test_runs_longer_than_an_entry_can_say(tmp_path):
    """Stages between two linears for one portion after the other: as many as an entry's nine bits can go back over, or portions one by one."""
    bad, short, long_ = _run(tmp_path, r'''
int main() {
  long bad = 0, programs[2] = {0, 0};
  for (int len = 490; len < 700; len++)
    for (int op : {(int)MK_OP_SILU_MUL, (int)MK_OP_HY_SCAN}) {
      std::vector<MkStage> st(len, stage(op));
      st.push_back(stage(MK_OP_LINEAR, 24576, 4096));
      bad += walks(st, &programs[len > 512]);
    }
  printf("%ld %ld %ld\n", bad, programs[0], programs[1]);
}
''')
    assert bad == 0 and short >= 44 and long_ == 0
