"""Whether a launch of the offline scheduler begins with a given number of pairs of portions (mk_pairs_ahead), against the batches that the scheduler oracle forms."""
import os
import random
import subprocess

import pytest

SOURCE = r'''
#include "mk_types.h"
#include <stdio.h>
int main() {
  int running, n, B, most, max_seq, need;
  while (scanf("%d %d %d %d %d %d", &running, &n, &B, &most, &max_seq, &need) == 6) {
    int st[64], plen[64];
    for (int i = 0; i < n; i++)
      if (scanf("%d %d", st + i, plen + i) != 2) return 1;
    printf("%d", mk_pairs_ahead(st, plen, running, n, B, most, max_seq, need));
  }
}
'''


def _iterations(plens, R, B, most, max_seq):
    """Of every iteration: (request, first position, rows) per slot."""
    from oracle.sched_ref import SchedulerOracle
    orc = SchedulerOracle([[1] * n for n in plens], R, B, R * -(-max_seq // 4), 4, max_seq, max_new_per_req=most)
    out = []
    while orc.step([1] * B):
        q = orc["qo_indptr"]
        out.append([(int(r), int(orc["step"][r]), int(q[i + 1] - q[i])) for i, r in enumerate(orc["request_ids"]) if r >= 0])
    return out


@pytest.mark.parametrize("seed", range(6))
def test_as_the_scheduler(tmp_path, seed):
    rng = random.Random(seed)
    asked, want = [], []
    for _ in range(60):
        B, R, total = rng.choice([33, 40, 64]), rng.choice([1, 2, 3, rng.randint(1, 12)]), rng.randint(1, 8)
        most, max_seq = rng.choice([9, 20, B, 64]), rng.randint(100, 620)
        plens = [rng.randint(1, min(max_seq - 3, rng.choice([20, 90, 600]))) for _ in range(total)]
        its = _iterations(plens, R, B, most, max_seq)
        inside = lambda it: all(at + n < plens[r] and at + n + 1 < max_seq for r, at, n in it if n > 0)
        for i in range(len(its)):
            if i and not inside(its[i - 1]):
                continue
            live = [(at + n, plens[r]) for r, at, n in its[i - 1]] if i else []
            first = max((r for it in its[:i] for r, _, _ in it), default=-1) + 1
            live_n, waiting = len(live), [(0, p) for p in plens[first:]][:max(0, R - len(live))]
            def pair(two):
                return (len(two) == 2 and all(map(inside, two)) and [r for r, _, _ in two[0]] == [r for r, _, _ in two[1]]
                        and 2 * sum(n for _, _, n in two[0]) > B and sum(n for _, _, n in two[1]) == B)
            need = rng.choice([1, 1, 2, 3])
            asked.append(" ".join(map(str, (live_n, live_n + len(waiting), B, most, max_seq, need, *(x for e in live + waiting for x in e)))))
            want.append(all(pair(its[i + 2 * k:i + 2 * k + 2]) for k in range(need)))
    src = tmp_path / "ahead.cpp"
    src.write_text(SOURCE)
    exe = tmp_path / "ahead"
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fleet-chiplet-megakernel_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", csrc, str(src), "-o", str(exe)], check=True)
    got = subprocess.run([str(exe)], input="\n".join(asked), capture_output=True, text=True, check=True).stdout
    assert got == "".join(str(int(w)) for w in want) and "1" in got and "0" in got
