"""Tasks of a linear over several portions (mk_group_plan, the function the kernels use): every weight tile, slice and portion once, slices as for one portion alone."""
import os
import subprocess


def test_tasks_cover_the_stage(tmp_path):
    src = tmp_path / "plan.cpp"
    src.write_text(r'''
#include "mk_types.h"
#include <stdio.h>
#include <string.h>
#include <vector>
int main() {
  long bad = 0, plans = 0;
  for (int G : {8, 32, 48, 256})
    for (int n : {16, 100, 1024, 2048, 4096, 6144, 6176, 24576, 32768})
      for (int k : {512, 1024, 2048, 4096, 12288, 4160})
        for (int silu = 0; silu < 2; silu++)
          for (int portions = 1; portions <= MK_GROUP; portions++) {
            MkStage st;
            memset(&st, 0, sizeof(st));
            st.n = n;
            st.k = k;
            st.flags = silu ? MK_F_SILU : 0;
            const XresPlan x = mk_xres_plan(st, G);
            const GroupPlan p = mk_group_plan(st, G, portions);
            if (x.S < 1) {
              bad += p.S >= 1;
              continue;
            }
            plans++;
            bad += p.S != x.S || p.wt != x.wt || p.tw < 2 || p.tw > 4 || k / p.S % 512 != 0;
            std::vector<int> times((size_t)p.wt * p.S * portions, 0);
            int next = 0;
            for (int v = 0; v < G; v++) {
              const int t0 = (int)((long long)v * p.tasks / G), t1 = (int)((long long)(v + 1) * p.tasks / G);
              bad += t0 != next;
              next = t1;
              for (int t = t0; t < t1; t++) {
                const int mb = t % p.mb, sl = t / p.mb % p.S, nb = t / p.mb / p.S;
                for (int w = nb * 4 * p.tw; w < (nb + 1) * 4 * p.tw && w < p.wt; w++)
                  for (int q = 2 * mb; q < 2 * mb + 2 && q < portions; q++) times[((size_t)w * p.S + sl) * portions + q]++;
              }
            }
            bad += next != p.tasks;
            for (int t : times) bad += t != 1;
          }
  printf("%ld %ld\n", bad, plans);
  return 0;
}
''')
    exe = tmp_path / "plan"
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fleet-chiplet-megakernel_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", csrc, str(src), "-o", str(exe)], check=True)
    bad, plans = map(int, subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split())
    assert bad == 0 and plans > 500
