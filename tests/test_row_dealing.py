"""Rows of a second portion are dealt to the workgroups behind those that took the first one's (mk_rows_ahead and mk_first_row, the same functions as in the kernels)."""
import os
import subprocess


def test_every_row_once_on_any_grid(tmp_path):
    src = tmp_path / "deal.cpp"
    src.write_text(r'''
#include "mk_types.h"
#include <stdio.h>
int main() {
  long bad = 0;
  for (int G = 1; G <= 256; G++)
    for (int M1 = 0; M1 <= MK_MAX_TOKENS; M1++)
      for (int M2 = 1; M2 <= MK_MAX_TOKENS; M2++) {
        int times[MK_MAX_TOKENS] = {}, behind = -1;
        for (int at = 0; at < G; at++) {
          const int t0 = mk_first_row(at, mk_rows_ahead(M1, G), G);
          if (t0 < 0 || t0 >= G) bad++;
          else if (t0 == 0) behind = at;
          for (int t = t0; t < M2; t += G) {
            if (t < 0) { bad++; break; }
            times[t]++;
          }
        }
        for (int t = 0; t < M2; t++) bad += times[t] != 1;
        bad += behind != M1 % G;  // the first one goes to the workgroup behind the first portion's last
      }
  printf("%ld\n", bad);
  return bad != 0;
}
''')
    exe = tmp_path / "deal"
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fleet-chiplet-megakernel_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", csrc, str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip() == "0", res.stdout
