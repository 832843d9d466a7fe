"""A launch is several calls on its stream: what is undone where one of them fails behind others (mk_enqueue_parts, the code the library runs)."""
import os
import subprocess


def test_calls_that_fail(tmp_path):
    src = tmp_path / "parts.cpp"
    src.write_text(r'''
#include "mk_launch.h"
#include <stdio.h>
int main() {
  for (int kind = 0; kind < 3; kind++)  // the main kernel alone, one in front of it, one in its place
    for (int fails = 0; fails < 5; fails++) {
      int calls = 0, undone = 0, lost = 0;
      printf("%d%d:", kind, fails);
      const int rc = mk_enqueue_parts(kind == 1, kind == 2, [&](MkLaunchPart p) { printf("%d", p); return calls++ == fails ? 7 : 0; }, [&](bool l) { undone++; lost = l; });
      printf(" rc %d undone %d lost %d\n", rc, undone, lost);
    }
}
''')
    exe = tmp_path / "parts"
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fleet-chiplet-megakernel_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-I", csrc, str(src), "-o", str(exe)], check=True)
    PAIRS, RESUME, MAIN, DONE = range(4)
    want = []
    for kind, parts in enumerate(([MAIN, DONE], [PAIRS, RESUME, MAIN, DONE], [PAIRS, DONE])):
        for fails in range(5):
            failed = parts[fails] if fails < len(parts) else None
            undone = failed is not None and fails > 0  # (nothing is on the stream yet when the first call fails)
            lost = undone and kind == 1 and failed != DONE
            want.append(f"{kind}{fails}:{''.join(map(str, parts[:fails + 1]))} rc {7 if failed is not None else 0} undone {undone:d} lost {lost:d}")
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines() == want
