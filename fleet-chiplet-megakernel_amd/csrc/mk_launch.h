// The calls that put one launch on its stream, in order, and what becomes of a launch of which a later call fails.  No HIP: tests/test_launch_parts.py
// runs the same code on the CPU.
#pragma once

enum MkLaunchPart { MK_PART_PAIRS, MK_PART_RESUME, MK_PART_MAIN, MK_PART_DONE };

// `first`: the kernel of several portions runs in front of the main one; `both`: in its place.  enqueue(part) returns 0 or an error.  What has been
// enqueued when a call fails runs all the same, so undo(lost) has to wait for it and clear the counters that the missing last part would have
// cleared: the next launch's workgroups would count on from them.  `lost`: the kernel in front has scheduled an iteration that nobody runs.
template <class Enqueue, class Undo>
int mk_enqueue_parts(bool first, bool both, Enqueue enqueue, Undo undo) {
  const bool wanted[] = {first || both, first, !both, true};  // (by part)
  bool begun = false;
  for (int part = MK_PART_PAIRS; part <= MK_PART_DONE; part++) {
    if (!wanted[part]) continue;
    if (const int error = enqueue((MkLaunchPart)part)) {
      if (begun) undo(first && part != MK_PART_DONE);
      return error;
    }
    begun = true;
  }
  return 0;
}
