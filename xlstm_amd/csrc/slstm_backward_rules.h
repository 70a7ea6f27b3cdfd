// Decisions of the reverse kernels that spread a head over several compute units, in plain C++ without a GPU's anything: the tests
// compile this file for the host and walk through it.
#pragma once

#ifdef __HIPCC__
#define XS_RULE __host__ __device__ constexpr
#else
#define XS_RULE constexpr
#endif

namespace {

// Whether a call has to be flagged as failed because of where a group's workgroups ran.  `seen`: the XCDs they found themselves on, one
// bit each.  Their exchange goes through ONE XCD's L2; a group of one workgroup, and a call with the recurrent gradient cut, in
// which nothing reaches the step before, exchange nothing and may run anywhere.
XS_RULE bool bwd_exchange_torn(int members, bool cut, unsigned int seen) { return members > 1 && !cut && (seen & (seen - 1u)) != 0u; }

// How the prefetching workgroups keep in front of the groups whose inputs they bring.  They look at the groups' progress every `every`
// steps, and a look lets them go on once no group is more than `ahead` steps behind: up to `ahead + every - 1` steps of inputs lie in
// front of a group.
struct BwdPace {
  int ahead, every;
};

// `rows`: rows of a row tile; `step_bytes`: what the groups of an XCD read in a step; `depth`: steps the feeder waves ask ahead.
// The steps in front of a group are 2 MiB of an XCD's 4 MiB L2 at most (or, beyond 233 KB a step, the nine steps that leave a look every
// second step in front of the feeder waves' six: 2.7 MiB at eight groups of head dim 256).  A look comes back
// behind the touches issued in front of it, a trip to memory: with row tiles of 4 rows it is made every eighth step (a training call at B 16 x
// T 1024 x 4 heads of 256, ms: every fourth step, 16 ahead, 1.75, every second 1.73, every one 1.89, every eighth 1.70), more often where
// 2 MiB are few steps.  us of the reverse kernel at 4 heads of 256, T 512, B 16 / 24 / 32 / 48: looks at multiples of eight steps, 2 MiB
// without the steps between two looks and a late prefetch sent back to such a multiple 434 / 509 / 670 / 705; this 419 / 474 / 644 /
// 665; with 2.5 MiB 424 / 479 / 652 / 673, with 1.2 MiB 422 / 474 / 627 / 669.
XS_RULE BwdPace bwd_pace(int rows, long long step_bytes, int depth) {
  const int furthest = rows == 4 ? 31 : 13, seldom = rows == 4 ? 8 : 2;
  const int least = depth + 2;  // steps ahead of the groups' progress that a look has to allow
  const long long room = (2 << 20) / (step_bytes > 0 ? step_bytes : 1);
  const int lead = room > furthest ? furthest : (room < least + 1 ? least + 1 : (int)room);
  const int every = lead - least + 1 < seldom ? lead - least + 1 : seldom;
  return BwdPace{lead - every + 1, every};
}

// The step to go on with behind a look at step m that found the slowest group at step `at`: what the feeder waves have asked for
// by then (up to step at + depth) is past help.
XS_RULE int bwd_pace_resume(int m, int at, int depth) { return m < at + depth + 1 ? at + depth + 1 : m; }

// Which of the two words the k-th look leaves its result in for the other waves: while one of them may still have to read a word, the wave
// that looks writes the other (between two looks it passes no barrier that they have not).
XS_RULE int bwd_look_word(int k) { return k & 1; }

}  // namespace
