"""The decisions of the reverse kernels in csrc/slstm_backward_rules.h, compiled for the host (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

CSRC = os.path.join(ROOT, "xlstm_amd", "csrc")
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs a C++ compiler")


def _run(tmp_path, body):
    source, binary = tmp_path / "rules.cpp", tmp_path / "rules"
    source.write_text('#include <cstdio>\n#include <initializer_list>\n#include "slstm_backward_rules.h"\n' + body)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, "-o", str(binary), str(source)], check=True)
    res = subprocess.run([str(binary)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
    return res.stdout


def test_a_call_is_flagged_for_its_placement_only_where_workgroups_exchange(tmp_path):
    """Several XCDs under one group matter where its workgroups exchange deltas: not in a group of one workgroup, and not
    with the recurrent gradient cut.  Every kernel that looks at its placement asks the one rule, with the call's cut."""
    _run(tmp_path, r"""
int main() {
  for (int members : {1, 2, 4, 8})
    for (unsigned seen = 1; seen < 256; ++seen)
      for (int cut = 0; cut < 2; ++cut) {
        const bool several = __builtin_popcount(seen) > 1;
        if (bwd_exchange_torn(members, cut != 0, seen) != (several && members > 1 && !cut)) { printf("%d %u %d\n", members, seen, cut); return 1; }
      }
  return 0;
}
""")
    asked = 0
    for name in sorted(os.listdir(CSRC)):
        if name.startswith("slstm_backward") and name != "slstm_backward_rules.h":
            text = open(os.path.join(CSRC, name)).read()
            assert "seen - 1" not in text, name  # (nobody decides this for itself)
            asked += len(re.findall(r"bwd_exchange_torn\([^;]*p\.cut != 0", text))
    assert asked == 2  # bwd_placement_mixed (split and quad kernels) and the unit kernel


_WALK = r"""
#include <cstdlib>
// the prefetching workgroups' walk of slstm_backward_kernels.h over groups whose slowest moves on by chance; what is touched must be
// neither too far in front of the groups nor, right behind a look, what their feeder waves have asked for already
static int walk(int rows, long long step_bytes, int depth, int T, int slow) {
  const BwdPace pace = bwd_pace(rows, step_bytes, depth);
  if (pace.every < 2 || pace.ahead < depth + 2) return 1;
  const long long most = 2 << 20 > (depth + 3) * step_bytes ? 2 << 20 : (depth + 3) * step_bytes;
  int at = 0, next_look = pace.ahead;
  for (int m = 0; m < T; ++m) {
    at += rand() % 100 < slow ? 0 : rand() % 3;
    if (m >= next_look) {
      while (at < m - pace.ahead) at += rand() % 2;
      if (rand() % 50 == 0) at += rand() % 40;  // (the prefetch is late)
      m = bwd_pace_resume(m, at, depth);
      if (m >= T) break;
      if (m <= at + depth) return 2;
      if (m > at + depth + 1 && m > at + pace.ahead) return 3;
      next_look = m + pace.every;
    }
    if ((m - at) * step_bytes > most) return 4;
  }
  return 0;
}
int main() {
  for (int rows : {4, 16})
    for (int groups = 1; groups <= 64; ++groups)
      for (int S : {1, 2, 4, 8})
        for (int slow : {0, 30, 60, 95}) {
          const int depth = rows == 4 ? 6 : 2;
          const long long bytes = (long long)groups * S * rows * (9 * 64 * 4 + 64 * 2);
          if (int why = walk(rows, bytes, depth, 4000, slow)) { printf("%d rows, %d groups of %d: %d\n", rows, groups, S, why); return 1; }
        }
  return 0;
}
"""


def test_the_prefetch_stays_in_its_share_of_the_cache_and_ahead_of_the_feeder_waves(tmp_path):
    """However the groups move: what the prefetching workgroups have brought and no group has reached is at most 2 MiB of an
    XCD's 4 MiB L2 (or three steps more than the feeder waves run ahead), also between two looks, and a prefetch that is late goes
    on at the first step that nobody has asked for."""
    _run(tmp_path, _WALK)
    kernel = open(os.path.join(CSRC, "slstm_backward_kernels.h")).read()
    assert "= bwd_pace(ROWS, " in kernel and "m = bwd_pace_resume(m, at, DEPTH);" in kernel and "next_look = m + pace.every;" in kernel


def test_a_look_leaves_its_result_where_no_wave_still_reads_the_one_before(tmp_path):
    """Look k: a first barrier, the result, a second barrier, everybody reads.  A wave may read as late as its first barrier of
    look k + 1, and the looking wave writes look k + 1's word in front of that barrier: not the same word.  Its write for look
    k + 2 is behind it."""
    _run(tmp_path, r"""
int main() {
  for (int k = 0; k < 1000; ++k)
    if (bwd_look_word(k) == bwd_look_word(k + 1) || bwd_look_word(k) < 0 || bwd_look_word(k) > 1) return 1;
  return 0;
}
""")
    kernel = open(os.path.join(CSRC, "slstm_backward_kernels.h")).read()
    assert "int *const found = &slowest[bwd_look_word(looks++)];" in kernel and "int slowest[2];" in kernel
    assert len(re.findall(r"\bslowest\b(?!\[)", kernel)) == 0  # (nothing goes past the rule)
