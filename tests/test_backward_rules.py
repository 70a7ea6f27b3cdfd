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
