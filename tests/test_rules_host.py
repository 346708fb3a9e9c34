"""The rules that choose a kernel or a launch shape (bfe_rules.hpp), compiled
for the host and walked over their ranges: the lines lie where the measured
forms cross, and no launch leaves CUs idle that another shape would use."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "exptool_amd", "csrc")

PROGRAM = r"""
#include "bfe_rules.hpp"
#include <cstdio>
#include <cstring>
int main() {
  char f[64];
  long long a[6];
  while (std::scanf("%63s %lld %lld %lld %lld %lld %lld", f, a, a + 1, a + 2, a + 3, a + 4, a + 5) == 7) {
    if (!std::strcmp(f, "eval_four_waves")) std::printf("%d\n", (int)bfe::eval_four_waves(a[0]));
    else return 1;
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(PROGRAM)
    exe = str(d / "rules")
    subprocess.run([cxx, "-O1", "-std=c++17", "-Wall", "-I", CSRC, str(d / "rules.cpp"), "-o", exe], check=True)

    def ask(name, calls):
        """The rule's answers (lists of integers) to a list of argument tuples."""
        text = "\n".join(" ".join([name] + [str(v) for v in c] + ["0"] * (6 - len(c))) for c in calls)
        r = subprocess.run([exe], input=text + "\n", capture_output=True, text=True, check=True)
        out = [[int(v) for v in line.split()] for line in r.stdout.splitlines()]
        assert len(out) == len(calls)
        return out
    return ask


def test_four_waves_only_where_the_chip_is_full(rule):
    """Up to three blocks of 256 points a CU (256 CUs) are resident with three
    waves a SIMD, so the four-wave build has nothing to give there."""
    ns = [1, 256, 65_536, 131_072, 196_608, 262_144, 500_000, 1_000_000, 2_000_000]
    got = [bool(v[0]) for v in rule("eval_four_waves", [(n,) for n in ns])]
    assert got == [False] * 7 + [True] * 2
