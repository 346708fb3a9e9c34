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
    if (!std::strcmp(f, "eval_four_waves")) std::printf("%d\n", (int)bfe::eval_four_waves(a[0], a[1] != 0));
    else if (!std::strcmp(f, "split_orbits_max"))
      std::printf("%lld\n", (long long)bfe::split_orbits_max(a[0], a[1], a[2], a[3] != 0));
    else if (!std::strcmp(f, "eval_form"))
      std::printf("%d\n", (int)bfe::eval_form(a[0], a[1], a[2], a[3] != 0, a[4], a[5]));
    else if (!std::strcmp(f, "eval_split_two"))
      std::printf("%d\n", (int)bfe::eval_split_two(a[0], a[1], a[2], a[3] != 0, a[4], a[5]));
    else if (!std::strcmp(f, "sl_fold_rows")) std::printf("%d\n", bfe::sl_fold_rows(a[0], a[1]));
    else if (!std::strcmp(f, "sl_three_blocks")) std::printf("%d\n", (int)bfe::sl_three_blocks(a[0], a[1]));
    else if (!std::strcmp(f, "mlp_grad_launch")) {
      const bfe::GradLaunch g = bfe::mlp_grad_launch(a[0]);
      std::printf("%d %d %d\n", g.waves, g.per, g.blocks);
    } else if (!std::strcmp(f, "mlp_leap_launch")) {
      const bfe::LeapLaunch g = bfe::mlp_leap_launch(a[0], a[1] != 0);
      std::printf("%d %d\n", g.waves, g.blocks);
    } else return 1;
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
        text = "\n".join(" ".join([name] + [str(int(v)) for v in c] + ["0"] * (6 - len(c))) for c in calls)
        r = subprocess.run([exe], input=text + "\n", capture_output=True, text=True, check=True)
        out = [[int(v) for v in line.split()] for line in r.stdout.splitlines()]
        assert len(out) == len(calls)
        return out
    return ask


def test_four_waves_only_where_the_chip_is_full(rule):
    """Up to three blocks of 256 points a CU (256 CUs) are resident with three
    waves a SIMD, so the four-wave build has nothing to give there; with
    cos(l phi) factors it gives from six, without from nine."""
    ns = [1, 256, 65_536, 131_072, 196_608, 262_144, 393_216, 500_000, 589_823, 600_000, 2_000_000]
    got = [bool(v[0]) for v in rule("eval_four_waves", [(n,) for n in ns])]
    assert got == [False] * 9 + [True] * 2
    got = [bool(v[0]) for v in rule("eval_four_waves", [(n, 1) for n in ns])]
    assert got == [False] * 6 + [True] * 5


# us of the one-lane and the split integrators on MI355X at (lmax, mmax), orbits
LEAPFROG = [((0, 0), 16_384, 321, 342), ((0, 0), 32_768, 303, 614), ((2, 2), 16_384, 552, 436),
            ((2, 2), 16_385, 555, 742), ((2, 2), 32_768, 578, 779), ((3, 3), 24_000, 762, 965),
            ((4, 4), 16_384, 833, 514), ((4, 4), 32_768, 814, 909), ((4, 4), 36_864, 812, 1285),
            ((4, 6), 32_768, 909, 905), ((4, 6), 36_864, 908, 1315), ((4, 8), 24_000, 1000, 939),
            ((4, 8), 32_769, 1007, 1320), ((6, 0), 32_768, 1006, 859), ((6, 4), 24_000, 1136, 1029),
            ((6, 4), 36_864, 1167, 1485), ((6, 6), 32_768, 1279, 804), ((6, 6), 36_864, 1274, 1112),
            ((8, 8), 32_768, 1629, 1312), ((8, 8), 36_864, 1614, 1905), ((10, 6), 16_384, 1927, 854),
            ((10, 6), 36_864, 1903, 2260), ((12, 12), 32_768, 2812, 1928)]
RK4 = [((2, 2), 16_384, 603, 418), ((2, 2), 24_000, 576, 747), ((3, 3), 32_768, 876, 956),
       ((2, 6), 32_768, 776, 838), ((4, 2), 32_768, 860, 820), ((4, 4), 24_000, 937, 869),
       ((4, 4), 36_864, 949, 1262), ((5, 5), 32_768, 1233, 986), ((5, 5), 36_864, 1229, 1391),
       ((6, 0), 36_864, 1254, 1164), ((6, 6), 36_864, 1535, 1076), ((8, 8), 36_864, 2069, 1896),
       ((10, 6), 36_864, 2603, 2276), ((12, 12), 36_864, 3805, 2796)]


def test_split_orbits_where_they_are_the_faster(rule):
    """At its default the limit takes, of the two forms, the one measured faster
    (within 8 %: the table's own spread, and the fixed cost at the smallest
    basis), for every basis; any other value is the limit."""
    for rk4, table in ((0, LEAPFROG), (1, RK4)):
        lim = rule("split_orbits_max", [(36_864, *b, rk4) for b, *_ in table])
        for (basis, n, one, split), (m,) in zip(table, lim):
            assert (split if n <= m else one) <= 1.08 * min(one, split), (rk4, basis, n, m)
    assert rule("split_orbits_max", [(0, 4, 4, 0), (1 << 40, 2, 2, 1), (5000, 10, 6, 0)]) == [[0], [1 << 40], [5000]]


# us of an evaluation on MI355X in input order, by split blocks (None: not taken by
# them, cos(l phi)) and in cell order at (lmax, mmax), points
EVALUATION = [((0, 0), 1000, 5.0, 7.4, 26), ((0, 0), 131_000, 6.6, 45, 33), ((2, 2), 16_384, 7.7, 10.1, 29),
              ((2, 2), 65_536, 9.0, 32, 31), ((4, 4), 16_384, 10.4, 11.4, 32), ((4, 4), 40_000, 11.7, 27, 33),
              ((4, 4), 65_536, 13, 36, 33), ((4, 4), 100_000, 23, 51, 37), ((4, 4), 131_071, 25, 66, 39),
              ((4, 8), 4096, 12.9, 9.7, 34), ((4, 8), 24_576, 16.7, 22.5, 34), ((4, 8), 98_304, 41, 59, 45),
              ((6, 4), 8192, 15, 10.9, 36), ((6, 4), 32_768, 17.7, 22.6, 36), ((6, 4), 131_071, 36, 73, 42),
              ((6, 6), 16_384, 16.7, 8.6, 37), ((6, 6), 49_152, 22, 20.5, 37), ((6, 6), 65_536, 22.6, 26.6, 37),
              ((6, 6), 80_000, 42, 32, 39), ((6, 6), 131_071, 44, 49, 43), ((8, 8), 16_384, 28, 18.7, 40),
              ((8, 8), 65_536, 31, 52, 41), ((8, 8), 98_304, 59, 73, 51), ((8, 8), 131_071, 59, 95, 57),
              ((10, 6), 16_384, 32, 20, 42), ((10, 6), 40_000, 33, 42, 43), ((10, 6), 65_536, 33, 54, 41),
              ((10, 6), 100_000, 63, 77, 49), ((12, 12), 20_000, 48, 39, 54), ((12, 12), 49_152, 48, 57, 58),
              ((12, 12), 80_000, 104, 88, 69), ((12, 12), 131_071, 98, 137, 69),
              ((4, 4), 100_000, 22.6, None, 39), ((6, 6), 65_536, 25.2, None, 40), ((6, 6), 131_071, 42.5, None, 47),
              ((10, 6), 65_536, 45, None, 53), ((10, 6), 100_000, 62, None, 58), ((12, 12), 65_536, 72, None, 76),
              ((12, 12), 100_000, 104, None, 90)]
TWO_INPUTS = [((0, 0), 49_152, 20.5, 28.2), ((2, 2), 80_000, 38, 32.5), ((4, 4), 49_152, 28, 33), ((4, 4), 57_344, 35, 33),
              ((4, 4), 131_071, 66, 39), ((6, 4), 65_536, 40, 36.5), ((6, 6), 65_536, 26.6, 37), ((6, 6), 114_688, 44, 46),
              ((6, 6), 131_071, 49, 43), ((10, 6), 40_000, 42, 43), ((10, 6), 65_536, 54, 41), ((12, 12), 130_000, 136, 69)]


def test_evaluation_takes_the_fastest_form(rule):
    """At the default limits the form taken is the one measured fastest, within
    10 % (the spread of the figures and the steps of the limits)."""
    got = rule("eval_form", [(n, *b, s is not None, 65_536, 131_072) for b, n, _, s, _ in EVALUATION])
    for (basis, n, *us), (form,) in zip(EVALUATION, got):
        assert us[form] is not None and us[form] <= 1.10 * min(u for u in us if u), (basis, n, form)
    got = rule("eval_split_two", [(n, *b, 1, 65_536, 131_072) for b, n, _, _ in TWO_INPUTS])
    for (basis, n, split, ordered), (yes,) in zip(TWO_INPUTS, got):
        assert (split if yes else ordered) <= 1.10 * min(split, ordered), (basis, n, yes)


def test_evaluation_form_follows_explicit_knobs(rule):
    """Other values than the defaults hold for every basis: split up to the knob
    where it can be, cell order from twice order_min points."""
    calls = [(5000, 2, 2, 1, 1 << 40, 1 << 40), (5000, 2, 2, 0, 1 << 40, 1 << 40), (5000, 12, 12, 1, 1 << 40, 0),
             (5000, 12, 12, 1, 1, 0), (1, 6, 6, 1, 1, 0), (131_071, 6, 6, 1, 65_536, 0), (131_072, 6, 6, 1, 65_536, 0)]
    assert [v[0] for v in rule("eval_form", calls)] == [1, 0, 0, 2, 0, 0, 2]
    calls = [(5000, 2, 2, 1, 1 << 40, 1 << 40), (5000, 2, 2, 0, 1 << 40, 1 << 40), (5000, 2, 2, 1, 1, 1 << 40),
             (5000, 2, 2, 1, 1 << 40, 4999), (131_072, 6, 6, 1, 65_536, 131_072)]
    assert [v[0] for v in rule("eval_split_two", calls)] == [1, 0, 0, 0, 0]


# us of a whole-table SL evaluation on MI355X with one and two nodes a group of lanes
# at numr, lmax (nmax 20)
SL_FOLD = [(300, 0, 7.6, 8.3), (300, 8, 21.1, 21.7), (1000, 1, 8.9, 9.6), (1000, 4, 13.2, 13.8), (1000, 6, 19.0, 18.2),
           (2000, 0, 7.8, 8.5), (2000, 2, 10.3, 11.0), (2000, 3, 12.9, 12.4), (2000, 6, 22.1, 20.4),
           (4000, 1, 9.2, 10.0), (4000, 2, 11.8, 11.2), (4000, 8, 41.0, 36.9)]


def test_sl_fold_shares_rows_where_it_is_the_faster(rule):
    for (numr, lmax, *us), (rows,) in zip(SL_FOLD, rule("sl_fold_rows", [v[:2] for v in SL_FOLD])):
        assert us[rows - 1] == min(us), (numr, lmax, rows)


# (particles, LDS bytes a block, us with two blocks a CU, us with three)
SL_ALONE = [(30_000, 49_284, 25.4, 26.3), (60_000, 49_284, 45.4, 43.7), (60_000, 49_476, 45.6, 43.7),
            (300_000, 49_476, 178.5, 151.2), (1_000_000, 49_476, 481.6, 401.6), (150_000, 54_756, 101.4, 104.1),
            (1_000_000, 54_756, 521.0, 531.9)]


def test_halo_sums_take_three_blocks_where_they_are_the_faster(rule):
    for (n, lds, *us), (three,) in zip(SL_ALONE, rule("sl_three_blocks", [(-(-n // 64), lds) for n, lds, *_ in SL_ALONE])):
        assert us[three] == min(us), (n, lds, three)


def test_surrogate_inference_fills_the_device(rule):
    """No size makes a wave take more tiles in sequence than the device's waves
    leave it (plus the rounding to rounds of equal length), one wave a SIMD where
    that is enough, every point covered."""
    ns = [1, 15, 16, 17, 64, 65, 1000, 16_383, 16_384, 16_385, 20_000, 32_768, 32_769, 40_000, 49_152, 65_536, 65_537,
          80_000, 98_305, 131_072, 131_073, 200_000, 262_145, 524_289, 1_000_000, 10_000_001]
    for n, (waves, per, blocks) in zip(ns, rule("mlp_grad_launch", [(n,) for n in ns])):
        tiles = -(-n // 16)
        assert waves == (4 if n <= 16_384 else 8) and 1 <= per <= 4 and 1 <= blocks <= 256
        sweep = blocks * waves * per
        steps = -(-tiles // sweep) * per          # tiles of the busiest wave
        ideal = -(-tiles // (256 * waves))
        assert steps <= ideal * 1.25, (n, waves, per, blocks)


@pytest.mark.parametrize("conservative,per_wave", [(1, 16), (0, 32)])
def test_surrogate_orbits_take_one_tile_a_block(rule, conservative, per_wave):
    """A block walks several tiles of orbits only once eight blocks a CU are there."""
    ns = [1, 64, 65, 128, 129, 1000, 16_384, 16_385, 20_000, 65_536, 100_000, 262_144, 262_145, 1_000_000]
    for n, (waves, blocks) in zip(ns, rule("mlp_leap_launch", [(n, conservative) for n in ns])):
        assert waves == (4 if conservative and n <= 16_384 else 8)
        assert blocks == min(2048, -(-n // (waves * per_wave))), n
