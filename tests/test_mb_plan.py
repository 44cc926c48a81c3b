"""The dispatcher's host arithmetic for launches of more than 16 rows (csrc/mb_plan.h), compiled here as it is: the partial tiles
of a split stay inside the scratch that the launch has, whatever the mix of tiles."""
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MIB = 1 << 20
WRAPPER = """
#include "mb_plan.h"
using namespace fp6m;
extern "C" long long split(int mb, long long tiles, long long tiles6, int mtiles, int k, int units, int cus, int sms, int fixed, long long scratch,
                           long long* ks6, int* wk, int* too_large)
{
    const MbSplit s = mb_split(mb, MbLaunch{tiles, tiles6, mtiles, k, units, cus, sms, 0, 0, false, fixed != 0, (size_t)scratch});
    *ks6 = s.ks6;
    *wk = s.wk;
    *too_large = s.too_large;
    return s.ks;
}
extern "C" double estimate(int mb, long long tiles, long long tiles6, int mtiles, int k, int units, int group)
{
    const MbSplit s = mb_split(mb, MbLaunch{tiles, tiles6, mtiles, k, units, 256, -1, 0, 0, false, false, (size_t)16 << 20});
    return mb_time(mb, s, tiles, tiles6, mtiles, k, units, group != 0, 256);
}
extern "C" long long slots(long long ks4, long long ks6, long long tiles4, long long tiles6, long long mtiles)
{
    return (long long)slots_used(ks4, ks6, tiles4, tiles6, mtiles);
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(WRAPPER)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{ROOT}/fp6-marlin_amd/csrc",
                           "-o", str(d / "plan.so"), str(d / "plan.cpp")])
    L = ctypes.CDLL(str(d / "plan.so"))
    i, ll = ctypes.c_int, ctypes.c_longlong
    L.split.restype = L.slots.restype = ll
    L.split.argtypes = [i, ll, ll, i, i, i, i, i, i, ll, ctypes.POINTER(ll), ctypes.POINTER(i), ctypes.POINTER(i)]
    L.slots.argtypes = [ll] * 5

    def split(mb, tiles, tiles6, mtiles, k, group, cus=256, sms=-1, fixed=False, scratch=16 * MIB):
        ks6, wk, large = ll(), i(), i()
        ks = L.split(mb, tiles, tiles6, mtiles, k, k // (128 if group else 64), cus, sms, fixed, scratch, ks6, wk, large)
        return ks, ks6.value, wk.value, bool(large.value)

    L.estimate.restype = ctypes.c_double
    L.estimate.argtypes = [i, ll, ll, i, i, i, i]

    def estimate(mb, m, k, n, qc, group):
        return L.estimate(mb, n // 128, qc // 128, -(-m // (16 * mb)), k, k // (128 if group else 64), group)

    split.slots, split.estimate = L.slots, estimate
    return split


def highest_slot(ks4, ks6, tiles4, tiles6, mtiles):
    """gemm_mb_kernel's slot_base + part, over every workgroup that shares its tile."""
    top = -1
    for mt in range(mtiles):
        base = mt * (tiles6 * ks6 + tiles4 * ks4)
        if ks6 > 1 and tiles6:
            top = max(top, base + tiles6 * ks6 - 1)
        if ks4 > 1 and tiles4:
            top = max(top, base + tiles6 * ks6 + tiles4 * ks4 - 1)
    return top


def test_slots_used_is_what_the_kernel_numbers(plan):
    for ks4 in (1, 2, 5):
        for ks6 in (1, 2, 3, 10):
            for tiles4 in (0, 1, 7):
                for tiles6 in (0, 1, 4):
                    for mtiles in (1, 2, 3):
                        assert plan.slots(ks4, ks6, tiles4, tiles6, mtiles) == highest_slot(ks4, ks6, tiles4, tiles6, mtiles) + 1


def test_a_finer_cut_of_the_fp6_tiles_alone_respects_the_scratch(plan):
    """Nothing is shared before the FP6 tiles' own cut: 200 of 300 tiles in two parts of 64 rows are 12.5 MiB, 254 of 258 almost
    16; the static scratch has 12, and the cells of later calls lie behind it."""
    for tiles6 in (200, 254):
        ks, ks6, _, large = plan(4, 300 if tiles6 == 200 else 258, tiles6, 1, 1024, False, fixed=True, scratch=12 * MIB)
        assert (ks, ks6, large) == (1, 1, False)
    assert plan(4, 300, 200, 1, 1024, False)[:2] == (1, 2)            # (16 MiB hold them)
    assert plan(4, 300, 20, 1, 1024, False, fixed=True, scratch=12 * MIB)[:2] == (1, 2)


def test_no_split_leaves_its_scratch(plan):
    rng = random.Random(5)
    shared = 0
    for _ in range(60000):
        mb, group = rng.choice([2, 3, 4, 8]), rng.random() < 0.5
        tiles = int(1.5 * 2 ** rng.uniform(0, 10))
        tiles6 = rng.choice([0, 1, 2, 4, tiles // 4, tiles // 2, tiles - 1, tiles, rng.randint(0, tiles)])
        tiles6 = min(tiles, max(0, tiles6))
        mtiles, k = rng.choice([1, 1, 1, 2, 2, 3, 5, 16]), 128 * rng.randint(1, 240)
        fixed = rng.random() < 0.5
        scratch = 12 * MIB if fixed else 16 * MIB
        ks, ks6, wk, large = plan(mb, tiles, tiles6, mtiles, k, group and tiles6 < tiles, cus=rng.choice([256, 256, 304, 64, 8]),
                                  sms=rng.choice([-1, -1, 2]), fixed=fixed, scratch=scratch)
        if large:
            continue
        assert ks >= 1 and ks <= ks6 <= 2 * ks and wk in (4, 8)
        top = highest_slot(ks, ks6, tiles - tiles6, tiles6, mtiles)
        shared += top >= 0
        assert (top + 1) * 16 * mb * 128 * 4 <= scratch, (mb, tiles, tiles6, mtiles, k, group, fixed, ks, ks6)
    assert shared > 10000


def longest(units, parts, wk):
    """Units of the longest slice of a wave that is served first, and of the two waves of a SIMD (make_wave_rule)."""
    per_part = units // parts
    lo = ly = per_part // wk
    if wk == 8 and per_part >= 16:
        lo = min((per_part * 100 + 344) // 688, per_part // 4)
        ly = min((per_part - 4 * lo) // 4, lo)
    rem = units - parts * (4 * lo + (wk - 4) * ly)
    older = lo + (rem > 0)
    return older, older + ((ly + (rem > 4 * parts)) if wk == 8 else 0)


def test_a_finer_cut_of_the_fp6_tiles_shortens_the_loop_and_keeps_row_tiles_together(plan):
    """Short of twice as finely as the INT4 tiles: with four waves or beyond eight parts only for 128 rows of k less at least, and
    not where two row tiles, a multiple of eight workgroups apart, would no longer read their words through one XCD's L2."""
    def of(mb, m, k, n, qc, group):
        return plan(mb, n // 128, qc // 128, -(-m // (16 * mb)), k, group)[:3]

    assert of(4, 86, 3840, 2048, 256, False) == (5, 5, 4)             # slices of 3 units in 5 parts and in 7
    assert of(2, 22, 9472, 2048, 1024, False) == (8, 8, 8)
    assert of(4, 110, 16384, 2560, 128, True)[:2] == (6, 6)         # 120 workgroups per row tile; 122 in 8 parts
    assert of(4, 114, 16128, 3584, 512, True)[:2] == (4, 6)           # 112; 120 in 6 parts, 124 in the 7 that fit
    assert of(3, 33, 13824, 5120, 512, False) == (6, 10, 8)
    assert of(2, 20, 4352, 9472, 1024, False) == (3, 4, 8)            # (a unit less, four parts)
    rng = random.Random(9)
    finer = 0
    for _ in range(40000):
        mb, group, mtiles = rng.choice([2, 3, 4]), rng.random() < 0.5, rng.choice([1, 1, 2])
        tiles, k = rng.randint(8, 160), 128 * rng.randint(8, 224)
        tiles6 = min(tiles, rng.choice([1, 2, 4, 8, tiles // 2]))
        group = group and tiles6 < tiles
        ks, ks6, wk, _ = plan(mb, tiles, tiles6, mtiles, k, group)
        if not ks < ks6 < 2 * ks:
            continue
        finer += 1
        unit = 128 if group else 64
        before, after = longest(k // unit, ks, wk), longest(k // unit, ks6, wk)
        apart = [mtiles > 1 and grid % 8 != 0 for grid in (tiles * ks, (tiles - tiles6) * ks + tiles6 * ks6)]
        less = max(b - a for a, b in zip(after, before)) * unit
        assert (apart[0] and not apart[1]) or (apart[0] == apart[1] and (less >= 128 or (wk == 8 and ks6 <= 8))), (mb, tiles, tiles6, mtiles, k, group)
    assert finer > 1000


# us on a 256-CU MI355X, weights not in any cache; each kind of launch that has constants of its own, the 32-row tiles of short k first
MEASURED = [(2, 64, 2048, 2560, 0, True, 9.23), (2, 64, 2048, 2048, 0, True, 9.05), (2, 40, 2048, 2304, 512, True, 9.15), (2, 77, 2560, 3584, 256, True, 11.62),
            (2, 35, 3328, 2560, 1024, True, 11.17), (2, 104, 10240, 5120, 256, True, 34.4), (2, 46, 4608, 8960, 1024, False, 16.5), (2, 305, 2304, 3584, 128, False, 18.1),
            (3, 67, 3328, 2560, 1024, True, 13.2), (3, 113, 13056, 4608, 1024, True, 31.7), (3, 283, 5888, 18944, 0, True, 98.4),
            (4, 62, 3584, 4608, 256, True, 15.0), (4, 115, 16384, 3072, 256, False, 23.6), (4, 77, 2560, 34816, 1024, True, 39.6)]


@pytest.mark.parametrize("mb,m,k,n,qc,group,us", MEASURED)
def test_estimated_times_are_near_measured_ones(plan, mb, m, k, n, qc, group, us):
    """Within 12 %: the fits' spread is 3-6 %, their worst points 11 %."""
    assert abs(plan.estimate(mb, m, k, n, qc, group) / us - 1) <= 0.12
