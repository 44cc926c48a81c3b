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

    split.slots = L.slots
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
