"""One row on tiles of 64 columns (gemm_m1.h): every ring, wave count and number of k parts forced on the smallest and on ragged problems,
against the oracle; both word orders, the additions, and which calls take it.  On the CPU: its fetch schedule replayed, and the
estimate (m1_plan.h) by itself."""
import ctypes
import os
import re
import subprocess

import pytest
import torch

from test_fetch_schedule import Memory
from test_gemm_gpu import dev, one_hot_case, problem, run
from test_repack_layout import gpu_case

# (n, k, quant_cols): one tile of one unit of 128 rows, all FP6, all INT4, waves without a slice, ragged slices, the longest slice
SHAPES = [(128, 128, -1), (256, 128, 256), (384, 640, 128), (512, 1152, 256), (640, 2048, -1), (256, 1408, 256), (256, 4096, 128)]

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def replay(steps, depth, fp6, group, staged, pieces=2, lenient=0):
    """stream_m1 and what the kernel issues in front of it: `steps` steps of 64 rows of k (even, 2 .. 16)."""
    group, ops = group and not fp6, 3 if fp6 else 2
    mem, issued, slot_in = Memory(), 0, 0

    def issue():
        nonlocal issued, slot_in
        for o in range(ops):
            mem.load(("step", slot_in, o), issued)
        mem.expect(("step", slot_in, 0), issued)
        issued, slot_in = issued + 1, (slot_in + 1) % depth

    def wait(newer, most):                                      # wait_steps
        newer = max(0, min(newer, most))
        mem.wait(ops * newer + (lenient if newer else 0))

    def fetch(step, slot):
        for o in range(ops):
            mem.read(("step", slot, o), step)
        if not staged:                                          # (staged: the wave wrote them itself)
            mem.read(("A", 0 if step < 8 else 1), "A")

    if not group:
        mem.load(("column scales", 0), "S")
    for o in range(pieces if staged else 0):
        mem.load(("row", o), "row")
    if staged:
        for t in range(-(-steps // 4) * 4):
            mem.load(("entry", t), t)
    else:
        for o in range(1 + (steps > 8)):
            mem.load(("A", o), "A")
    if group:
        mem.load(("group scales", 0), "S")
    for _ in range(depth - 1):
        if issued < steps:
            issue()
    if staged:
        wait(issued, depth - 1)
        for o in range(pieces):                                 # (for the others too, behind the barrier)
            mem.read(("row", o), "row")
        for t in range(-(-steps // 4) * 4):
            mem.read(("entry", t), t)
    wait(issued - 1, depth - 2)
    fetch(0, 0)
    slot_rd = 1 % depth
    for s in range(0, steps, 2):
        for u in range(2):
            if issued < steps:
                issue()
            wait(issued - (s + u + 2), depth - 2)
            if s + u + 1 < steps:
                fetch(s + u + 1, slot_rd)
            else:                                               # the look-ahead past the end reads what nobody uses
                mem.pending_reads.clear()
            slot_rd = (slot_rd + 1) % depth
        if group:
            mem.read(("group scales", 0), "S")
    mem.wait(0)


@pytest.mark.parametrize("staged", [False, True])
def test_fetch_schedule(staged):
    for steps in range(2, 17, 2):
        for depth in (3, 4):
            for group in (False, True):
                replay(steps, depth, False, group, staged)
        replay(steps, 3, True, False, staged)


@pytest.mark.parametrize("staged", [False, True])
def test_fetch_schedule_notices_a_lenient_wait(staged):
    for fp6, group in ((False, True), (False, False), (True, False)):
        with pytest.raises(AssertionError, match="before its load completed"):
            replay(16, 3, fp6, group, staged, lenient=1)


def test_every_wave_of_a_staged_row_meets_one_barrier():
    """The row's pieces are for the whole workgroup: a wave with a slice meets the barrier inside stream_m1, one without meets its own,
    each behind a wait for its pieces."""
    with open(os.path.join(ROOT, "fp6-marlin_amd", "csrc", "gemm_m1.h")) as f:
        text = f.read()
    inside, kernel = text.split("__global__")
    assert inside.count("__builtin_amdgcn_s_barrier") == 1 and kernel.count("__builtin_amdgcn_s_barrier") == 1
    assert re.search(r"if constexpr \(STAGED\) \{\s+wait_steps<[^;]*;[^\n]*\n\s+__builtin_amdgcn_s_barrier", inside)
    assert re.search(r"else if constexpr \(STAGED\) \{\s+__builtin_amdgcn_s_waitcnt\(vmcnt_only\(0\)\);[^\n]*\n\s+__builtin_amdgcn_s_barrier", kernel)


WRAPPER = """
#include "m1_plan.h"
extern "C" int takes(int units, long long n4, long long qc, int group) { return fp6m::m1_choice(units, n4, qc, group != 0, 256, 72).us > 0.0; }
"""


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    d = tmp_path_factory.mktemp("m1_plan")
    (d / "plan.cpp").write_text(WRAPPER)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{ROOT}/fp6-marlin_amd/csrc",
                           "-o", str(d / "plan.so"), str(d / "plan.cpp")])
    takes = ctypes.CDLL(str(d / "plan.so")).takes
    takes.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_longlong, ctypes.c_int]
    return lambda k, n, qc, gs: bool(takes(k // 128, n - qc, qc, gs == 128))


def test_fp6_columns_alone_are_estimated_by_their_own_cuts(choice):
    """us of one-wave workgroups and of the best cut of 64-column tiles, where one of them is 3 % to 40 % behind."""
    for k, n, one_wave, tiles64 in ((2816, 17664, 10.67, 11.79), (3328, 19328, 12.06, 13.40), (3200, 33152, 17.97, 19.69),
                                    (2688, 33152, 15.45, 16.98), (4608, 18304, 15.55, 16.95), (2688, 37120, 16.39, 17.86)):
        assert not choice(k, n, n, -1), (k, n, one_wave, tiles64)
    for k, n, one_wave, tiles64 in ((4224, 5760, 7.39, 7.19), (12928, 1024, 8.50, 5.68), (16512, 1024, 9.45, 6.10), (8832, 1792, 9.07, 5.77),
                                    (11136, 1408, 9.08, 5.71), (8064, 1280, 8.74, 5.49)):
        assert choice(k, n, n, -1), (k, n, one_wave, tiles64)


def test_no_third_workgroup_on_a_cu(choice):
    """us of one-wave workgroups and of 64-column tiles, three workgroups to a CU; and launches that fit by twos."""
    for k, n, qc, one_wave, tiles64 in ((21632, 5888, 256, 14.36, 15.55), (17536, 7808, 0, 14.53, 15.68), (22400, 5376, 256, 14.25, 15.27),
                                        (1920, 33664, 256, 9.08, 9.71), (2560, 37888, 256, 11.56, 12.16), (16896, 6144, 512, 12.88, 13.53)):
        assert not choice(k, n, qc, 128), (k, n, one_wave, tiles64)
    for k, n, qc, one_wave, tiles64 in ((1152, 2432, 1024, 4.46, 4.86), (1280, 3968, 1024, 4.54, 4.90), (1280, 4608, 1024, 4.68, 4.93)):
        assert not choice(k, n, qc, -1) and not choice(k, n, qc, 128), (k, n, one_wave, tiles64)    # (short k, much of it FP6)
    assert choice(8192, 8192, 256, 128) and choice(4096, 4096, 256, 128) and choice(4096, 12288, 256, 128) and choice(11008, 4096, 256, -1)


@pytest.mark.gpu
@pytest.mark.parametrize("wk", [4, 8])
@pytest.mark.parametrize("depth", [3, 4])
def test_against_oracle(oracle, depth, wk):
    for n, k, qc in SHAPES:
        for gs in (-1, 128):
            for ks, ks6 in ((1, 1), (1, 3), (2, 2), (5, 8)):
                run(oracle, 1, n, k, 128, 128, qc=qc, gs=gs, ksplit=ks, env={"FP6M_M1": depth, "FP6M_WK16": wk, "FP6M_SHARE6": ks6})
    for gs in (-1, 128):
        for ks in (1, 3):
            one_hot_case(oracle, 1, 512, 1152, 256, gs, {"m1": depth, "wk16": wk, "ksplit": ks})


@pytest.mark.gpu
@pytest.mark.parametrize("gs", [-1, 128])
def test_gfx950_order_gives_the_same_bits(oracle, gs):
    for ks in (1, 3):
        env = {"FP6M_M1": 3, "FP6M_WK16": 4, "FP6M_KSPLIT": ks}
        for k, n, qc in ((128, 256, 128), (1152, 640, 256), (640, 256, 256)):
            gpu_case(oracle, 1, k, n, qc, gs, env)


@pytest.mark.gpu
@pytest.mark.parametrize("m1", [4, 0])
@pytest.mark.parametrize("ks", [1, 3])
def test_additions(oracle, ks, m1):
    """Column map, bias and residual (in place too) are added in float32 and rounded once, here and by one-wave workgroups."""
    import fp6_marlin
    n, k, qc = 640, 1152, 128
    g = torch.Generator().manual_seed(ks)
    _, B, s = problem(oracle, n, k, qc, 128)
    A = torch.randn((1, k), generator=g).half().to(dev())
    c_cols = torch.randperm(n, generator=g).to(torch.int32).to(dev())
    bias, res = torch.randn(n, generator=g).half().to(dev()), torch.randn((1, n), generator=g).half().to(dev())
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    plain, mapped, full = (torch.empty((1, n), dtype=torch.half, device=dev()) for _ in range(3))
    with fp6_marlin.cabi.tuning(m1=m1, ksplit=ks):
        fp6_marlin.mul(A, B, plain, s, ws, qc, group_size=128)
        fp6_marlin.mul_fused(A, B, mapped, s, ws, qc, 128, c_cols=c_cols)
        fp6_marlin.mul_fused(A, B, full, s, ws, qc, 128, c_cols=c_cols, bias=bias, residual=res)
        inplace = res.clone()
        fp6_marlin.mul_fused(A, B, inplace, s, ws, qc, 128, c_cols=c_cols, bias=bias, residual=inplace)
        torch.cuda.synchronize()
    assert torch.equal(mapped[:, c_cols.long()], plain) and torch.equal(full, inplace)
    want = mapped.float() + bias.float() + res.float()           # (mapped is rounded once more: half an ulp of the product)
    assert ((full.float() - want).abs() <= 2 ** -10 * want.abs() + 2 ** -10 * mapped.float().abs() + 1e-6).all()


@pytest.mark.gpu
@pytest.mark.parametrize("more", [40, 41, 11000])
@pytest.mark.parametrize("k", [128, 640, 2048, 4096])
def test_gather_is_an_exact_reorder(oracle, k, more):
    """Slices of two steps to the longest, among them ones that end inside a group of four; entries out of range are clamped.
    Rows that are staged in LDS, and rows that are too long or not in whole 16 bytes."""
    import fp6_marlin
    n, qc, lda = 512, 256, k + more
    _, B, s = problem(oracle, n, k, qc, 128)
    g = torch.Generator().manual_seed(k)
    A = torch.randn((1, lda), generator=g).half().to(dev())
    cols = torch.randperm(lda, generator=g)[:k].to(torch.int32)
    cols[0], cols[k - 1] = -5, lda + 3
    cols = cols.to(dev())
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    for wk in (4, 8):
        for ks in (1, 3):
            out = [torch.full((1, n), float("nan"), dtype=torch.half, device=dev()) for _ in range(2)]
            with fp6_marlin.cabi.tuning(m1=3, wk16=wk, ksplit=ks):
                fp6_marlin.mul(A[:, cols.long().clamp(0, lda - 1)].contiguous(), B, out[0], s, ws, qc, group_size=128)
                fp6_marlin.mul_fused(A, B, out[1], s, ws, qc, 128, a_cols=cols)
                torch.cuda.synchronize()
            assert torch.equal(*out)


@pytest.mark.gpu
def test_which_calls_take_it(oracle, capfd):
    """Both sides of the estimate; k not in whole 128 rows, scales off their 16 bytes, and `sms` stay with the other kernel."""
    import fp6_marlin

    def takes(n, k, qc=256, gs=128, shift=0, **kw):
        n6 = max(qc, 0)
        B = torch.zeros(k * (n - n6) // 8 + k * n6 * 3 // 16, dtype=torch.int32, device=dev())
        s = torch.zeros((k // 128 if gs == 128 else 1) * (n - n6) + n6 + shift, dtype=torch.half, device=dev())[shift:]
        A = torch.zeros((1, k), dtype=torch.half, device=dev())
        C = torch.full((1, n), float("nan"), dtype=torch.half, device=dev())
        ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
        capfd.readouterr()
        with fp6_marlin.cabi.tuning(verbose=1):
            fp6_marlin.mul(A, B, C, s, ws, qc, group_size=gs, **kw)
            torch.cuda.synchronize()
        assert int(C.count_nonzero()) == 0
        return "64-column tiles" in capfd.readouterr().err

    assert takes(4096, 4096) and takes(12288, 4096) and takes(8192, 8192) and takes(4096, 11008, gs=-1)
    assert not takes(57344, 8192) and not takes(4096, 512)
    assert not takes(4096, 4096 + 64, gs=-1, thread_k=64, thread_n=256) and not takes(4096, 4096, sms=2)
    assert not takes(4096, 4096, shift=2)


@pytest.mark.gpu
def test_a_gather_that_no_staged_row_serves_stays_with_the_one_wave_kernel(oracle, capfd):
    """Gathered from memory, 64-column tiles were up to a third slower than one-wave workgroups: rows longer than the slab, rows
    not in whole 16 bytes, and launches whose workgroups share a CU by threes."""
    import fp6_marlin

    def takes(n, k, lda, qc=256, gs=128):
        B = torch.zeros(k * (n - qc) // 8 + k * qc * 3 // 16, dtype=torch.int32, device=dev())
        s = torch.zeros((k // 128 if gs == 128 else 1) * (n - qc) + qc, dtype=torch.half, device=dev())
        A = torch.zeros((1, lda), dtype=torch.half, device=dev())
        C = torch.full((1, n), float("nan"), dtype=torch.half, device=dev())
        ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
        cols = torch.arange(k - 1, -1, -1, dtype=torch.int32, device=dev())
        capfd.readouterr()
        with fp6_marlin.cabi.tuning(verbose=1):
            fp6_marlin.mul_fused(A, B, C, s, ws, qc, gs, a_cols=cols)
            torch.cuda.synchronize()
        assert int(C.count_nonzero()) == 0
        return "64-column tiles" in capfd.readouterr().err

    assert takes(4096, 11008, 11008) and takes(12288, 4096, 4104) and takes(8192, 8192, 14336)
    assert not takes(4096, 11008, 11009) and not takes(8192, 8192, 14344) and not takes(24192, 2048, 18432)
    assert not takes(4096, 28672, 28672) and not takes(40960, 2048, 2048)


@pytest.mark.gpu
@pytest.mark.parametrize("wk", [4, 8])
def test_gather_on_gfx950_order_gives_the_same_bits(oracle, wk):
    import fp6_marlin
    for n, k, qc, gs in ((512, 640, 256, 128), (256, 2048, 256, -1), (384, 1152, 128, -1)):
        _, B, s = problem(oracle, n, k, qc, gs)
        Bn = fp6_marlin.repack_gfx950(B, k, n, qc)
        g, lda = torch.Generator().manual_seed(k), k + 72
        A = torch.randn((1, lda), generator=g).half().to(dev())
        cols = torch.randperm(lda, generator=g)[:k].to(torch.int32).to(dev())
        ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
        for ks in (1, 3):
            out = [torch.full((1, n), float("nan"), dtype=torch.half, device=dev()) for _ in range(3)]
            with fp6_marlin.cabi.tuning(m1=3, wk16=wk, ksplit=ks):
                fp6_marlin.mul(A[:, cols.long()].contiguous(), B, out[0], s, ws, qc, group_size=gs)
                fp6_marlin.mul_fused(A, B, out[1], s, ws, qc, gs, a_cols=cols)
                fp6_marlin.mul_fused(A, Bn, out[2], s, ws, qc, gs, a_cols=cols, layout="gfx950")
                torch.cuda.synchronize()
            assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


@pytest.mark.gpu
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_an_activation_that_is_not_finite_leaves_no_finite_output(oracle, value):
    """Times a weight of zero it is a NaN too; a tile in parts saturates beyond the range of half."""
    import fp6_marlin
    n, k, qc = 384, 1152, 128
    for gs in (-1, 128):
        _, B, s = problem(oracle, n, k, qc, gs)
        A = torch.randn((1, k), generator=torch.Generator().manual_seed(1)).half()
        A[0, 700] = value
        ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
        for wk in (4, 8):
            for ks in (1, 3):
                C = torch.zeros((1, n), dtype=torch.half, device=dev())
                with fp6_marlin.cabi.tuning(m1=4, wk16=wk, ksplit=ks):
                    fp6_marlin.mul(A.to(dev()), B, C, s, ws, qc, group_size=gs)
                    torch.cuda.synchronize()
                assert not torch.isfinite(C).any()
