"""The m <= 16 kernel on tiles of 64 columns (gemm_m16h.h): its fetch schedule replayed on the CPU, and on the GPU every ring width,
wave count and protocol forced on the smallest and on ragged problems, against the oracle and, where only the split of the
columns differs, bit for bit against tiles of 128."""
import numpy as np
import pytest
import torch

from test_fetch_schedule import Memory
from test_gemm_gpu import dev, one_hot_case, problem, run
from test_rows_gpu import run as run_rows


def replay(steps, depth, arows, fp6, group, lenient=0):
    """stream_half: `steps` steps of 64 rows of k (even)."""
    group = group and not fp6
    ops = (2 if arows == 16 else 1) + (3 if fp6 else 2)
    mem, issued = Memory(), 0

    def issue(slot, even):
        nonlocal issued
        assert even == (issued % 2 == 0)
        for o in range(ops):
            mem.load(("step", slot, o), issued)
        mem.expect(("step", slot, 0), issued)
        if group and even:
            mem.load(("S", (issued >> 1) % 4), issued >> 1)
            mem.expect(("S", (issued >> 1) % 4), issued >> 1)
        issued += 1

    def wait(newer, even):                                      # wait_steps
        newer = max(0, min(newer, depth - 2))
        mem.wait(ops * newer + ((newer + even) // 2 if group else 0) + (lenient if newer else 0))

    def fetch(step, slot):
        for o in range(ops):
            mem.read(("step", slot, o), step)

    slot_in, slot_rd = 0, 1
    for d in range(depth - 1):
        if issued < steps:
            issue(slot_in, d % 2 == 0)
            slot_in = (slot_in + 1) % depth
    wait(issued - 1, 0)
    fetch(0, 0)
    for s in range(0, steps, 2):
        for u in range(2):
            if issued < steps:
                issue(slot_in, (u + depth - 1) % 2 == 0)
                slot_in = (slot_in + 1) % depth
            wait(issued - (s + u + 2), 1 - u)
            if s + u + 1 < steps:
                fetch(s + u + 1, slot_rd)
            else:                                               # the look-ahead past the end reads what nobody uses
                mem.pending_reads.clear()
            slot_rd = (slot_rd + 1) % depth
        if group:
            mem.read(("S", (s >> 1) % 4), s >> 1)
    mem.wait(0)


@pytest.mark.parametrize("arows", [4, 8, 16])
def test_fetch_schedule(arows):
    for steps in (2, 4, 6, 8, 14, 32):
        replay(steps, 4, arows, fp6=False, group=True)
        replay(steps, 4, arows, fp6=False, group=False)
        replay(steps, 3, arows, fp6=True, group=False)


def test_fetch_schedule_notices_a_lenient_wait():
    with pytest.raises(AssertionError, match="before its load completed"):
        replay(16, 4, 16, fp6=False, group=True, lenient=1)


# (n, k, quant_cols): one tile of one unit, all FP6, all INT4, ragged numbers of units and tiles
SHAPES = [(128, 128, -1), (256, 128, 256), (384, 640, 128), (512, 1152, 256), (640, 2048, -1), (256, 1408, 256)]


@pytest.mark.gpu
@pytest.mark.parametrize("wk", [4, 8])
@pytest.mark.parametrize("m", [2, 4, 5, 8, 9, 16])
def test_against_oracle(oracle, m, wk):
    for n, k, qc in SHAPES:
        for gs in (-1, 128):
            for ks in (1, 2, 5):
                run(oracle, m, n, k, 128, 128, qc=qc, gs=gs, ksplit=ks, env={"FP6M_HALF": 1, "FP6M_WK16": wk})
    run(oracle, m, 512, 1152, qc=256, gs=128, ksplit=3, env={"FP6M_HALF": 1, "FP6M_XCD": 1})
    for gs in (-1, 128):
        one_hot_case(oracle, m, 512, 1152, 256, gs, {"half": 1, "wk16": wk, "ksplit": 2})
        one_hot_case(oracle, m, 384, 640, 128, gs, {"half": 1, "wk16": wk, "ksplit": 1})


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 2, 4, 5, 8, 9, 16])
def test_tiles_of_128_columns_give_the_same_bits(oracle, m):
    """Whole numbers and scales of one: every order of the sums is exact, whatever the tile, its parts and how they meet."""
    import fp6_marlin
    for k, n, qc, gs in ((1152, 640, 256, 128), (1152, 640, 256, -1), (640, 256, 256, -1), (2048, 384, -1, 128)):
        rng, n6 = np.random.default_rng(k + m), max(qc, 0)
        w = rng.integers(-4, 5, (k, n)).astype(np.float16)
        w[::128, :n - n6] = 7.5                                     # the largest of every group of rows: INT4 scale 1
        w[0, n - n6:] = 28.0                                        # and of every column: FP6 scale 1
        ref, b, s = oracle.gen_mixed_weight(w, qc, gs, strict=False)
        assert (s == 1).all()
        B, sd = torch.from_numpy(b).to(dev()), torch.from_numpy(s).to(dev())
        a = rng.integers(-1, 2, (m, k)).astype(np.float16)
        A, ws = torch.from_numpy(a).to(dev()), torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
        want = (a.astype(np.float64) @ ref.astype(np.float64)).astype(np.float16)
        plans = [{"m1": 0}, {"m1": 3, "wk16": 4, "ksplit": 2}, {"m1": 4, "wk16": 8, "ksplit": 1}] if m == 1 else [{"half": 0}]
        plans += [{"half": 1, "wk16": wk, "ksplit": ks} for wk in (4, 8) for ks in (1, 3)] if m > 1 else []
        for plan in plans:
            C = torch.full((m, n), float("nan"), dtype=torch.half, device=dev())
            with fp6_marlin.cabi.tuning(**plan):
                fp6_marlin.mul(A, B, C, sd, ws, qc, group_size=gs)
                torch.cuda.synchronize()
            assert np.array_equal(C.cpu().numpy(), want), plan


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 7, 16])
def test_rows_that_are_not_finite_stay_their_own(oracle, m):
    """One row with an infinity and one with a NaN: none of their outputs is finite, and the other rows are what they are without."""
    import fp6_marlin
    n, k, qc = 384, 1152, 128
    _, B, s = problem(oracle, n, k, qc, 128)
    clean = torch.randn((m, k), generator=torch.Generator().manual_seed(m)).half()
    bad = clean.clone()
    bad[0, 700], bad[m - 1, 3] = float("-inf"), float("nan")
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    for wk in (4, 8):
        for ks in (1, 3):
            out = []
            for A in (clean, bad):
                out.append(torch.zeros((m, n), dtype=torch.half, device=dev()))
                with fp6_marlin.cabi.tuning(half=1, wk16=wk, ksplit=ks):
                    fp6_marlin.mul(A.to(dev()), B, out[-1], s, ws, qc, group_size=128)
                    torch.cuda.synchronize()
            assert torch.isfinite(out[0]).all() and torch.equal(out[0][1:m - 1], out[1][1:m - 1])
            assert not torch.isfinite(out[1][0]).any() and not torch.isfinite(out[1][m - 1]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [5, 8, 16])
def test_placement_per_xcd_only_where_it_is_built(oracle, capfd, m):
    """Ten tiles of 64 columns in two parts are 20 workgroups; placed per XCD the grid is padded to 32.  Workgroups of eight waves
    have no build that knows the twelve surplus ones, whatever is asked for."""
    for wk, placed in ((8, False), (4, True)):
        capfd.readouterr()
        run(oracle, m, 640, 2048, qc=-1, gs=128, ksplit=2, thread_k=128, thread_n=128,
            env={"FP6M_HALF": 1, "FP6M_XCD": 1, "FP6M_WK16": wk, "FP6M_VERBOSE": 1})
        err = capfd.readouterr().err
        assert f" half (1x{wk} waves)" in err and ("placed per XCD" in err) == placed and ("grid=20" in err) == (not placed), err


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 4])
def test_no_more_parts_than_the_cells_count(oracle, capfd, m):
    """Up to four rows these tiles have no way to meet but the cells, whose count of arrivals ends at 255."""
    for ks, want in ((300, "ks4=255 ks6=255"), (255, "ks4=255 ks6=255"), (254, "ks4=254 ks6=254")):
        capfd.readouterr()
        run(oracle, m, 256, 640, 128, 128, qc=128, gs=128, ksplit=ks, env={"FP6M_HALF": 1, "FP6M_VERBOSE": 1})
        err = capfd.readouterr().err
        assert " half " in err and want in err, err


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 4, 7, 16])
def test_row_mix(oracle, m):
    import fp6_marlin
    for k, qr in ((512, 256), (1024, 128), (1024 + 896, 896), (256, 128)):
        for ks in (None, 3):
            real = fp6_marlin.cabi.tuning
            try:
                fp6_marlin.cabi.tuning = lambda **kw: real(half=1, **kw)
                run_rows(oracle, m, k, 384, qr, ksplit=ks)
            finally:
                fp6_marlin.cabi.tuning = real


@pytest.mark.gpu
@pytest.mark.parametrize("m", [3, 6, 16])
def test_additions_are_an_exact_reorder_of_the_plain_call(oracle, m):
    """Column map, bias and residual (in place too) with everything a power of two, so that any order of the sums is exact."""
    import fp6_marlin
    n, k, qc = 640, 1152, 128
    g = torch.Generator().manual_seed(m)
    _, B, s = problem(oracle, n, k, qc, 128)
    A = torch.randn((m, k), generator=g).half().to(dev())
    c_cols = torch.randperm(n, generator=g).to(torch.int32).to(dev())
    bias = torch.randn(n, generator=g).half().to(dev())
    res = torch.randn((m, n), generator=g).half().to(dev())
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    for ks in (1, 3):
        with fp6_marlin.cabi.tuning(half=1, ksplit=ks):
            plain = torch.empty((m, n), dtype=torch.half, device=dev())
            fp6_marlin.mul(A, B, plain, s, ws, qc, group_size=128)
            mapped = torch.empty_like(plain)
            fp6_marlin.mul_fused(A, B, mapped, s, ws, qc, 128, c_cols=c_cols)
            full = torch.empty_like(plain)
            fp6_marlin.mul_fused(A, B, full, s, ws, qc, 128, c_cols=c_cols, bias=bias, residual=res)
            inplace = res.clone()
            fp6_marlin.mul_fused(A, B, inplace, s, ws, qc, 128, c_cols=c_cols, bias=bias, residual=inplace)
            torch.cuda.synchronize()
        assert torch.equal(mapped[:, c_cols.long()], plain)
        assert torch.equal(full, inplace)
        want = mapped.float() + bias.float() + res.float()       # (mapped is rounded once more: half an ulp of the product)
        assert ((full.float() - want).abs() <= 2 ** -10 * want.abs() + 2 ** -10 * mapped.float().abs() + 1e-6).all()
        assert int(ws.abs().sum()) == 0


@pytest.mark.gpu
def test_where_the_narrow_tiles_are_taken(oracle, capfd):
    """Both sides of the choice, and what keeps calls on 128 columns: k or quant_rows not in whole 128 rows, one counter per tile."""
    import fp6_marlin

    def takes(m, n, k, qc=256, gs=128, max_par=16, **kw):
        _, B, s = None, torch.zeros(k * n // 8 + k * max(qc, 0) // 16, dtype=torch.int32, device=dev()), \
            torch.zeros((k // 128 if gs == 128 else 1) * (n - max(qc, 0)) + max(qc, 0), dtype=torch.half, device=dev())
        A = torch.zeros((m, k), dtype=torch.half, device=dev())
        C = torch.full((m, n), float("nan"), dtype=torch.half, device=dev())
        ws = torch.zeros(n // 128 * max_par, dtype=torch.int32, device=dev())
        capfd.readouterr()
        with fp6_marlin.cabi.tuning(verbose=1):
            fp6_marlin.mul(A, B, C, s, ws, qc, max_par=max_par, group_size=gs, **kw)
            torch.cuda.synchronize()
        assert int(C.count_nonzero()) == 0 and int(ws.abs().sum()) == 0
        return " half " in capfd.readouterr().err

    assert takes(16, 4096, 4096) and takes(5, 15360, 5120) and takes(8, 4096, 11008) and takes(2, 4096, 4096)
    assert not takes(16, 8192, 8192, gs=-1) and not takes(8, 28672, 6144)
    assert not takes(16, 4096, 4096, max_par=1) and takes(2, 4096, 4096, max_par=1)
    assert not takes(16, 4096, 4096 + 64, gs=-1, thread_k=64, thread_n=256) and not takes(16, 4096, 4096, sms=2)


@pytest.mark.gpu
def test_calls_near_the_line_keep_the_wide_tiles(oracle, capfd):
    """Calls on which tiles of 64 columns were 5 to 12 % slower than tiles of 128, and some on which they are far faster."""
    import fp6_marlin

    def takes(m, k, n, qc, gs, qr=0):
        B = torch.zeros((k - qr) * (n - qc) // 8 + (k * qc + qr * n) * 3 // 16, dtype=torch.int32, device=dev())
        s = torch.zeros(((k - qr) // 128 if gs == 128 else 1) * (n - qc) + (n if qr else qc), dtype=torch.half, device=dev())
        A, C = torch.zeros((m, k), dtype=torch.half, device=dev()), torch.empty((m, n), dtype=torch.half, device=dev())
        ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
        capfd.readouterr()
        with fp6_marlin.cabi.tuning(verbose=1):
            if qr:
                fp6_marlin.mul_rows(A, B, C, s, ws, qr)
            else:
                fp6_marlin.mul(A, B, C, s, ws, qc if qc else -1, group_size=gs)
            torch.cuda.synchronize()
        return " half " in capfd.readouterr().err

    for m, k, n, qr in ((1, 1792, 20224, 512), (1, 1792, 17664, 512), (3, 1664, 21248, 512), (12, 1664, 17024, 512)):
        assert not takes(m, k, n, 0, 128, qr=qr)
    assert takes(16, 4096, 4096, 0, 128, qr=256)
    for m, k, n, qc, gs in ((9, 18560, 4352, 256, 128), (7, 14464, 7040, 0, -1), (10, 17664, 4864, 256, 128), (15, 15616, 3968, 256, 128)):
        assert not takes(m, k, n, qc, gs)
    for m, k, n in ((14, 19328, 4608), (12, 12288, 7296), (10, 10752, 6912), (16, 17024, 5248), (15, 18560, 4608), (10, 11392, 7424)):
        assert not takes(m, k, n, n, -1)
    assert takes(6, 27776, 1536, 0, 128) and takes(7, 19968, 1024, 256, 128) and takes(5, 4096, 1024, 1024, -1)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 7, 16])
def test_gfx950_order_gives_the_same_bits(oracle, m):
    """Words in either order through tiles of 64 columns: the smallest tile, ragged units, all FP6, FP6 rows."""
    import fp6_marlin
    from test_repack_layout import gpu_case
    for wk in (4, 8):
        for ks in (1, 3):
            env = {"FP6M_HALF": 1, "FP6M_WK16": wk, "FP6M_KSPLIT": ks}
            gpu_case(oracle, m, 128, 256, 128, 128, env)
            gpu_case(oracle, m, 1152, 640, 256, -1, env)
            gpu_case(oracle, m, 640, 256, 256, -1, env)
    k, n, qr = 1024 + 384, 384, 384
    ref, b, s = oracle.gen_row_mix_weight(np.random.default_rng(m).normal(0, 0.02, (k, n)).astype(np.float16), qr)
    B, sd = torch.from_numpy(b).to(dev()), torch.from_numpy(s).to(dev())
    Bn = fp6_marlin.repack_gfx950(B, k, n, quant_rows=qr)
    A = torch.randn((m, k), generator=torch.Generator().manual_seed(m)).half().to(dev())
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    out = [torch.empty((m, n), dtype=torch.half, device=dev()) for _ in range(2)]
    with fp6_marlin.cabi.tuning(half=1, ksplit=2):
        fp6_marlin.mul_rows(A, B, out[0], sd, ws, qr)
        fp6_marlin.mul_rows(A, Bn, out[1], sd, ws, qr, layout="gfx950")
        torch.cuda.synchronize()
    assert torch.equal(*out) and oracle.rel_err(out[0].cpu().numpy(), oracle.matmul_ref(A.cpu().numpy(), ref)) <= 1e-3
