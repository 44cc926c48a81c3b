"""GPU tests of `mul_fused` (C ABI fp6m_mul_fused): the activation gather, the output column scatter and the
bias / residual additions around the GEMM.  The reference has no such entry; what pins it here:

* with nothing to add, the scattered result is the plain `mul` result bit for bit (C_fused[:, c_cols] == C);
* a gathered A equals `mul` on the materialised A[:, a_cols] bit for bit;
* bias / residual: fp16(x + bias + residual) where x is recovered exactly from a bias-free run whose outputs are
  integers (A and the dequantised weight are chosen so that every product sum is a small integer, hence exact in
  fp16 and fp32), and, on random data, the oracle's fp32 product plus the additions within the GEMM tolerance
  (mean |d| / mean |ref| <= 1e-3).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 1e-3


@pytest.fixture(scope="module")
def oracle():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from oracle import fp6m_oracle
    return fp6m_oracle


def dev():
    return torch.device("cuda:0")


def packed(oracle, k, n, qc, gs, seed=0):
    rng = np.random.default_rng(seed)
    w = rng.normal(0, 0.02, (k, n)).astype(np.float16)
    ref, b, s = oracle.gen_mixed_weight(w, qc, gs, strict=False)
    return ref, torch.from_numpy(b).to(dev()), torch.from_numpy(s).to(dev())


def plain(fp6_marlin, A, B, s, n, qc, gs):
    C = torch.full((A.shape[0], n), float("nan"), dtype=torch.half, device=dev())
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    fp6_marlin.cabi.mul(A, B, C, s, ws, qc, -1, -1, -1, 16, gs)
    torch.cuda.synchronize()
    assert int(ws.abs().sum()) == 0
    return C


@pytest.mark.parametrize("m", [1, 16, 48, 200, 1100])
def test_scatter_and_gather_are_exact_reorders(oracle, m):
    import fp6_marlin
    k, n, qc, gs = 1024, 768, 256, 128
    print(f"case fused reorder m={m}", flush=True)
    ref, B, s = packed(oracle, k, n, qc, gs)
    g = torch.Generator().manual_seed(m)
    lda = k + 64
    A_wide = torch.randn((m, lda), generator=g).half().to(dev())
    a_cols = torch.randperm(lda, generator=g)[:k].to(torch.int32).to(dev())
    c_cols = torch.randperm(n, generator=g).to(torch.int32).to(dev())
    fp6_marlin.check_column_map(a_cols, lda)
    fp6_marlin.check_column_map(c_cols, n, permutation=True)
    A = A_wide[:, a_cols.long()].contiguous()
    want = plain(fp6_marlin, A, B, s, n, qc, gs)

    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    for use_a, use_c in ((False, True), (True, False), (True, True), (False, False)):
        C = torch.full((m, n), float("nan"), dtype=torch.half, device=dev())
        fp6_marlin.mul_fused(A_wide if use_a else A, B, C, s, ws, qc, gs, a_cols=a_cols if use_a else None,
                             c_cols=c_cols if use_c else None)
        torch.cuda.synchronize()
        got = C[:, c_cols.long()] if use_c else C
        assert torch.equal(got, want), (use_a, use_c)
        assert int(ws.abs().sum()) == 0
    err = oracle.rel_err(want.cpu().numpy(), oracle.matmul_ref(A.cpu().numpy(), ref))
    assert err <= TOL


@pytest.mark.parametrize("m", [3, 16])
def test_fused_epilogue_with_int4_tiles_in_two_classes(oracle, m):
    """The scatter, bias-free fused path through the m <= 16 kernel's two-class plan (forced by pretending a chip of
    eight CUs): an exact reorder of the plain call's result, which takes the same plan."""
    import fp6_marlin
    k, n, qc, gs = 2048, 1536, 256, 128
    print(f"case fused two classes m={m}", flush=True)
    ref, B, s = packed(oracle, k, n, qc, gs)
    g = torch.Generator().manual_seed(m)
    A = torch.randn((m, k), generator=g).half().to(dev())
    c_cols = torch.randperm(n, generator=g).to(torch.int32).to(dev())
    with fp6_marlin.cabi.tuning(cls=1, cus=8):
        want = plain(fp6_marlin, A, B, s, n, qc, gs)
        ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
        C = torch.full((m, n), float("nan"), dtype=torch.half, device=dev())
        fp6_marlin.mul_fused(A, B, C, s, ws, qc, gs, c_cols=c_cols)
        torch.cuda.synchronize()
    assert torch.equal(C[:, c_cols.long()], want)
    assert int(ws.abs().sum()) == 0
    assert oracle.rel_err(want.cpu().numpy(), oracle.matmul_ref(A.cpu().numpy(), ref)) <= TOL


@pytest.mark.parametrize("m1", [None, 0])
@pytest.mark.parametrize("k,n,qc,gs", [(4096, 4096, 256, 128), (4096, 4096, 256, -1), (1024, 768, 256, 128), (2048, 512, -1, 128),
                                       (2048, 512, -1, -1), (1024, 384, 384, -1), (11008, 1024, 128, 128), (8192, 2048, 256, -1)])
def test_one_row_gather_inside_the_decode_kernel(oracle, capfd, k, n, qc, gs, m1):
    """One row: the decode kernels gather A themselves (no pass of its own): the one on 64-column tiles, which all of these shapes take
    except the one with a short k and many FP6 columns, and with m1 = 0 the one of one-wave workgroups.  Bit for bit the result of `mul` on the
    materialised row, and of the same call with the gather forced into the separate pass; map entries outside the row
    are clamped to it, as the pass does."""
    import fp6_marlin
    print(f"case gather inside k={k} n={n} qc={qc} gs={gs}", flush=True)
    ref, B, s = packed(oracle, k, n, qc, gs, seed=k + n)
    g = torch.Generator().manual_seed(k)
    lda = k + 192
    A_wide = torch.randn((1, lda), generator=g).half().to(dev())
    a_cols = torch.randperm(lda, generator=g)[:k].to(torch.int32)
    a_cols[5], a_cols[k - 3] = -7, lda + 11                        # clamped to columns 0 and lda - 1
    clamped = a_cols.clamp(0, lda - 1).long().to(dev())
    a_cols = a_cols.to(dev())
    knobs = {} if m1 is None else {"m1": m1}
    capfd.readouterr()
    with fp6_marlin.cabi.tuning(verbose=1, **knobs):
        want = plain(fp6_marlin, A_wide[:, clamped].contiguous(), B, s, n, qc, gs)
    kernel = "64-column tiles" if m1 is None and (k, n) != (1024, 768) else "one-wave workgroups"
    assert kernel in capfd.readouterr().err
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    for inside in (1, 0, 1):
        C = torch.full((1, n), float("nan"), dtype=torch.half, device=dev())
        with fp6_marlin.cabi.tuning(gather=inside, verbose=1, **knobs):
            fp6_marlin.mul_fused(A_wide, B, C, s, ws, qc, gs, a_cols=a_cols)
        torch.cuda.synchronize()
        assert kernel in capfd.readouterr().err
        assert torch.equal(C, want), inside
        assert int(ws.abs().sum()) == 0
    err = oracle.rel_err(want.cpu().numpy(), oracle.matmul_ref(A_wide[:, clamped].cpu().numpy(), ref))
    assert err <= TOL


@pytest.mark.parametrize("m", [3, 16, 40, 130])
def test_bias_and_residual_round_once(oracle, m):
    """Integer-valued products: the bias-free output x is exact, so the fused result must be fp16(x + b + r)
    with one rounding, bit for bit."""
    import fp6_marlin
    k, n, qc, gs = 256, 512, 128, -1
    print(f"case fused bias m={m}", flush=True)
    rng = np.random.default_rng(5)
    # weights on both grids: INT4 codes times scale 1 -> integers in [-8, 7]; FP6 values {0, +-1, +-2, +-3, +-4}
    w = rng.integers(-4, 5, (k, n)).astype(np.float16)
    w[:, :n - qc] = rng.integers(-7, 8, (k, n - qc))
    w[0, :n - qc] = 7.5                                               # max |w| = 7.5 -> INT4 scale 2 * 7.5 / 15 = 1
    w[0, n - qc:] = 28.0                                              # max |w| = 28 per column -> FP6 scale 1
    ref, b, s = oracle.gen_mixed_weight(w, qc, gs, strict=False)
    B, sd = torch.from_numpy(b).to(dev()), torch.from_numpy(s).to(dev())
    g = torch.Generator().manual_seed(m)
    A = torch.randint(-1, 2, (m, k), generator=g).half().to(dev())
    x = plain(fp6_marlin, A, B, sd, n, qc, gs)
    x_ref = A.float().cpu().numpy() @ ref.astype(np.float32)
    assert np.array_equal(x.float().cpu().numpy(), x_ref.astype(np.float16).astype(np.float32))
    assert np.abs(x_ref).max() < 2048                                 # integers below 2048: exact in fp16

    bias = (torch.randn(n, generator=g) * 3).half().to(dev())
    res = (torch.randn((m, n), generator=g) * 5).half().to(dev())
    c_cols = torch.randperm(n, generator=g).to(torch.int32).to(dev())
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    for use_b, use_r, use_c in ((True, False, False), (False, True, False), (True, True, False), (True, True, True)):
        C = torch.full((m, n), float("nan"), dtype=torch.half, device=dev())
        fp6_marlin.mul_fused(A, B, C, sd, ws, qc, gs, c_cols=c_cols if use_c else None, bias=bias if use_b else None,
                             residual=res if use_r else None)
        torch.cuda.synchronize()
        xs = torch.empty_like(x)
        if use_c:
            xs[:, c_cols.long()] = x
        else:
            xs = x
        want = xs.float() + (bias.float() if use_b else 0) + (res.float() if use_r else 0)
        assert torch.equal(C, want.half()), (use_b, use_r, use_c)
    # in place: residual is C itself
    C = res.clone()
    fp6_marlin.mul_fused(A, B, C, sd, ws, qc, gs, residual=C)
    torch.cuda.synchronize()
    assert torch.equal(C, (x.float() + res.float()).half())


def test_fused_on_random_data_against_oracle(oracle):
    import fp6_marlin
    for m, k, n, qc, gs in ((1, 2048, 1024, 256, 128), (16, 1024, 1536, 512, -1), (300, 1024, 1024, 256, 128)):
        print(f"case fused random m={m} k={k} n={n}", flush=True)
        ref, B, s = packed(oracle, k, n, qc, gs, seed=m)
        g = torch.Generator().manual_seed(m)
        A = torch.randn((m, k), generator=g).half()
        a_cols = torch.randperm(k, generator=g).to(torch.int32)
        c_cols = torch.randperm(n, generator=g).to(torch.int32)
        bias = torch.randn(n, generator=g).half()
        res = torch.randn((m, n), generator=g).half()
        C = torch.full((m, n), float("nan"), dtype=torch.half, device=dev())
        ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
        fp6_marlin.mul_fused(A.to(dev()), B, C, s, ws, qc, gs, a_cols=a_cols.to(dev()), c_cols=c_cols.to(dev()),
                             bias=bias.to(dev()), residual=res.to(dev()))
        torch.cuda.synchronize()
        prod = oracle.matmul_ref(A[:, a_cols.long()].numpy(), ref).astype(np.float32)
        want = np.empty_like(prod)
        want[:, c_cols.numpy()] = prod
        want = want + bias.float().numpy() + res.float().numpy()
        assert oracle.rel_err(C.cpu().numpy(), want) <= TOL


def test_fused_argument_errors():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fp6_marlin
    m, k, n = 4, 256, 256
    A = torch.zeros((m, k), dtype=torch.half, device=dev())
    B = torch.zeros(k * n // 8, dtype=torch.int32, device=dev())
    s = torch.ones(n, dtype=torch.half, device=dev())
    C = torch.zeros((m, n), dtype=torch.half, device=dev())
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    with pytest.raises(RuntimeError):
        fp6_marlin.mul_fused(A, B, C, s, ws, c_cols=torch.zeros(n - 1, dtype=torch.int32, device=dev()))
    with pytest.raises(RuntimeError):
        fp6_marlin.mul_fused(A, B, C, s, ws, bias=torch.zeros(n, dtype=torch.float32, device=dev()))
    with pytest.raises(RuntimeError):
        fp6_marlin.mul_fused(A, B, C, s, ws, residual=torch.zeros((m + 1, n), dtype=torch.half, device=dev()))
    with pytest.raises(ValueError):
        fp6_marlin.check_column_map(torch.full((n,), n, dtype=torch.int32, device=dev()), n)
    with pytest.raises(ValueError):
        fp6_marlin.check_column_map(torch.zeros(n, dtype=torch.int32, device=dev()), n, permutation=True)
    fp6_marlin.mul_fused(A, B, C, s, ws)                               # nothing to fuse: plain GEMM
    torch.cuda.synchronize()
    assert float(C.abs().sum()) == 0


def test_graph_replays_of_fused_and_row_mix_calls(oracle):
    """`mul`, `mul_fused` (gather + scatter + bias + residual) and `mul_rows` captured in one HIP graph: every
    replay, with eager work and synchronisation in between, reproduces the eager results bit for bit."""
    import fp6_marlin
    m, k, n, qc, gs, qr = 16, 1024, 512, 256, 128, 256
    ref, B, s = packed(oracle, k, n, qc, gs, seed=21)
    w = np.random.default_rng(22).normal(0, 0.02, (k, n)).astype(np.float16)
    _, br, sr = oracle.gen_row_mix_weight(w, qr)
    Br, Sr = torch.from_numpy(br).to(dev()), torch.from_numpy(sr).to(dev())
    g = torch.Generator().manual_seed(23)
    A = torch.randn((m, k), generator=g).half().to(dev())
    a_cols = torch.randperm(k, generator=g).to(torch.int32).to(dev())
    c_cols = torch.randperm(n, generator=g).to(torch.int32).to(dev())
    bias = torch.randn(n, generator=g).half().to(dev())
    res = torch.randn((m, n), generator=g).half().to(dev())
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    outs = [torch.empty((m, n), dtype=torch.half, device=dev()) for _ in range(3)]
    fp6_marlin.init_workspace(ws, gather=True)                          # nothing may allocate during capture

    def work():
        fp6_marlin.mul(A, B, outs[0], s, ws, qc, -1, -1, -1, 16, gs)
        fp6_marlin.mul_fused(A, B, outs[1], s, ws, qc, gs, a_cols=a_cols, c_cols=c_cols, bias=bias, residual=res)
        fp6_marlin.mul_rows(A, Br, outs[2], Sr, ws, qr, a_cols=a_cols)

    work()
    torch.cuda.synchronize()
    eager = [o.clone() for o in outs]
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        work()                                                          # warm-up on the capture stream
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        work()
    for rep in range(4):
        for o in outs:
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for o, e in zip(outs, eager):
            assert torch.equal(o, e), rep
        assert int(ws.abs().sum()) == 0
        fp6_marlin.mul(A, B, outs[0], s, ws, qc, -1, -1, -1, 16, gs)     # eager work between replays
        torch.cuda.synchronize()


def test_random_shapes_maps_and_additions_against_unpacked_words():
    """A seeded random walk over the fused entry point: shapes, FP6 column counts, scale modes, 1 .. 1100 rows (every
    kernel), any subset of activation gather (from a wider matrix), output permutation, bias and residual; random
    packed words against the pinned unpacker and an fp32 matmul with the same reorders and additions."""
    import random
    import fp6_marlin
    from fp6_marlin import cabi
    rnd = random.Random(7)
    g = torch.Generator().manual_seed(7)
    for ci in range(60):
        k = 256 * rnd.choice([1, 2, 3, 4, 8, 11, 16])
        n = 256 * rnd.choice([1, 2, 3, 5, 8, 16, 24, 43])
        qc = min(n, rnd.choice([0, 256, 256, 512, n, 128]))
        gs = rnd.choice([-1, 128])
        m = rnd.choice([1, 1, rnd.randint(2, 16), rnd.randint(17, 64), rnd.randint(65, 300), rnd.randint(300, 1100)])
        max_par = rnd.choice([16, 16, 2])
        n4 = n - qc
        B = torch.randint(-2 ** 31, 2 ** 31 - 1, (k * n4 // 8 + k * qc * 3 // 16,), generator=g, dtype=torch.int64).to(torch.int32)
        s = (torch.rand(((k // gs) * n4 if gs > 0 else n4) + qc, generator=g) * 0.01 + 0.001).half()
        qarg = qc if qc else -1
        use_a, use_c, use_b, use_r = [rnd.random() < 0.6 for _ in range(4)]
        lda = k + (rnd.choice([0, 64, 1000]) if use_a else 0)
        case = (ci, m, k, n, qc, gs, max_par, use_a, use_c, use_b, use_r, lda)
        print("case random fused", case, flush=True)
        w = fp6_marlin.unpack_to_fp16(B, s, k, n, qarg, gs).to(dev())
        ws = torch.zeros(n // 128 * max_par, dtype=torch.int32, device=dev())
        A = torch.randn((m, lda), generator=g).half().to(dev())
        a_cols = torch.randperm(lda, generator=g)[:k].to(torch.int32).to(dev()) if use_a else None
        c_cols = torch.randperm(n, generator=g).to(torch.int32).to(dev()) if use_c else None
        bias = (torch.randn(n, generator=g) * 0.5).half().to(dev()) if use_b else None
        resid = (torch.randn((m, n), generator=g) * 0.5).half().to(dev()) if use_r else None
        C = torch.full((m, n), float("nan"), dtype=torch.half, device=dev())
        cabi.mul_fused(A, B.to(dev()), C, s.to(dev()), ws, qarg, gs, a_cols=a_cols, c_cols=c_cols, bias=bias, residual=resid,
                       max_par=max_par)
        torch.cuda.synchronize()
        ref = (A[:, a_cols.long()] if use_a else A[:, :k]).float() @ w.float()
        if use_c:
            out = torch.empty_like(ref)
            out[:, c_cols.long()] = ref
            ref = out
        if use_b:
            ref = ref + bias.float()
        if use_r:
            ref = ref + resid.float()
        assert torch.isfinite(C).all(), case
        assert int(ws.abs().sum().item()) == 0, case
        d = (C.float() - ref).abs()
        assert (d.mean() / ref.abs().mean()).item() <= TOL, case
        assert bool((d <= 4e-3 * ref.abs() + 0.13 * ref.abs().mean()).all()), case
        del w, A, C, ref
        torch.cuda.empty_cache()
