"""On-GPU weight preparation against the host path (which tests/test_cpu_routines.py pins to the oracle bit for
bit): packed words, scales and the dequantised check weight must be identical."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev():
    return torch.device("cuda:0")


def same_bits(a, b):
    return torch.equal(a.cpu().contiguous().view(torch.int16), b.cpu().contiguous().view(torch.int16))


def same_values(a, b):
    # the host INT4 check weight writes +0 where the GPU kernel writes the product's sign: compare as numbers
    return np.array_equal(a.cpu().numpy().astype(np.float32), b.cpu().numpy().astype(np.float32))


@pytest.mark.parametrize("k,n,qc,gs", [(256, 512, 256, 128), (256, 512, 256, -1), (512, 768, 128, 128), (256, 256, 256, -1),
                                       (256, 512, -1, 128), (1024, 1024, 512, -1), (128, 192, 64, 128)])
@pytest.mark.parametrize("harness", [True, False])
def test_device_pack_matches_host_pack(k, n, qc, gs, harness):
    import fp6_marlin
    g = torch.Generator().manual_seed(k * 7 + n + (qc if qc > 0 else 0))
    w = (torch.randn((k, n), generator=g) * 0.02).half()
    w[3, 5] = 0.0
    n4 = n - max(qc, 0)
    if n4 > 7:
        w[:, 7] = 0.0                                                 # an all-zero INT4 column: scale 0, codes 8
    if qc > 0 and not harness:
        w[:, n4 + 3] = 0.0                                            # an all-zero FP6 column: its scale becomes 1
    Bh, sh, rh = fp6_marlin.pack_mixed_weight(w, qc, gs, harness_layout=harness)
    Bd, sd, rd = fp6_marlin.pack_mixed_weight(w.to(dev()), qc, gs, harness_layout=harness)
    assert Bd.is_cuda and sd.is_cuda and rd.is_cuda
    assert torch.equal(Bd.cpu(), Bh)
    assert same_bits(sd, sh)
    assert same_values(rd, rh)


@pytest.mark.parametrize("k,n,qc,gs", [(64, 64, -1, -1), (192, 320, 64, 64), (960, 512, 64, 48), (320, 512, 256, 16), (576, 448, 192, -1),
                                       (128, 832, 64, 128), (8256, 192, 64, -1), (512, 1088, 320, 512)])
def test_device_pack_at_the_edges_of_its_workgroups(k, n, qc, gs):
    """Regions that end inside a workgroup's 256 columns, rows that end inside its 128, every kind of scale group, more row
    ranges than one for the column maxima; INT4 scales down to zero and through the sub-normal range.  Bit for bit."""
    import fp6_marlin
    g = torch.Generator().manual_seed(k + 3 * n)
    w = torch.randn((k, n), generator=g) * 0.02
    n4 = n - max(qc, 0)
    w[:, :n4:5] *= 2.0 ** -torch.randint(0, 16, (1, w[:, :n4:5].shape[1]), generator=g).float()
    w = w.half()
    w[:, 9] = 0.0
    Bh, sh, rh = fp6_marlin.pack_mixed_weight(w, qc, gs, harness_layout=False)
    Bd, sd, rd = fp6_marlin.pack_mixed_weight(w.to(dev()), qc, gs, harness_layout=False)
    assert torch.equal(Bd.cpu(), Bh)
    assert same_bits(sd, sh)
    assert same_values(rd, rh)


def test_every_fp6_code_and_range_errors():
    """A column whose largest magnitude is 28 has scale 1, so its entries are cast as they are: feed every
    binary16 pattern inside [0.0625, 28] (and both zeros) through the GPU cast and compare with the host's."""
    import fp6_marlin
    allh = torch.arange(0, 65536, dtype=torch.int32).to(torch.int16).view(torch.float16)
    mag = allh.float().abs()
    ok = allh[((mag >= 0.0625) & (mag <= 28.0)) | (mag == 0)]
    k, qc = 256, 128
    reps = (k * qc + ok.numel() - 1) // ok.numel()
    w6 = ok.repeat(reps)[: k * qc].reshape(k, qc).clone()
    w6[0, :] = 28.0                                                   # every column: max 28 -> scale 1
    w = torch.cat([torch.randn(k, 128).half() * 0.02, w6], dim=1).contiguous()
    for harness in (True, False):
        Bh, sh, rh = fp6_marlin.pack_mixed_weight(w, qc, -1, harness_layout=harness)
        Bd, sd, rd = fp6_marlin.pack_mixed_weight(w.to(dev()), qc, -1, harness_layout=harness)
        assert torch.equal(Bd.cpu(), Bh) and same_bits(sd, sh) and same_values(rd, rh)
    bad = w.clone()
    bad[5, 130] = float("nan")
    with pytest.raises(ValueError):
        fp6_marlin.pack_mixed_weight(bad.to(dev()), qc, -1)
    with pytest.raises(ValueError):                                   # shape rule: quant_cols % 64
        fp6_marlin.pack_mixed_weight(w.to(dev()), 96, -1)


def test_a_pack_that_fails_at_its_launches_still_waits_for_them():
    """The range flag's word goes to the next call, so nothing that may write it can be left on the stream, also where the
    call reports a launch error (here one that an earlier HIP call of this thread left behind)."""
    import ctypes
    import fp6_marlin
    lib = fp6_marlin.cabi.lib                                         # (its handle also finds the HIP runtime that it is linked to)
    w = (torch.randn((4096, 2048), device=dev()) * 0.02).half()
    want = fp6_marlin.pack_mixed_weight(w, 256, 128, harness_layout=False)
    a = torch.randn((8192, 8192), device=dev())
    torch.cuda.synchronize()
    for _ in range(4):
        a @ a                                                         # (tens of milliseconds in front of the packer's kernels)
    assert lib.hipSetDevice(ctypes.c_int(10000)) != 0                 # no such device: the error stays with the thread
    if lib.hipPeekAtLastError() == 0:
        pytest.skip("this runtime does not keep the error of an earlier call")
    with pytest.raises(RuntimeError):
        fp6_marlin.cabi.pack_mixed_weight_device(w, 256, 128, False)
    assert torch.cuda.current_stream().query()
    got = fp6_marlin.pack_mixed_weight(w, 256, 128, harness_layout=False)
    assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_packing_fp6_columns_is_refused_under_capture():
    """The call waits for its kernels, which a capture forbids; it says so, keeps no flag, and the capture goes on.  More
    often than there are flags."""
    import fp6_marlin
    w = (torch.randn((256, 512), device=dev()) * 0.02).half()
    want = fp6_marlin.pack_mixed_weight(w, 256, 128, harness_layout=False)
    out = torch.zeros(4, device=dev())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(70):
            with pytest.raises(RuntimeError):
                fp6_marlin.cabi.pack_mixed_weight_device(w, 256, 128, False)
        out.add_(1.0)
    for i in range(3):
        graph.replay()
        got = fp6_marlin.pack_mixed_weight(w, 256, 128, harness_layout=False)
        assert all(torch.equal(x, y) for x, y in zip(got, want)) and out.tolist() == [i + 1.0] * 4


@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
def test_range_errors_of_the_true_transpose(value):
    """Layer.pack's layout has an FP6 kernel of its own: a NaN or infinite weight in that region is a range error there too,
    wherever it lies, and the call after it is clean."""
    import fp6_marlin
    g = torch.Generator().manual_seed(17)
    w = (torch.randn((1024, 384), generator=g) * 0.02).half().to(dev())
    want = fp6_marlin.pack_mixed_weight(w, 192, 128, harness_layout=False)
    for row, col in ((0, 192), (511, 383), (512, 250), (1023, 200)):
        bad = w.clone()
        bad[row, col] = value
        with pytest.raises(ValueError):
            fp6_marlin.pack_mixed_weight(bad, 192, 128, harness_layout=False)
        got = fp6_marlin.pack_mixed_weight(w, 192, 128, harness_layout=False)
        assert all(torch.equal(x, y) for x, y in zip(got, want)), (row, col)


def entry_outputs(k, n, qc):
    """B, s, w_ref for the C entries, per-column scales."""
    return [torch.empty(size, dtype=dtype, device=dev()) for size, dtype in
            ((k * (n - qc) // 8 + k * qc * 3 // 16, torch.int32), (n, torch.half), ((k, n), torch.half))]


def entry(name, w, qc, out, stream):
    import ctypes
    import fp6_marlin
    return getattr(fp6_marlin.cabi.lib, name)(w.data_ptr(), w.shape[0], w.shape[1], qc, -1, 0, *(ctypes.c_void_p(t.data_ptr()) for t in out),
                                              0, ctypes.c_void_p(stream.cuda_stream))


@pytest.mark.parametrize("harness", [True, False])
@pytest.mark.parametrize("own", [False, True])
def test_packed_weights_are_ready_for_every_stream_when_the_call_returns(own, harness):
    """On the default stream as on one of the caller's own: torch's streams are not ordered against the default one, so a
    `mul` on another stream and a copy that refills the source may follow without an event."""
    import fp6_marlin
    k, n, qc, gs = 4096, 8192, 256, 128
    g = torch.Generator().manual_seed(37)
    staged = (torch.randn((k, n), generator=g) * 0.02).half()
    A = torch.randn((16, k), generator=g).half().to(dev())
    big = torch.randn((4096, 4096), device=dev()).half()
    want = fp6_marlin.pack_mixed_weight(staged.to(dev()), qc, gs, harness_layout=harness)
    ws = torch.zeros(n // 128 * 16, dtype=torch.int32, device=dev())
    C = torch.empty((16, n), dtype=torch.half, device=dev())
    fp6_marlin.mul(A, want[0], C, want[1], ws, qc, group_size=gs)
    torch.cuda.synchronize()
    other = torch.cuda.Stream()
    for busy in (0, 30):                               # (alone, and with more work in front than a short poll outlasts)
        w = staged.to(dev())
        nan = torch.full_like(w, float("nan"))
        C1 = torch.full_like(C, float("nan"))
        torch.cuda.synchronize()
        stream = torch.cuda.Stream() if own else torch.cuda.default_stream()
        with torch.cuda.stream(stream):
            for _ in range(busy):
                big @ big
            got = fp6_marlin.pack_mixed_weight(w, qc, gs, harness_layout=harness)
            assert stream.query()
        with torch.cuda.stream(other):
            w.copy_(nan)
            fp6_marlin.mul(A, got[0], C1, got[1], ws, qc, group_size=gs)
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got, want)) and torch.equal(C, C1)


@pytest.mark.parametrize("k,n,qc", [(64, 128, 64), (1024, 384, 192), (4160, 1088, 1088)])
@pytest.mark.parametrize("own", [False, True])
def test_the_entry_that_leaves_the_packing_to_the_stream(own, k, n, qc):
    """fp6m_pack_mixed_device_async on either kind of stream, alone and with other work in front (longer than it polls): its
    results in stream order, and for another stream after an event, with the source's memory used again in stream order in
    between; a weight out of range is still an error by value, with nothing left on the stream."""
    import fp6_marlin
    g = torch.Generator().manual_seed(31)
    w = (torch.randn((k, n), generator=g) * 0.02).half().to(dev())
    bad = w.clone()
    bad[k - 1, n - 1] = float("inf")
    want = entry_outputs(k, n, qc)
    assert entry("fp6m_pack_mixed_device", w, qc, want, torch.cuda.default_stream()) == 0
    big = torch.randn((4096, 4096), device=dev()).half()
    torch.cuda.synchronize()
    stream, other = torch.cuda.Stream() if own else torch.cuda.default_stream(), torch.cuda.Stream()
    for busy in (0, 30):
        out = entry_outputs(k, n, qc)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            mine = w.clone()
            for _ in range(busy):
                big @ big
            assert entry("fp6m_pack_mixed_device_async", mine, qc, out, stream) == 0
            del mine
            torch.full((k, n), float("nan"), dtype=torch.half, device=dev())
            copies = [t.clone() for t in out]
            ready = stream.record_event()
        with torch.cuda.stream(other):
            other.wait_event(ready)
            late = [t.clone() for t in out]
        torch.cuda.synchronize()
        for got in (out, copies, late):
            assert all(torch.equal(x, y) for x, y in zip(got, want))
        with torch.cuda.stream(stream):
            for _ in range(busy):
                big @ big
            assert entry("fp6m_pack_mixed_device_async", bad, qc, out, stream) == fp6_marlin.cabi.ERR_RANGE
            assert stream.query()


def test_the_entry_that_leaves_the_packing_to_the_stream_returns_before_it_is_done():
    """Half a millisecond of packing is still running when the call returns."""
    k, n, qc = 8192, 28672, 256
    w = torch.randn((k, n), dtype=torch.half, device=dev()).mul_(0.02)
    out, want = entry_outputs(k, n, qc), entry_outputs(k, n, qc)
    stream = torch.cuda.default_stream()
    assert entry("fp6m_pack_mixed_device", w, qc, want, stream) == 0
    assert stream.query()
    early = 0
    for _ in range(5):                                 # (a host thread that is descheduled in between would see it done)
        assert entry("fp6m_pack_mixed_device_async", w, qc, out, stream) == 0
        early += not stream.query()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(out, want))
    assert early >= 1


def test_fp6_columns_with_sub_normal_scales():
    """Columns down to the smallest binary16 values: their scales are rounded to few bits, half way cases among them (a maximum
    of 70 * 2^-24 was scaled by 3 units instead of 2), so that quotients reach beyond 28 (clamped) and fall below 0.0625 (a
    zero, without its sign), and at last the scale is zero and replaced by one."""
    import fp6_marlin
    g = torch.Generator().manual_seed(23)
    w = torch.randn((576, 320), generator=g) * 0.02
    w[:, 128:] *= 2.0 ** -(torch.arange(192) % 24).float()
    w = w.half()
    for col, units in ((128, 14), (129, 42), (130, 70), (131, 126), (132, 14 * 63)):   # (exactly half way between two scales)
        w[:, col] = torch.randint(-units, units + 1, (576,), generator=g).float().mul(2.0 ** -24).half()
        w[0, col] = units * 2.0 ** -24
    for gs in (-1, 64):
        Bh, sh, rh = fp6_marlin.pack_mixed_weight(w, 192, gs, harness_layout=False)
        Bd, sd, rd = fp6_marlin.pack_mixed_weight(w.to(dev()), 192, gs, harness_layout=False)
        assert torch.equal(Bd.cpu(), Bh)
        assert same_bits(sd, sh)
        assert same_values(rd, rh)


@pytest.mark.parametrize("gs", [-1, 128, 64])
def test_infinite_and_nan_weights_in_the_int4_region(gs):
    """They are no error there.  Scales and check weight are the host path's, with a NaN where it has one, and so are the words,
    but for the finite weights of a group with an infinite scale: their code is 8 where the host, which packs the
    re-quantised check weight (a NaN there), has 0."""
    import fp6_marlin
    g = torch.Generator().manual_seed(29)
    k, n = 256, 512
    w = (torch.randn((k, n), generator=g) * 0.02).half()
    for col, values in ((3, ["inf"]), (70, ["-inf"]), (131, ["nan"]), (200, ["inf", "-inf"]), (255, ["nan", "inf"]), (301, ["-inf", "nan"])):
        for i, v in enumerate(values):
            w[10 + 100 * i, col] = float(v)
    w[:, 400] = float("inf")
    w[:, 401] = float("nan")
    same = lambda a, b: np.array_equal(a.cpu().numpy().astype(np.float32), b.cpu().numpy().astype(np.float32), equal_nan=True)
    Bh, sh, rh = fp6_marlin.pack_mixed_weight(w, -1, gs, harness_layout=False)
    Bd, sd, rd = fp6_marlin.pack_mixed_weight(w.to(dev()), -1, gs, harness_layout=False)
    assert same(sd, sh)
    assert same(rd, rh)
    ones = torch.ones(n, dtype=torch.half)                            # (the words alone: code - 8, with per-column scales of one)
    got, host = (fp6_marlin.unpack_to_fp16(B.cpu(), ones, k, n, -1, -1) for B in (Bd, Bh))
    most = w.abs().float().reshape(k // (k if gs == -1 else gs), -1, n).amax(1, keepdim=True)
    infinite = (most.isinf() & w.isfinite().reshape(most.shape[0], -1, n)).reshape(k, n)
    assert bool((host[infinite] == -8).all()) and bool((got[infinite] == 0).all()) and int(infinite.sum()) > 300
    assert torch.equal(got[~infinite], host[~infinite])


def test_fp6_scale_rule_vectors_through_the_gpu_packer():
    """The constructed columns of tests/fp6_scale_vectors.py (exact scales 1, 0.5, 0.0625; values around every e3m2
    grid point; entries below the 0.0625 threshold; a quotient that rounds above 28) through the on-GPU packer: scales
    and check weight against the independent numpy evaluation, words against the host packer."""
    import fp6_marlin
    import fp6_scale_vectors as fv
    import kernel_rules as kr
    w = fv.vectors()
    k, n = w.shape
    s_want, ref_want = fv.expected(w)
    # (the harness layout reads the flat [k, n] buffer as [n, k] without transposing; with k == n that is the transpose)
    wt = torch.from_numpy(np.ascontiguousarray(w.T))
    Bd, sd, rd = fp6_marlin.pack_mixed_weight(wt.to(dev()), n, -1, harness_layout=True)
    Bh, sh, rh = fp6_marlin.pack_mixed_weight(wt, n, -1, harness_layout=True)
    assert torch.equal(Bd.cpu(), Bh) and same_bits(sd, sh) and same_values(rd, rh)
    Bd, sd, rd = fp6_marlin.pack_mixed_weight(torch.from_numpy(w).to(dev()), n, -1, harness_layout=False)
    s_perm = sd.cpu().numpy()
    s_nat = np.array([s_perm[32 * (c // 32) + kr.scale_slot(c % 32)] for c in range(n)], dtype=np.float16)
    assert np.array_equal(s_nat.view(np.uint16), s_want.view(np.uint16))
    assert np.array_equal(rd.cpu().numpy().astype(np.float32), ref_want.astype(np.float32))


def test_layer_pack_on_gpu_matches_cpu_and_runs():
    import fp6_marlin
    torch.manual_seed(3)
    lin = torch.nn.Linear(512, 768, bias=False).half()
    a = fp6_marlin.Layer(512, 768, groupsize=128, quant_cols=256)
    ref_cpu = a.pack(lin)
    b = fp6_marlin.Layer(512, 768, groupsize=128, quant_cols=256).to(dev())
    ref_gpu = b.pack(lin.to(dev()))
    assert torch.equal(b.B.cpu(), a.B) and same_bits(b.s, a.s) and same_values(ref_gpu, ref_cpu)
    x = torch.randn((4, 512), dtype=torch.half, device=dev())
    y = b(x)
    y_ref = x.float() @ ref_gpu.float()
    assert ((y.float() - y_ref).abs().mean() / y_ref.abs().mean()).item() <= 1e-3
