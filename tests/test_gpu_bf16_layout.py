"""The layout kernels of the bf16 operands at the edges of their vector paths: the same values read through aligned rows
(16-byte loads) and through rows that are not (element by element) have to give the same bits, and both the loss of a plain
fp32 evaluation of the bf16 head.  Bound: a logit on the other side of a bf16 rounding moves by 2^-8 of itself (|u| < 8 here)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,d,V", [(1, 16, 7), (5, 112, 130), (61, 144, 1002), (257, 128, 256), (300, 256, 515)])
def test_aligned_and_unaligned_rows_give_the_same_loss(dtype, N, d, V):
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(N)
    Va, da = (V + 7) // 8 * 8, d
    x = torch.randn(N, d, device="cuda", generator=gen).to(dtype)
    w = (torch.randn(d, V, device="cuda", generator=gen) * d ** -0.5).to(dtype)
    y = torch.randint(0, V, (N,), device="cuda", generator=gen)
    losses = []
    for wpad, xpad, off in ((Va - V, 0, 0), (Va - V + 1, 1, 0), (Va - V + 8, 8, 1)):       # rows aligned; an odd stride; an odd base
        wb = torch.full((d, V + wpad), 100.0, device="cuda", dtype=dtype)
        xb = torch.full((N, da + xpad), 100.0, device="cuda", dtype=dtype)
        wv, xv = wb[:, off: off + V] if off + V <= V + wpad else wb[:, :V], xb[:, off: off + d] if xpad else xb
        wv.copy_(w); xv.copy_(x)
        losses.append(ck.softcapped_cross_entropy(xv, wv, y, reduction="none", operand_dtype=torch.bfloat16))
    assert torch.equal(losses[0], losses[1]) and torch.equal(losses[0], losses[2])
    u = (x.bfloat16().float() @ w.bfloat16().float()).bfloat16().float()
    ref = F.cross_entropy(15.0 * torch.tanh(u / 15.0), y, reduction="none")
    assert float((losses[0] - ref).abs().max()) < 8 * 2 ** -8
    assert float((losses[0] - ref).abs().mean()) < 2e-3


@pytest.mark.parametrize("xdtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,d,V,vocab,offsets", [(1, 16, 8, 8, 1), (31, 48, 248, 241, 1), (64, 64, 256, 256, 2), (65, 272, 264, 257, 4), (128, 1040, 3000, 2999, 1),
                                                 (129, 96, 33000, 32990, 3), (256, 528, 32776, 32776, 1), (61, 32, 131072, 131072, 1), (200, 16, 70000, 69999, 1)])
def test_few_rows_against_the_general_path(xdtype, N, d, V, vocab, offsets):
    """Few rows (up to 128, or 256 of a large vocabulary) of aligned bf16 weights are read as they lie; the same weights in rows of odd length take the general path.
    Small whole numbers make every logit exact, whatever the order of its sum: the maximum's column is the same, and the
    losses differ by the order of the row sums (fp32 sums of at most V positive terms)."""
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(V + N)
    x = torch.randint(-2, 3, (N, d), device="cuda", generator=gen).to(xdtype) / 4
    w = torch.randint(-2, 3, (d, V), device="cuda", generator=gen).bfloat16() / 4
    y = torch.randint(0, vocab, (N,), device="cuda", generator=gen)
    y[::5] = -1
    odd = torch.zeros(d, V + 1, device="cuda", dtype=torch.bfloat16)
    odd[:, :V] = w
    mtp = torch.tensor([1.0, 0.5, 0.25, 0.125][:offsets], device="cuda")
    got = [ck.ce_forward(x, m, y, 1.0, 1.0, 15.0, "none", want_argmax=True, mtp_weights=mtp, vocab_size=vocab, operand_dtype=torch.bfloat16)
           for m in (w, odd[:, :V])]
    (l0, _, lse0, am0, nv0), (l1, _, lse1, am1, nv1) = got
    assert torch.equal(am0, am1) and torch.equal(nv0, nv1)
    assert torch.allclose(lse0, lse1, rtol=2e-6, atol=2e-5) and torch.allclose(l0, l1, rtol=2e-6, atol=2e-5)
    if offsets == 1:
        u = (x.float() @ w.float())[:, :vocab].bfloat16().float()
        ref = F.cross_entropy(15.0 * torch.tanh(u / 15.0), y, reduction="none", ignore_index=-1)
        assert torch.allclose(l0, ref, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("N,d,V", [(64, 8208, 264), (65, 8192, 264), (128, 8208, 1792), (128, 8208, 1800)])
def test_deep_contractions_of_few_column_tiles(N, d, V):
    """The lines in d and in column tiles at which 65 to 128 rows change their way: exact logits, as above."""
    test_few_rows_against_the_general_path(torch.bfloat16, N, d, V, V, 1)


@pytest.mark.parametrize("n,shape", [(1, (1,)), (255, (255,)), (257, (257,)), (4098, (2, 2049))])
def test_target_probability_is_the_exponential_of_the_losses(n, shape):
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(*shape, 32, device="cuda", generator=gen).bfloat16()
    w = torch.randn(32, 200, device="cuda", generator=gen).bfloat16()
    y = torch.randint(0, 200, (2 * n,), device="cuda", generator=gen)[::2].reshape(shape)      # (strided where it is one row)
    y.view(-1)[::7] = -1 if n > 1 else 3
    p = ck.target_probability(x, w, y, operand_dtype=torch.bfloat16)
    losses = ck.softcapped_cross_entropy(x, w, y, reduction="none", operand_dtype=torch.bfloat16)
    assert p.shape == losses.shape and torch.allclose(p, torch.where(y == -1, torch.zeros_like(losses), torch.exp(-losses)), rtol=1e-6, atol=0)


@pytest.mark.parametrize("operands", ["bf16", "e4m3"])
@pytest.mark.parametrize("N", [1, 61, 300, 16640])
def test_both_entry_points_give_the_same_probabilities(operands, N):
    """sce_forward_probability, which target_probability calls, and sce_target_probability of the losses of a call of its own: the same bits."""
    from slowrun_amd import _lib, cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(N, 64, device="cuda", generator=gen).bfloat16()
    w = (torch.randn(64, 264, device="cuda", generator=gen) / 8).bfloat16()
    y = torch.randint(0, 264, (N,), device="cuda", generator=gen)
    y[::7], y[N // 2] = -1, 264 if N > 1 else 5                 # (a target out of range: NaN, or whatever its loss gives)
    ops = dict(operand_dtype=torch.bfloat16) if operands == "bf16" else dict(x_s=0.02, w_s=0.002)
    losses = ck.softcapped_cross_entropy(x, w, y, reduction="none", **ops)
    got = torch.full((N,), -1.0, device="cuda")
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    assert lib.sce_target_probability(losses.data_ptr(), y.data_ptr(), N, -1, got.data_ptr(), 0, stream) == 0
    want = ck.target_probability(x, w, y, **ops)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32)) and bool((got[y == -1] == 0).all()) and bool((got[(y >= 0) & (y < 264)] > 0).all())


@pytest.mark.parametrize("N,d,V", [(3, 48, 264), (64, 64, 2056), (128, 96, 520), (200, 32, 33000)])
def test_infinities_and_nan_of_few_rows_as_in_the_general_path(N, d, V):
    """Rows with an infinity, a NaN, a largest finite value, and a column of W with each: the few-rows kernel gives what the general
    path gives -- the same maxima, the same infinities and NaN, and the same losses elsewhere (row sums in another order)."""
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(V)
    inf, big = float("inf"), float(torch.finfo(torch.bfloat16).max)
    for case in ("rows", "columns"):
        x = torch.randint(-2, 3, (N, d), device="cuda", generator=gen).bfloat16() / 4
        w = torch.randint(-2, 3, (d, V), device="cuda", generator=gen).bfloat16() / 4
        if case == "rows":
            for i, v in enumerate((inf, -inf, float("nan"), big)):
                x[i * 7 % N, i] = v
        else:
            for i, v in enumerate((inf, -inf, float("nan"), big)):
                w[i, (i * 61 + 5) % V] = v
        y = torch.randint(0, V, (N,), device="cuda", generator=gen)
        y[0], y[N // 2] = 5, 66
        odd = torch.zeros(d, V + 1, device="cuda", dtype=torch.bfloat16)
        odd[:, :V] = w
        got = [ck.ce_forward(x, m, y, 1.0, 1.0, 15.0, "none", want_argmax=True, operand_dtype=torch.bfloat16) for m in (w, odd[:, :V])]
        (l0, _, lse0, am0, nv0), (l1, _, lse1, am1, nv1) = got
        assert torch.equal(am0, am1) and torch.equal(nv0, nv1)
        assert torch.allclose(lse0, lse1, rtol=2e-6, atol=2e-5, equal_nan=True) and torch.allclose(l0, l1, rtol=2e-6, atol=2e-5, equal_nan=True)


@pytest.mark.parametrize("N,d,V", [(61, 272, 33000), (200, 96, 33000)])
def test_scoring_captured_in_a_hip_graph(N, d, V):
    """The scoring call captured once and replayed on new rows, weights and targets: each replay the bits of the direct call."""
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(N, d, device="cuda", generator=gen).bfloat16()
    w = (torch.randn(d, V, device="cuda", generator=gen) * d ** -0.5).bfloat16()
    y = torch.randint(0, V, (N,), device="cuda", generator=gen)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ck.target_probability(x, w, y, operand_dtype=torch.bfloat16)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = ck.target_probability(x, w, y, operand_dtype=torch.bfloat16)
    for trial in range(4):
        x.copy_(torch.randn(N, d, device="cuda", generator=gen).bfloat16())
        w.mul_(1.25)
        y.copy_(torch.randint(0, V, (N,), device="cuda", generator=gen))
        y[trial::5] = -1
        graph.replay()
        torch.cuda.synchronize()
        got = captured.clone()
        want = ck.target_probability(x, w, y, operand_dtype=torch.bfloat16)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and bool((got[y != -1] > 0).all()) and bool((got[y == -1] == 0).all())
