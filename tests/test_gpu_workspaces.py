"""Workspaces smaller than the default: what they have room for is what the call does with."""
import pytest
import torch

from slowrun_amd import _lib, configs

pytestmark = pytest.mark.gpu


def _with_sizes(monkeypatch, **bytes_):
    """ce_forward / ce_backward allocate what sizes_for says: this says something else."""
    real = _lib.sizes_for

    def sizes_for(*a):
        s = real(*a)
        for k, v in bytes_.items():
            setattr(s, k, v)
        return s
    monkeypatch.setattr(_lib, "sizes_for", sizes_for)


@pytest.mark.parametrize("bf16,keep", [(True, False), (False, False), (False, True)])
@pytest.mark.parametrize("N,d,V", [(1, 16, 5000), (61, 272, 33000), (256, 64, 70000), (300, 128, 1000), (1000, 256, 4096), (2048, 128, 50304), (3840, 64, 9000)])
def test_forward_of_few_rows_takes_the_splits_that_fit(monkeypatch, N, d, V, bf16, keep):
    """A forward of fewer than 16 row tiles cuts the vocabulary as fine as there are CUs; its default workspace holds that many
    records.  One with room for 16 splits' or 8 gives the same maxima and losses, up to the order of the row sums (at most V positive fp32 terms)."""
    from slowrun_amd import cuda_kernels as ck
    inp = configs.make_inputs("tiny_track", N=N, d=d, V=V)
    x, w, y = inp.x.cuda().bfloat16(), inp.w.cuda().bfloat16(), inp.targets.cuda()

    def call():
        out, _saved, lse, argmax, n_valid = ck.ce_forward(x, w, y, inp.x_s, inp.w_s, 15.0, "none", want_argmax=True, keep_dlogits=keep,
                                                          operand_dtype=torch.bfloat16 if bf16 else None)
        return out, lse, argmax, n_valid
    want = call()
    Np = -(-N // 256) * 256
    for room in (16 * 16 * Np + 256, 16 * 16 * Np):
        _with_sizes(monkeypatch, fwd_workspace_bytes=room)
        got = call()
        assert torch.equal(got[2], want[2]) and torch.equal(got[3], want[3])
        assert torch.allclose(got[0], want[0], rtol=2e-6, atol=2e-5) and torch.allclose(got[1], want[1], rtol=2e-6, atol=2e-5)
        monkeypatch.undo()
    _with_sizes(monkeypatch, fwd_workspace_bytes=16 * Np * min(8, -(-V // 256)) - 1)      # not even that: refused
    with pytest.raises(RuntimeError, match="too small"):
        call()


@pytest.mark.parametrize("N,offsets,d,V", [(257, 1, 272, 300), (700, 2, 64, 1003), (2000, 4, 256, 4096), (5000, 1, 16, 130)])
def test_backward_in_the_least_workspace(N, offsets, d, V):
    """The least that backward accepts gives the gradients of the default workspace, bit for bit with the dlogits kept (the same
    launches but for a K-split last round of dW: fp32 sums in another order, 2^-20 of the largest element), up to the same order with them formed again.  Columns
    of fewer than 8, of 8 to 15 and of more entries are there: where dW takes several launches the line lies at 16."""
    from slowrun_amd import cuda_kernels as ck
    inp = configs.make_inputs("tiny_track", N=N, d=d, V=V)
    gen = torch.Generator().manual_seed(N)
    y = (torch.rand(N, generator=gen) ** 3 * V).long().clamp_(max=V - 1)
    y[: N // 8] = torch.arange(N // 8) // 12 % V              # runs of 12
    y = y.cuda()
    x, w = inp.x.cuda().bfloat16(), inp.w.cuda().bfloat16()
    mw = torch.tensor([1.0, 0.5, 0.25, 0.125][:offsets], device="cuda") if offsets > 1 else None
    go = torch.rand(N, generator=gen).cuda() / N
    sz = _lib.sizes_for(N, d, V, offsets)
    for keep, least, default in ((True, None, sz.bwd_workspace_kept_bytes), (False, sz.bwd_workspace_min_bytes, sz.bwd_workspace_bytes)):
        _out, saved, *_ = ck.ce_forward(x, w, y, inp.x_s, inp.w_s, 15.0, "none", mtp_weights=mw, keep_dlogits=keep)

        def call(nbytes):
            return ck.ce_backward(saved, y, go, N, d, V, inp.x_s, inp.w_s, 15.0, 1.0, "none", torch.float32, torch.float32, mtp_weights=mw, keep_dlogits=keep,
                                  workspace_bytes=nbytes)
        if keep:                                              # the kept mode's least is not in the sizes: what the refusal names
            with pytest.raises(RuntimeError, match="workspace too small") as e:
                call(256)
            least = int(str(e.value).split("<")[1].split()[0].strip(")."))
        want, got = call(default), call(least)
        for a, b in zip(want, got):
            assert float((a - b).abs().max()) <= 2.0 ** -20 * float(a.abs().max()) + 1e-30
        with pytest.raises(RuntimeError, match="too small"):
            call(least - 1)


@pytest.mark.parametrize("N", [130001, 131073])
def test_one_launch_of_dw_up_to_131072_rows(N):
    """Rows between the last whole dX panel below 131072 (128000 at d = 2560) and 131072, dlogits kept: one launch, no partial of dW in the
    workspace; one row more: two launches.  Values that e4m3 holds exactly, so that only the dlogits are rounded: against fp32, 1e-2 of the norm as for every 8-bit dlogits."""
    from slowrun_amd import cuda_kernels as ck
    d, V = 2560, 300
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randint(-2, 3, (N, d), device="cuda", generator=gen).bfloat16()
    w = (torch.randint(-2, 3, (d, V), device="cuda", generator=gen) / 64).bfloat16()
    y = torch.randint(0, V, (N,), device="cuda", generator=gen)
    _out, saved, *_ = ck.ce_forward(x, w, y, 1.0, 1.0 / 64, 15.0, "mean", keep_dlogits=True)
    dx, dw = ck.ce_backward(saved, y, torch.ones((), device="cuda"), N, d, V, 1.0, 1.0 / 64, 15.0, 1.0, "mean", torch.float32, torch.float32, keep_dlogits=True)
    xf, wf = x.float().requires_grad_(True), w.float().requires_grad_(True)
    torch.nn.functional.cross_entropy(15.0 * torch.tanh(xf @ wf / 15.0), y).backward()
    assert float((dw - wf.grad).norm() / wf.grad.norm()) < 1e-2
    assert float((dx - xf.grad).norm() / xf.grad.norm()) < 4e-2      # (a row's 300 dlogits: their e4m3 rounding, 2^-4 / sqrt(3) of each at most)


@pytest.mark.parametrize("bf16,keep", [(True, False), (False, False), (False, True)])
@pytest.mark.parametrize("N,offsets,d,V", [(1, 1, 16, 264), (61, 1, 272, 33000), (129, 2, 96, 33000), (300, 3, 1040, 4096), (1100, 1, 528, 263), (4200, 2, 256, 2056)])
def test_nothing_depends_on_what_the_buffers_held(monkeypatch, N, offsets, d, V, bf16, keep):
    """State and workspaces full of ones (NaN as floats, -1 as indices) or of zeros before the calls: the same bits after them."""
    from slowrun_amd import cuda_kernels as ck
    inp = configs.make_inputs("tiny_track", N=N, d=d, V=V)
    x, w, y = inp.x.cuda().bfloat16(), inp.w.cuda().bfloat16(), inp.targets.cuda()
    y[::5] = -1
    mw = torch.tensor([1.0, 0.5, 0.25, 0.125][:offsets], device="cuda") if offsets > 1 else None
    go = torch.rand(N, generator=torch.Generator().manual_seed(N)).cuda() / N
    real, res = torch.empty, []
    for fill in (0, 255):
        def empty(*a, **k):
            t = real(*a, **k)
            if t.is_cuda:
                t.view(torch.uint8).fill_(fill) if t.dtype == torch.uint8 else t.fill_(float("nan") if fill and t.is_floating_point() else 0)
            return t
        monkeypatch.setattr(torch, "empty", empty)
        out, saved, lse, argmax, n_valid = ck.ce_forward(x, w, y, inp.x_s, inp.w_s, 15.0, "none", want_argmax=True, mtp_weights=mw, keep_dlogits=keep,
                                                         operand_dtype=torch.bfloat16 if bf16 else None)
        grads = () if bf16 else ck.ce_backward(saved, y, go, N, d, V, inp.x_s, inp.w_s, 15.0, 1.0, "none", torch.bfloat16, torch.float32, mtp_weights=mw,
                                               keep_dlogits=keep)
        monkeypatch.undo()
        res.append((out, lse, argmax, n_valid, *grads))
    for a, b in zip(*res):
        assert torch.equal(a, b) and bool(torch.isfinite(a.float()).all())
