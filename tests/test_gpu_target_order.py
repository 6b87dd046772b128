"""The rows grouped by target: up to 4096 (offset, row) entries are ranked in one launch, more go through the radix sort.  A
batch just below that limit and the same batch with ignored rows behind it (no gradient of their own, past the limit) have
the same gradients: dX row by row, dW up to the order of its fp32 sums over the rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("N,offsets,d,V", [(4096, 1, 64, 300), (2048, 2, 272, 5000), (1365, 3, 128, 40000), (1024, 4, 16, 3)])
def test_ranked_and_sorted_targets_give_the_same_gradients(N, offsets, d, V, keep):
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(V)
    more = 4096 // offsets + 40
    x = torch.randn(more, d, device="cuda", generator=gen)
    w = torch.randn(d, V, device="cuda", generator=gen) * d ** -0.5
    y = (torch.rand(more, device="cuda", generator=gen) ** 3 * V).long()          # some columns hit by many rows, most by few
    y[torch.rand(more, device="cuda", generator=gen) < 0.1] = -1
    y[N:] = -1
    mtp = torch.tensor([1.0, 0.5, 0.25, 0.125][:offsets], device="cuda")
    got = []
    for n in (N, more):
        loss, saved, *_ = ck.ce_forward(x[:n], w, y[:n], 0.02, 0.01, 15.0, "none", mtp_weights=mtp, keep_dlogits=keep)
        go = torch.rand(more, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))[:n]
        dx, dw = ck.ce_backward(saved, y[:n], go, n, d, V, 0.02, 0.01, 15.0, 1.0, "none", torch.float32, torch.float32, mtp_weights=mtp, keep_dlogits=keep)
        got.append((loss[:N], dx[:N], dw))
    for a, b in zip(got[0], got[1]):
        assert float((a - b).norm() / b.norm()) < 2e-5


@pytest.mark.parametrize("N,offsets,V", [(1, 1, 5), (15, 4, 3), (65, 2, 1000)])
def test_one_hot_part_of_dw_of_few_entries(N, offsets, V):
    """x = 0: every logit is 0, p = 1 / V, and what is left of dW is zero too; with x = e_0 in row i only, row 0 of dW is the
    row's (p - onehot), summed here in fp64."""
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(N)
    d = 16
    x = torch.zeros(N, d, device="cuda")
    x[:, 0] = 1.0
    w = torch.zeros(d, V, device="cuda")
    y = torch.randint(0, V, (N,), device="cuda", generator=gen)
    mtp = torch.tensor([1.0, 0.5, 0.25, 0.125][:offsets], device="cuda")
    loss, saved, *_ = ck.ce_forward(x, w, y, 1.0, 1.0, 15.0, "none", mtp_weights=mtp, keep_dlogits=True)
    dx, dw = ck.ce_backward(saved, y, torch.ones(N, device="cuda"), N, d, V, 1.0, 1.0, 15.0, 1.0, "none", torch.float32, torch.float32, mtp_weights=mtp, keep_dlogits=True)
    ref = torch.zeros(V, dtype=torch.float64)
    for i in range(N):
        for k in range(offsets):
            if i + k < N:
                ref += float(mtp[k]) / V
                ref[int(y[i + k])] -= float(mtp[k])
    # the softmax part goes through e4m3 (3 bits of mantissa: half a unit is 2^-4 of it), the one-hot part does not
    soft = float(mtp.sum()) * N / V
    assert float((dw[0].double().cpu() - ref).abs().max()) <= soft * 2 ** -4 + 1e-5
    assert float(dw[1:].abs().max()) == 0.0


@pytest.mark.parametrize("N,offsets,V", [(513, 1, 256), (5000, 2, 512), (3000, 2, 64), (40000, 1, 1024)])
def test_one_hot_part_of_dw_of_more_entries_than_columns(N, offsets, V):
    """A small vocabulary with many entries: workgroups beyond those of the columns bring the entries' rows and coefficients.  With
    x = e_0, a zero head and powers of two for V and for the row's weight, p = 1 / V is exact in e4m3 (dlogits formed again in
    backward are stored as the probability), so row 0 of dW is sum_i sum_k (1 / V - onehot) up to the fp32 sums: 2^-20 of the N additions that a column sees."""
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(N)
    d = 16
    x = torch.zeros(N, d, device="cuda")
    x[:, 0] = 1.0
    w = torch.zeros(d, V, device="cuda")
    y = torch.randint(0, V, (N,), device="cuda", generator=gen)
    y[::9] = V // 2                        # one column in chunks
    mtp = torch.ones(offsets, device="cuda")
    loss, saved, *_ = ck.ce_forward(x, w, y, 1.0, 1.0, 15.0, "none", mtp_weights=mtp, keep_dlogits=False)
    dx, dw = ck.ce_backward(saved, y, torch.ones(N, device="cuda"), N, d, V, 1.0, 1.0, 15.0, 1.0, "none", torch.float32, torch.float32, mtp_weights=mtp, keep_dlogits=False)
    count = sum(torch.bincount(y[k:], minlength=V).double() for k in range(offsets))
    ref = float(sum(N - k for k in range(offsets))) / V - count
    assert float((dw[0].double() - ref).abs().max()) <= 2.0 ** -20 * N * offsets
    assert float(dw[1:].abs().max()) == 0.0


@pytest.mark.parametrize("panel_rows", [0, 256])
@pytest.mark.parametrize("N,offsets,d,V", [(257, 1, 16, 64), (3000, 1, 272, 256), (9000, 2, 64, 512), (2000, 1, 4352, 256), (1100, 2, 8448, 64), (70000, 1, 32, 1024)])
def test_columns_of_many_rows(N, offsets, d, V, panel_rows):
    """Columns that are the target of hundreds to tens of thousands of rows: the sums of their chunks are added up before dW is
    stored, in the grid that finishes a K-split dX or by themselves, for one launch of dW and for several.  Whole numbers in x
    and a zero head: every product and sum is exact, and dW is sum_i x_i (1 / V - onehot), to the last fp32 rounding of each step."""
    from slowrun_amd import _lib
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randint(-2, 3, (N, d), device="cuda", generator=gen).float()
    w = torch.zeros(d, V, device="cuda")
    y = torch.randint(0, V, (N,), device="cuda", generator=gen)
    r = torch.rand(N, device="cuda", generator=gen)
    y[r < 0.6], y[r < 0.2] = V - 1, 5
    y[::11] = -1
    mtp = torch.ones(offsets, device="cuda")
    _out, saved, *_ = ck.ce_forward(x, w, y, 1.0, 1.0, 15.0, "none", mtp_weights=mtp, keep_dlogits=False)
    args = (saved, y, torch.ones(N, device="cuda"), N, d, V, 1.0, 1.0, 15.0, 1.0, "none", torch.float32, torch.float32)
    nbytes = _lib.sizes_for(N, d, V, offsets).bwd_workspace_min_bytes if panel_rows else None
    first = None
    for _ in range(3):                     # (the same bits every time)
        dx, dw = ck.ce_backward(*args, mtp_weights=mtp, panel_rows=panel_rows, workspace_bytes=nbytes)
        assert first is None or torch.equal(dw, first)
        first = dw
    ref = torch.zeros(d, V, dtype=torch.float64, device="cuda")
    xd = x.double()
    for k in range(offsets):
        ok = torch.arange(N - k, device="cuda")[y[k:] >= 0]
        ref += xd[ok].sum(0)[:, None] / V
        ref.index_add_(1, y[k:][ok], -xd[ok].t().contiguous())
    # 2 |x| N offsets bounds what any partial sum reaches; a handful of roundings of it at 2^-24
    assert float((dw.double() - ref).abs().max()) <= 2.0 ** -20 * 2 * N * offsets
