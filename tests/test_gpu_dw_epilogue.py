"""dW stored from the accumulators of its main loop (one launch over all rows) against the way over fp32 partials that a
small workspace takes (one launch per 256 rows, summed by the finalising kernel): the same products, so the two differ by
the order of an fp32 sum of a few parts -- 2^-20 of the largest element here, generously -- and by the rounding to the
output type that this can tip over, one unit: 2^-8 of a bf16 value."""
import pytest
import torch

from slowrun_amd import configs

pytestmark = pytest.mark.gpu


def _targets(kind, N, V, gen):
    if kind == "spread":                  # a few entries to a tile: their rows fit beside the main loop's buffers
        return torch.randint(0, V, (N,), generator=gen)
    if kind == "crowded":                 # about five entries to a column in some tiles: taken in groups after the main loop
        return torch.randint(0, min(V, 150), (N,), generator=gen) + max(0, V - 160) // 256 * 256
    y = torch.randint(0, V, (N,), generator=gen)      # "hot": one column with hundreds of entries (chunk sums), next to ordinary ones
    y[torch.rand(N, generator=gen) < 0.5] = V // 2
    y[::7] = -1
    return y


@pytest.mark.parametrize("kind", ["spread", "crowded", "hot"])
@pytest.mark.parametrize("w_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,d,V,K", [(256, 16, 8, 1), (257, 272, 1003, 1), (512, 256, 2056, 2), (300, 1040, 4096, 3), (1100, 528, 263, 4)])
def test_dw_from_the_accumulators(kind, w_dtype, N, d, V, K):
    from slowrun_amd import _lib
    from slowrun_amd import cuda_kernels as ck
    inp = configs.make_inputs("tiny_track", N=N, d=d, V=V)
    y = _targets(kind, N, V, torch.Generator().manual_seed(N + K)).clamp_(max=V - 1).cuda()
    x, w = inp.x.cuda().bfloat16(), inp.w.cuda().to(w_dtype)
    mw = torch.tensor([1.0, 0.5, 0.25, 0.125][:K], device="cuda") if K > 1 else None
    go = torch.rand(N, generator=torch.Generator().manual_seed(1)).cuda() / N
    _out, saved, *_ = ck.ce_forward(x, w, y, inp.x_s, inp.w_s, inp.cap, "none", mtp_weights=mw, keep_dlogits=False)
    args = (saved, y, go, N, d, V, inp.x_s, inp.w_s, inp.cap, 1.0, "none", torch.bfloat16, w_dtype)
    sz = _lib.sizes_for(N, d, V, K)
    # the last round of tiles shared out along K (where it is), and every tile with one workgroup: a workspace without room for the former's partial tiles
    tiles, pairs = -(-d // 256) * -(-V // 256), -(-N // 256)
    shared = tiles % 256 > 0 and 2 * -(-(tiles % 256) * pairs // 256) <= pairs
    room = sz.bwd_workspace_bytes - (256 + tiles % 256) * 256 * 256 * 4 * shared
    ways = [ck.ce_backward(*args, mtp_weights=mw, workspace_bytes=b)[1] for b in {sz.bwd_workspace_bytes, room}]
    ref = ck.ce_backward(*args, mtp_weights=mw, panel_rows=256, workspace_bytes=sz.bwd_workspace_min_bytes)[1].double()
    unit = 2.0 ** -8 if w_dtype == torch.bfloat16 else 2.0 ** -23
    for dw in ways:
        assert bool(((dw.double() - ref).abs() <= unit * ref.abs() + 2.0 ** -20 * ref.abs().max()).all())
    assert float(ref.abs().max()) > 0
