"""The layout kernels of the bf16 operands at the edges of their vector paths: the same values read through aligned rows
(16-byte loads) and through rows that are not (element by element) have to give the same bits, and both the loss of a plain
fp32 evaluation of the bf16 head.  Bound: a logit on the other side of a bf16 rounding moves by 2^-8 of itself (|u| < 8 here)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,d,V", [(1, 16, 7), (5, 112, 130), (61, 144, 1000), (257, 128, 256), (300, 256, 515)])
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
