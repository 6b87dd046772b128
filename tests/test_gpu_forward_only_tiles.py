"""The forward pass that leaves no dlogits, whole row tiles: last tiles of the vocabulary of every raggedness, K loops of one pair of
blocks and of several.  Small whole numbers make every logit exact, so the maximum's column is that of a 64-bit evaluation; the loss differs
from it by fp32 sums of at most V positive terms and the hardware's exp2, log2 and reciprocal (2^-22 relative each, of an exponent of up
to 2 cap log2(e) = 87: 2e-5)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("operands", ["bf16", "e4m3", "e4m3, targets from the accumulators"])
@pytest.mark.parametrize("N,d,V,vocab", [(257, 16, 1, 1), (300, 64, 127, 127), (513, 128, 256, 255), (300, 144, 257, 257), (1000, 272, 640, 513), (700, 528, 33000, 32897),
                                         (2048, 1040, 2304, 2304)])
def test_every_way_a_last_tile_can_end(N, d, V, vocab, operands):
    from slowrun_amd import _lib, cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(V + d)
    x = torch.randint(-2, 3, (N, d), device="cuda", generator=gen).bfloat16() / 4
    w = torch.randint(-2, 3, (d, V), device="cuda", generator=gen).bfloat16() / 4
    w[:, vocab:] = x[0, :, None]                                # beyond the vocabulary: what would be row 0's maximum
    x[5], w[:, 0] = -2.0, 2.0                                   # a row that is far below zero in column 0 ...
    x[6] = 0.0                                                  # ... and one of equal logits
    y = torch.randint(0, vocab, (N,), device="cuda", generator=gen)
    y[::5] = -1
    y[5] = 0
    bf16 = operands == "bf16"
    limit = _lib.lib().sce_test_set_gather_limit(1) if "accumulators" in operands else None
    try:
        loss, _saved, lse, am, nv = ck.ce_forward(x, w, y, 1.0, 1.0, 15.0, "none", want_argmax=True, vocab_size=vocab,
                                                  operand_dtype=torch.bfloat16 if bf16 else None)
    finally:
        if limit is not None:
            _lib.lib().sce_test_set_gather_limit(limit)
    u = x.double() @ w.double()[:, :vocab]
    if bf16:
        u = u.bfloat16().double()
    z = 15.0 * torch.tanh(u / 15.0)
    assert torch.equal(am.long(), (u == u.max(1, keepdim=True).values).int().argmax(1))
    assert int(nv[0]) == int((y >= 0).sum())
    assert torch.allclose(lse.double()[:N], torch.logsumexp(z, 1), rtol=0, atol=1e-4)
    assert torch.allclose(loss.double(), F.cross_entropy(z, y, reduction="none", ignore_index=-1), rtol=0, atol=1e-4)
