"""Target logits and exponent boosts ahead of the forward pass: a pass of up to 32 row tiles takes them from a kernel of its own
(32 rows to a workgroup), a larger one from the tile kernel.  Both have to give the same bits (the forward kernel knows a
target by its value), so the rows of a batch of 8192 are compared with the same rows at the head of a batch of 8448."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _saved(saved, N, d, n_predict):
    """(z_y [n_predict][Np], boosts [Np]) as the forward pass left them in `saved`."""
    Np, ldx = (N + 255) // 256 * 256, (d + 255) // 256 * 256 + 128
    up = lambda n: (n + 255) // 256 * 256
    off = 256 + up(Np * ldx) + 2 * up(Np * 4)
    zy = saved[off: off + Np * 4 * n_predict].view(torch.float32).view(n_predict, Np)
    off += up(Np * 4 * n_predict) + up(Np * 4)
    return zy, saved[off: off + Np * 4].view(torch.float32)


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("offsets,d,V", [(1, 16, 7), (1, 272, 2049), (2, 256, 515), (4, 528, 1000), (3, 1024, 300)])
def test_few_row_tiles_and_many_give_the_same_bits(offsets, d, V, keep):
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(d)
    few, many = 8192, 8448
    x = torch.randn(many, d, device="cuda", generator=gen).bfloat16()
    x[7] *= 8.0
    w = (torch.randn(d, V, device="cuda", generator=gen) * d ** -0.5).bfloat16()
    y = torch.randint(0, V, (many,), device="cuda", generator=gen)
    y[torch.rand(many, device="cuda", generator=gen) < 0.2] = -1
    y[1000:1300] = -1
    mtp = torch.tensor([1.0, 0.5, 0.25, 0.125][:offsets], device="cuda")
    got = []
    for n in (few, many):
        loss, saved, *_ = ck.ce_forward(x[:n], w, y[:n], float(x.float().abs().max()) / 448, float(w.float().abs().max()) / 448, 15.0, "none", mtp_weights=mtp, keep_dlogits=keep)
        zy, lam = _saved(saved, n, d, offsets)
        got.append((loss[: few - 4], zy[:, : few - 4], lam[: few - 256]))       # (offsets of the last rows look past the smaller batch)
    assert torch.allclose(got[0][0], got[1][0], rtol=1e-5, atol=1e-5)             # (the splits of the vocabulary differ: the sums' order)
    assert torch.equal(got[0][1], got[1][1]) and bool((got[0][1] != 0).any())
    if keep:
        assert torch.equal(got[0][2], got[1][2]) and bool((got[0][2] == -64).any()) and bool((got[0][2] != -64).any())
