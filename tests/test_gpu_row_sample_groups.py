"""Exponent boosts and target logits ahead of the forward pass, from workgroups of 32, 64 and 128 rows and from the kernel of whole row
tiles: the same bits for the same rows, either side of every line between them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _saved(saved, N, d, n_predict):
    Np, ldx = (N + 255) // 256 * 256, (d + 255) // 256 * 256 + 128
    up = lambda n: (n + 255) // 256 * 256
    off = 256 + up(Np * ldx) + up(Np * 4)
    lam2 = saved[off: off + Np * 4].view(torch.float32)
    off += up(Np * 4)
    zy = saved[off: off + Np * 4 * n_predict].view(torch.float32).view(n_predict, Np)
    off += up(Np * 4 * n_predict) + up(Np * 4)
    return zy, torch.minimum(saved[off: off + Np * 4].view(torch.float32), lam2).clamp(-64.0, 120.0)


@pytest.mark.parametrize("few,more", [(255, 4097), (4096, 4352), (8192, 32768), (32768, 33024)])
@pytest.mark.parametrize("offsets,d,V", [(1, 272, 2049), (4, 16, 515)])
def test_rows_to_a_workgroup(offsets, d, V, few, more):
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(d)
    x = torch.randn(more, d, device="cuda", generator=gen).bfloat16()
    x[7] *= 8.0
    w = (torch.randn(d, V, device="cuda", generator=gen) * d ** -0.5).bfloat16()
    y = torch.randint(0, V, (more,), device="cuda", generator=gen)
    y[torch.rand(more, device="cuda", generator=gen) < 0.2] = -1
    y[100:110] = -1
    mtp = torch.tensor([1.0, 0.5, 0.25, 0.125][:offsets], device="cuda") if offsets > 1 else None
    got = []
    for n in (few, more):
        _loss, saved, *_ = ck.ce_forward(x[:n], w, y[:n], float(x.float().abs().max()) / 448, float(w.float().abs().max()) / 448, 15.0, "none",
                                         mtp_weights=mtp, keep_dlogits=True)
        zy, lam = _saved(saved, n, d, offsets)
        # (offsets of the last rows look past the smaller batch, and so do the targets that the last tile's rows are sampled at)
        got.append((zy[:, : few - 4], lam[: (few - 1) // 256 * 256 if few > 256 else 0]))
    assert torch.equal(got[0][0], got[1][0]) and bool((got[0][0] != 0).any())
    assert torch.equal(got[0][1], got[1][1])
    if few > 256:
        assert bool((got[0][1] == -64).any()) and bool((got[0][1] != -64).any())
