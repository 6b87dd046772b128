"""Tiles that the forward pass shares out as halves of the wave's rows: the same dlogits, bit for bit, as in a longer batch whose tiles
are all whole, and row sums that differ by the order of their terms alone (fp32 sums of at most V positive terms)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _dlogits(saved, sz, N, V):
    Np, Vp = (N + 255) // 256 * 256, (V + 255) // 256 * 256
    g = saved[sz.saved_bytes:]
    return g[: Np * Vp].view(Np // 256, Vp * 256), g[Np * Vp: Np * Vp + Vp // 128 * (Np // 128) * 4].view(Vp // 128, Np // 128, 4)


# (one round of workgroups on 256 CUs: 256 / row tiles splits, of which as many as the remainder twice have half a tile more)
@pytest.mark.parametrize("tiles,V", [(8, 33 * 256), (8, 48 * 256 - 5), (16, 17 * 256 - 255), (16, 40 * 256), (15, 18 * 256)])
@pytest.mark.parametrize("offsets,d", [(1, 64), (3, 528)])
def test_halves_against_whole_tiles(tiles, V, offsets, d):
    from slowrun_amd import _lib, cuda_kernels as ck
    few, more = tiles * 256 - 3, 33024
    gen = torch.Generator(device="cuda").manual_seed(V + d)
    x = torch.randn(more, d, device="cuda", generator=gen).bfloat16()
    x[7] *= 8.0
    w = (torch.randn(d, V, device="cuda", generator=gen) * d ** -0.5).bfloat16()
    y = torch.randint(0, V, (more,), device="cuda", generator=gen)
    y[:600] %= 512                                              # targets in the first tiles, which are the ones in halves
    y[torch.rand(more, device="cuda", generator=gen) < 0.1] = -1
    mtp = torch.tensor([1.0, 0.5, 0.25][:offsets], device="cuda") if offsets > 1 else None
    got = []
    for n in (few, more):
        loss, saved, lse, am, _nv = ck.ce_forward(x[:n], w, y[:n], float(x.float().abs().max()) / 448, float(w.float().abs().max()) / 448, 15.0, "none",
                                                  want_argmax=True, mtp_weights=mtp, keep_dlogits=True)
        g, e = _dlogits(saved, _lib.sizes_for(n, d, V, offsets), n, V)
        keep = tiles - 1                                        # (the last row tile of the shorter batch looks past its end)
        got.append((loss[: keep * 256], lse[: keep * 256], am[: keep * 256], g[:keep], e[:, : 2 * keep]))
    (l0, s0, a0, g0, e0), (l1, s1, a1, g1, e1) = got
    assert torch.equal(a0, a1) and torch.equal(g0, g1) and torch.equal(e0, e1) and bool((g0 != 0).any())
    assert torch.allclose(s0, s1, rtol=2e-6, atol=2e-5) and torch.allclose(l0, l1, rtol=2e-6, atol=2e-5)
