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


# (both heads have 16 of their 48 tiles in halves, or 5 of 37, as long as all of those lie within the vocabulary: 4096 columns, 1280)
@pytest.mark.parametrize("tiles,V,vocab", [(8, 48 * 256, v) for v in (2, 200, 1024, 3000, 4095, 4096, 4097, 12000)] +
                         [(8, 37 * 256 - 5, v) for v in (1000, 1279, 1280, 1281, 37 * 256 - 6)])
@pytest.mark.parametrize("offsets", [1, 3])
def test_columns_beyond_the_vocabulary(tiles, V, vocab, offsets):
    """A vocabulary that ends in the first tiles, which are the ones in halves: the dlogits of a longer batch, bit for bit and zero beyond
    it, and the losses and gradients of a head that has those columns alone."""
    from slowrun_amd import _lib, cuda_kernels as ck
    few, more, d = tiles * 256 - 3, 33024, 64
    gen = torch.Generator(device="cuda").manual_seed(vocab)
    x = torch.randn(more, d, device="cuda", generator=gen).bfloat16()
    w = (torch.randn(d, V, device="cuda", generator=gen) * d ** -0.5).bfloat16()
    w[:, vocab:] *= 4.0                                         # columns that would be noticed
    y = torch.randint(0, vocab, (more,), device="cuda", generator=gen)
    y[torch.rand(more, device="cuda", generator=gen) < 0.1] = -1
    mtp = torch.tensor([1.0, 0.5, 0.25][:offsets], device="cuda") if offsets > 1 else None
    x_s, w_s, go = float(x.float().abs().max()) / 448, float(w.float().abs().max()) / 448, torch.full((few,), 1.0 / few, device="cuda")

    def forward(n, head, **more_args):
        return ck.ce_forward(x[:n], head, y[:n], x_s, w_s, 15.0, "none", want_argmax=True, mtp_weights=mtp, **more_args)

    loss, saved, lse, am, _nv = forward(few, w, keep_dlogits=True, vocab_size=vocab)
    g, e = _dlogits(saved, _lib.sizes_for(few, d, V, offsets), few, V)
    keep = tiles - 1
    l1, saved1, s1, a1, _nv = forward(more, w, keep_dlogits=True, vocab_size=vocab)
    g1, e1 = _dlogits(saved1, _lib.sizes_for(more, d, V, offsets), more, V)
    assert torch.equal(am[: keep * 256], a1[: keep * 256]) and torch.equal(g[:keep], g1[:keep]) and torch.equal(e[:, : 2 * keep], e1[:, : 2 * keep])
    # the head of those columns alone (its tiles are split otherwise: the order of a sum of at most V positive fp32 terms)
    head = w[:, :vocab].contiguous()
    l2, saved2, s2, a2, _nv = forward(few, head, keep_dlogits=True)
    assert torch.equal(am, a2) and int(am.max()) < vocab
    assert torch.allclose(lse, s2, rtol=2e-6, atol=2e-5) and torch.allclose(loss, l2, rtol=2e-6, atol=2e-5)
    back = lambda s, v, **more_args: ck.ce_backward(s, y[:few], go, few, d, v, x_s, w_s, 15.0, 1.0, "none", torch.float32, torch.float32,
                                                    mtp_weights=mtp, keep_dlogits=True, **more_args)
    (dx, dw), (dx2, dw2) = back(saved, V, vocab_size=vocab), back(saved2, vocab)
    assert not bool(dw[:, vocab:].any())
    # the estimates behind the rows' boosts look at other tiles, so the e4m3 dlogits (unit 2^-4 of an element, independent of each other) are not the same bytes
    for ours, ref in ((dx, dx2), (dw[:, :vocab], dw2)):
        assert float((ours - ref).double().norm()) <= 2.0 ** -4 * float(ref.double().norm())
