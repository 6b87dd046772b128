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
