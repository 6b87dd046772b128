"""The mean over the rows that have a target, and the counts of rows with one and of targets out of range: from the last block of the
combining kernel, or of many rows from a launch of its own.  Against the per-row losses of the same call in float64; what is left is the mean's
own rounding to float32 and, in a row, that of its loss (a difference of two numbers below 32: 2^-20 of absolute error at most)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (64 rows to a block, of rows rounded up to 256 where a backward call can follow; up to 256 blocks are added up without a launch)
@pytest.mark.parametrize("operands,N,launch", [
    ("e4m3", 1, False), ("e4m3", 257, False), ("e4m3", 16384, False), ("e4m3", 16385, True), ("e4m3", 70001, True),
    ("bf16", 64, False), ("bf16", 65, False), ("bf16", 16384, False), ("bf16", 16385, True), ("bf16", 65537, True)])
def test_mean_and_counts(operands, N, launch):
    from slowrun_amd import cuda_kernels as ck
    from .test_gpu_dw_last_round import _kernels
    d, V = 64, 300
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(N, d, device="cuda", generator=gen).bfloat16()
    w = (torch.randn(d, V, device="cuda", generator=gen) * d ** -0.5).bfloat16()
    x_s, w_s = float(x.float().abs().max()) / 448, float(w.float().abs().max()) / 448
    y = torch.randint(0, V, (N,), device="cuda", generator=gen)
    y[torch.rand(N, device="cuda", generator=gen) < 0.1] = -1
    y[0] = 5
    if N > 64:
        y[N // 2: N // 2 + 3] = torch.tensor([V, -2, 10 ** 12], device="cuda")
    out_of_range = 3 if N > 64 else 0
    kw = dict(operand_dtype=torch.bfloat16) if operands == "bf16" else {}
    losses = ck.ce_forward(x, w, y, x_s, w_s, 15.0, "none", **kw)[0].double()
    valid = (y >= 0) & (y < V)
    for _ in range(3):                                          # (the count of the blocks starts anew in every call)
        (loss, _saved, _lse, _am, n_valid), names = _kernels(lambda: ck.ce_forward(x, w, y, x_s, w_s, 15.0, "mean", **kw))
        assert ("fwd_reduce" in names) == launch, names
        assert n_valid.tolist() == [int(valid.sum()), out_of_range]
        assert abs(float(loss) - float(losses[valid].mean())) <= 2.0 ** -20 + 2.0 ** -24 * abs(float(loss))
    if operands == "e4m3":
        empty = ck.ce_forward(x, w, torch.full_like(y, -1), x_s, w_s, 15.0, "mean")
        assert bool(empty[0].isnan()) and empty[4].tolist() == [0, 0]
