"""The last round of dW's tiles -- 128 rows of a tile to a workgroup, shared out along K, or a workgroup to each tile like the full
rounds -- against the way over fp32 partials that a small workspace takes: the same products, so that the difference is the
order of an fp32 sum of a few parts, 2^-20 of the largest element here, and one unit of the output type's rounding.  And dX of
few tiles, whose K loop is cut into up to 16 parts."""
import json

import pytest
import torch

from slowrun_amd import configs
from . import parity_util as pu
from .test_gpu_dw_epilogue import _targets

pytestmark = pytest.mark.gpu


def _profiled(fn):
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        out = fn()
        torch.cuda.synchronize()
    return out, p


def _kernels(fn):
    out, p = _profiled(fn)
    return out, " ".join(e.key for e in p.key_averages())


def _workgroups(p, path):
    """{kernel: workgroups of its last launch}"""
    p.export_chrome_trace(path)
    with open(path) as f:
        events = [e for e in json.load(f)["traceEvents"] if "grid" in e.get("args", {})]
    return {e["name"].split("(")[0].split("<")[0].split("::")[-1]: e["args"]["grid"][0] for e in events}


@pytest.mark.parametrize("kind", ["spread", "crowded", "hot"])
@pytest.mark.parametrize("w_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("way,N,d,V,K", [
    ("half", 1, 16, 8, 1), ("half", 513, 272, 2049, 2), ("half", 300, 1040, 4096, 3), ("half", 2048, 528, 5000, 1), ("half", 700, 112, 32701, 1), ("half", 300, 528, 25000, 1),
    ("tail", 4700, 16, 250, 1), ("tail", 6000, 272, 1003, 2),
    ("out", 300, 16, 33100, 1), ("out", 600, 16, 65536, 1)])
def test_last_round_of_dw(kind, w_dtype, way, N, d, V, K, tmp_path):
    from slowrun_amd import _lib
    from slowrun_amd import cuda_kernels as ck
    inp = configs.make_inputs("tiny_track", N=N, d=d, V=V)
    y = _targets(kind, N, V, torch.Generator().manual_seed(N + K)).clamp_(max=V - 1).cuda()
    if N == 1:
        y[0] = V // 2
    x, w = inp.x.cuda().bfloat16(), inp.w.cuda().to(w_dtype)
    mw = torch.tensor([1.0, 0.5, 0.25, 0.125][:K], device="cuda") if K > 1 else None
    go = torch.rand(N, generator=torch.Generator().manual_seed(1)).cuda() / N
    _out, saved, *_ = ck.ce_forward(x, w, y, inp.x_s, inp.w_s, inp.cap, "none", mtp_weights=mw)
    args = (saved, y, go, N, d, V, inp.x_s, inp.w_s, inp.cap, 1.0, "none", torch.bfloat16, w_dtype)
    (_dx, dw), p = _profiled(lambda: ck.ce_backward(*args, mtp_weights=mw))
    grid = _workgroups(p, str(tmp_path / "trace.json"))
    assert ("bwd_dw_tail_kernel" in grid) == (way == "tail") and ("bwd_dw_out_kernel" in grid) == (way != "tail"), grid
    # whole tiles are dealt out 256 at a time; of the half tiles there are two to a tile of the last round, on eight XCDs
    tiles = ((d + 255) // 256) * ((V + 255) // 256)
    if way != "tail":
        assert grid["bwd_dw_out_kernel"] == ((tiles + 255) // 256 * 256 if way == "out" else tiles // 256 * 256 + (2 * (tiles % 256) + 7) // 8 * 8), grid
    ref = ck.ce_backward(*args, mtp_weights=mw, panel_rows=256, workspace_bytes=_lib.sizes_for(N, d, V, K).bwd_workspace_min_bytes)[1].double()
    unit = 2.0 ** -8 if w_dtype == torch.bfloat16 else 2.0 ** -23
    assert bool(((dw.double() - ref).abs() <= unit * ref.abs() + 2.0 ** -20 * ref.abs().max()).all())
    assert float(ref.abs().max()) > 0


@pytest.mark.parametrize("N,d,V", [(100, 16, 4096), (300, 272, 33001), (257, 64, 50257)])
def test_dx_in_many_parts(N, d, V):
    inp = configs.make_inputs("irregular", N=N, d=d, V=V)
    ours = pu.run_ours(inp, "mean", keep_dlogits=True)
    pu.check_parity(ours, pu.run_oracle(inp, ours, "mean"), "mean")
