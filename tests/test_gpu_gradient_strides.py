"""Gradients into rows with a stride and at addresses of the caller's: through the C ABI, since the Python wrapper allocates
contiguous ones.  The kernels choose 16-byte or single stores by base, stride and tile; the same sums go out either way, so
every element has the bits of the contiguous call, and what lies between the rows stays untouched."""
import ctypes as C

import pytest
import torch

from slowrun_amd import _lib, configs

pytestmark = pytest.mark.gpu


def _backward(saved, y, go, inp, N, d, V, keep, dtype, dx, dx_ld, dw, dw_ld):
    from slowrun_amd import cuda_kernels as ck
    sz = _lib.sizes_for(N, d, V, 1)
    ws = torch.empty(sz.bwd_workspace_kept_bytes if keep else sz.bwd_workspace_bytes, dtype=torch.uint8, device="cuda")
    a = ck._base_args(saved, N, d, V, inp.x_s, inp.w_s, inp.cap, 1.0, "none", y)
    a.saved, a.saved_bytes, a.workspace, a.workspace_bytes = saved.data_ptr(), saved.numel(), ws.data_ptr(), ws.numel()
    a.grad_output, a.dlogits_from_forward = go.data_ptr(), int(keep)
    code = _lib.SCE_F32 if dtype == torch.float32 else _lib.SCE_BF16
    a.dx, a.dx_dtype, a.dx_ld = dx.data_ptr(), code, dx_ld
    a.dw, a.dw_dtype, a.dw_ld = dw.data_ptr(), code, dw_ld
    _lib.check(_lib.lib().sce_backward(C.byref(a)), "sce_backward")
    torch.cuda.synchronize()


def _rows(rows, cols, pad, off, dtype):
    """A (rows, cols) view `off` elements into a buffer of 77s, `pad` elements between its rows, and the buffer."""
    buf = torch.full((off + rows * (cols + pad) + 64,), 77.0, dtype=dtype, device="cuda")
    return buf.as_strided((rows, cols), (cols + pad, 1), off), buf


# tiles of dX and dW that are shared out along K and tiles that are not; V a multiple of 8 and not, with a last tile of one column
@pytest.mark.parametrize("N,d,V", [(300, 272, 1003), (300, 272, 1000), (2000, 528, 257), (1100, 1040, 4099), (70000, 16, 264)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("keep", [True, False])
def test_gradients_into_strided_rows(N, d, V, dtype, keep):
    from slowrun_amd import cuda_kernels as ck
    inp = configs.make_inputs("tiny_track", N=N, d=d, V=V)
    x, w, y = inp.x.cuda().bfloat16(), inp.w.cuda().bfloat16(), inp.targets.cuda()
    go = torch.rand(N, generator=torch.Generator().manual_seed(1)).cuda() / N
    _out, saved, *_ = ck.ce_forward(x, w, y, inp.x_s, inp.w_s, inp.cap, "none", keep_dlogits=keep)
    want = [torch.zeros(N, d, dtype=dtype, device="cuda"), torch.zeros(d, V, dtype=dtype, device="cuda")]
    _backward(saved, y, go, inp, N, d, V, keep, dtype, want[0], d, want[1], V)
    assert all(float(t.float().abs().max()) > 0 for t in want)
    # (elements between rows of dX and of dW, elements before the first): rows of whole 16 bytes, odd rows, an odd base
    for xpad, wpad, off in ((16, -V % 8, 0), (16, -V % 8 + 8, 8), (1, 1, 0), (8, -V % 8, 1), (3, 0, 2)):
        dx, xbuf = _rows(N, d, xpad, off, dtype)
        dw, wbuf = _rows(d, V, wpad, off, dtype)
        _backward(saved, y, go, inp, N, d, V, keep, dtype, dx, d + xpad, dw, V + wpad)
        for got, ref, buf in ((dx, want[0], xbuf), (dw, want[1], wbuf)):
            assert torch.equal(got, ref), (xpad, wpad, off)
            got.fill_(77.0)
            assert bool((buf == 77.0).all()), (xpad, wpad, off)
