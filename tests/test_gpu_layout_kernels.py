"""The casts, maxima and transposes at the edges of their vector paths: lengths around a load, misaligned bases, ragged
tiles.  All exact: bytes of a defined cast, a maximum, a permutation."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (16, 16), (128, 128), (129, 127), (144, 272), (127, 4096), (1008, 130), (300, 1024)])
@pytest.mark.parametrize("off", [0, 5])
def test_transpose_copy_edges(rows, cols, off):
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(rows)
    src = torch.randint(0, 256, (rows * cols + off,), dtype=torch.uint8, device="cuda", generator=gen)[off:].view(rows, cols)
    buf = torch.full((rows * cols + 32,), 77, dtype=torch.uint8, device="cuda")
    dst = buf[off: off + rows * cols].view(cols, rows)
    ck.transpose_copy(src, dst)
    assert torch.equal(dst, src.t().contiguous())
    assert bool((buf[:off] == 77).all()) and bool((buf[off + rows * cols:] == 77).all())


@pytest.mark.parametrize("rows,cols", [(15, 17), (143, 129), (300, 257), (65, 2561)])
@pytest.mark.parametrize("soff,doff", [(1, 2), (3, 0), (0, 7), (9, 15)])
def test_transpose_copy_of_rows_at_any_address(rows, cols, soff, doff):
    """Rows and bases that are no multiple of 16 bytes move in 16-byte accesses too: nothing beside the output is written."""
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(rows + soff)
    src = torch.randint(0, 256, (rows * cols + soff,), dtype=torch.uint8, device="cuda", generator=gen)[soff:].view(rows, cols)
    buf = torch.full((rows * cols + 32,), 77, dtype=torch.uint8, device="cuda")
    dst = buf[doff: doff + rows * cols].view(cols, rows)
    ck.transpose_copy(src, dst)
    assert torch.equal(dst, src.t().contiguous())
    assert bool((buf[:doff] == 77).all()) and bool((buf[doff + rows * cols:] == 77).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 7, 16, 17, 2047, 4096 * 8 + 3, 1 << 20])
@pytest.mark.parametrize("off", [0, 1])
def test_amax_and_cast_edges(dtype, n, off):
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(n)
    t = torch.randn(n + off, device="cuda", generator=gen).to(dtype)[off:]
    for at in {0, n - 1, n // 2}:             # the largest value in the first, the last and a middle place
        u = t.clone() if off == 0 else torch.cat([t[:1], t])[1:]
        u[at] = -9.0
        assert float(ck.amax_scale(u)) == float(u.float().abs().max().cpu() / 448)      # (a true division; torch multiplies by 1 / 448 on the GPU)
    for scale in (0.0123, ck.amax_scale(u)):
        assert torch.equal(ck.quantize_e4m3(u, scale).view(torch.uint8), u.div(scale).to(torch.float8_e4m3fn).view(torch.uint8))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [5, 16, 31, 4096 + 17])
@pytest.mark.parametrize("soff,doff", [(1, 0), (0, 1), (3, 13), (7, 6)])
def test_cast_between_any_addresses(dtype, n, soff, doff):
    """The C entry takes source and destination wherever they lie (elements of the source aligned to themselves): the same bytes, and
    none beside them."""
    from slowrun_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(n + soff)
    t = torch.randn(n + soff, device="cuda", generator=gen).to(dtype)[soff:]
    buf = torch.full((n + 32,), 77, dtype=torch.uint8, device="cuda")
    _lib.check(_lib.lib().sce_quantize_e4m3(t.data_ptr(), _lib.SCE_F32 if dtype == torch.float32 else _lib.SCE_BF16, buf.data_ptr() + doff, 0.0123, n, t.device.index,
                                           torch.cuda.current_stream().cuda_stream), "sce_quantize_e4m3")
    assert torch.equal(buf[doff: doff + n], t.div(0.0123).to(torch.float8_e4m3fn).view(torch.uint8))
    assert bool((buf[:doff] == 77).all()) and bool((buf[doff + n:] == 77).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("norm", [None, 1e-6])
@pytest.mark.parametrize("N,d,V", [(5, 48, 130), (61, 272, 1003), (300, 144, 515)])
def test_operands_quantised_from_rows_at_any_address(dtype, norm, N, d, V):
    """The e4m3 operands of a step from aligned rows, from rows of odd length and from an odd base: the same bytes, so the same bits."""
    from slowrun_amd import cuda_kernels as ck
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(N, d, device="cuda", generator=gen).to(dtype)
    w = (torch.randn(d, V, device="cuda", generator=gen) * d ** -0.5).to(dtype)
    y = torch.randint(0, V, (N,), device="cuda", generator=gen)
    res = []
    for wpad, xpad, off in ((-V % 8, 0, 0), (-V % 8 + 1, 1, 0), (-V % 8 + 8, 8, 1), (-V % 8 + 8, 16, 3)):
        wb, xb = torch.full((d * (V + wpad) + 8,), 9.0, device="cuda", dtype=dtype), torch.full((N * (d + xpad) + 8,), 9.0, device="cuda", dtype=dtype)
        wv, xv = wb.as_strided((d, V), (V + wpad, 1), off), xb.as_strided((N, d), (d + xpad, 1), off)
        wv.copy_(w); xv.copy_(x)
        out, saved, lse, am, _n = ck.ce_forward(xv, wv, y, 0.02, 0.01, 15.0, "none", want_argmax=True, norm_eps=norm, keep_dlogits=True)
        dx, dw = ck.ce_backward(saved, y, torch.ones(N, device="cuda"), N, d, V, 0.02, 0.01, 15.0, 1.0, "none", dtype, dtype, keep_dlogits=True,
                                hidden=xv if norm else None, norm_eps=norm)
        res.append((out, lse, am, dx, dw))
    for r in res[1:]:
        assert all(torch.equal(a, b) for a, b in zip(r, res[0]))
