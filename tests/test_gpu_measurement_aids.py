"""The measurement aids of the C ABI (sce_bench_mfma, sce_bench_gemm; slowrun_amd.ceiling builds its
report from them): they run at small sizes, return figures that make sense for this part, and refuse shapes their
kernels do not take."""
import ctypes as C

import pytest
import torch

from slowrun_amd import _lib, ceiling

pytestmark = pytest.mark.gpu


def _scratch():
    return torch.empty(64 << 20, dtype=torch.uint8, device="cuda")


def test_matrix_instruction_alone():
    scratch = _scratch()
    tf_const, mhz_const = ceiling._mfma(False, scratch, iters=2000, reps=2)
    tf_rand, mhz_rand = ceiling._mfma(True, scratch, iters=2000, reps=2)
    # constant operands reach the published rate at the full clock; random operands are slower, never faster
    assert 0.5 * ceiling.PEAK_FP8_TFLOPS < tf_const < 1.05 * ceiling.PEAK_FP8_TFLOPS
    assert 1000 < mhz_rand <= mhz_const * 1.02 < 2600
    assert 0.3 * ceiling.PEAK_FP8_TFLOPS < tf_rand < tf_const * 1.02


def test_main_loop_alone():
    scratch = _scratch()
    tf, mhz = ceiling._gemm(4096, 4096, 2048, "random", scratch, reps=3)
    assert 500 < tf < ceiling.PEAK_FP8_TFLOPS and 1000 < mhz < 2600


def test_shapes_the_kernels_do_not_take_are_refused():
    scratch = _scratch()
    lib = _lib.lib()
    a = ceiling._operand(4096, 1024, "zero", scratch.device)
    tf, mhz = C.c_double(), C.c_double()
    args = (scratch.data_ptr(), scratch.numel(), scratch.device.index, None)
    assert lib.sce_bench_gemm(a.data_ptr(), a.data_ptr(), 4096, 4000, 1024, 1, *args, C.byref(tf), C.byref(mhz)) == 1
    assert b"multiples of 256" in lib.sce_last_error()
    assert lib.sce_bench_gemm(None, a.data_ptr(), 4096, 4096, 1024, 1, *args, C.byref(tf), C.byref(mhz)) == 1
    assert lib.sce_bench_mfma(None, 0, 0, 1, *args, C.byref(tf), C.byref(mhz)) == 1
    assert lib.sce_bench_mfma(a.data_ptr(), 4096, 10, 1, *args, C.byref(tf), C.byref(mhz)) == 1      # operand bytes too few
    assert b"random_bytes" in lib.sce_last_error()
    assert lib.sce_bench_gemm(a.data_ptr(), a.data_ptr(), 4096, 4096, 1024, 1, scratch.data_ptr(), 16, scratch.device.index, None,
                              C.byref(tf), C.byref(mhz)) == 1                                                       # scratch too small


def test_no_launch_is_counted_twice():
    """The times by kind of a backward pass add up to no more than the pass.  Few rows with the same target and a wide hidden state: the sum of that
    column's rows, which only dW waits for, is a good part of the whole."""
    from slowrun_amd import cuda_kernels as ck
    N, d, V = 4096, 65536, 256
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(N, d, device="cuda", generator=gen, dtype=torch.bfloat16)
    w = torch.randn(d, V, device="cuda", generator=gen, dtype=torch.bfloat16) * d ** -0.5
    y = torch.full((N,), 7, device="cuda")
    _loss, saved, *_ = ck.ce_forward(x, w, y, 0.02, 0.02 * d ** -0.5, 15.0, "mean", keep_dlogits=True)
    back = lambda: ck.ce_backward(saved, y, torch.ones((), device="cuda"), N, d, V, 0.02, 0.02 * d ** -0.5, 15.0, 1.0, "mean", torch.bfloat16, torch.bfloat16,
                                  keep_dlogits=True)
    back()
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    _lib.timing_enable(True)
    try:
        begin.record()
        back()
        end.record()
        kinds = _lib.timing_read()
    finally:
        _lib.timing_enable(False)
    assert kinds["dw_final"][1] >= 1 and kinds["dw"][1] == 1
    assert sum(ms for ms, _launches in kinds.values()) <= begin.elapsed_time(end) + 0.002      # (the clock of the time stamps: 10 ns a tick)
