"""When the autograd functions call the loss head as an operator and when they call its body: whatever traces, records or transforms
operator calls still meets the operator."""
import json

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from slowrun_amd import cuda_kernels as ck


class _Subclass(torch.Tensor):
    pass


class _Names(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


def test_only_plain_calls_pass_the_operator_by():
    x = torch.zeros(4)
    with torch.no_grad():
        assert not ck._seen_as_op(x, None, torch.nn.Parameter(x))
        assert ck._seen_as_op(x.as_subclass(_Subclass)) and ck._seen_as_op([1.0]) and ck._seen_as_op(x, 1.0)
        with _Names():
            assert ck._seen_as_op(x)
        with torch.overrides.BaseTorchFunctionMode():
            assert ck._seen_as_op(x)
        with torch.autograd.profiler.profile(use_device=None):
            assert ck._seen_as_op(x)
        seen = []
        torch.func.vmap(lambda t: (seen.append(ck._seen_as_op(x)), t)[1])(torch.zeros(2, 3))
        torch.jit.trace(lambda t: (seen.append(ck._seen_as_op(x)), t + 1)[1], (x,), check_trace=False)
        assert seen and all(seen)
        assert not ck._seen_as_op(x)
    assert ck._seen_as_op(x)                                   # a backward pass that is itself differentiated


FUNCTIONS = [ck.FusedSoftcappedCrossEntropy, ck.FusedNormSoftcappedCrossEntropy]


def _apply(fn, x, w, y, reduction="mean"):
    return fn.apply(x, y, None, w, 0.02, 0.02, 1.0, 1.0, 15.0, reduction)


@pytest.fixture
def cpu_kernels(monkeypatch):
    """Stand-ins for the two library calls, linear in the upstream gradient, that read their arguments' memory as the library does."""
    def forward(x, w, targets, x_s, w_s, cap, reduction, **_more):
        assert all(t.data_ptr() for t in (x, w, targets))
        rows = torch.from_numpy(x.float().numpy()).sum(1)
        return rows.mean() if reduction == "mean" else rows, torch.zeros(8, dtype=torch.uint8), None, None, None

    def backward(saved, targets, grad_output, N, d, V, x_s, w_s, cap, grad_scale, reduction, x_dtype, w_dtype, **_more):
        assert grad_output.data_ptr() and not grad_output.is_neg()
        g = torch.from_numpy(grad_output.numpy()).expand(N)
        return g[:, None].expand(N, d).to(x_dtype).contiguous(), g.sum().expand(d, V).to(w_dtype).contiguous()

    monkeypatch.setattr(ck, "ce_forward", forward)
    monkeypatch.setattr(ck, "ce_backward", backward)


def _inputs(device="cpu", N=5, d=16, V=7):
    return torch.ones(N, d, device=device, requires_grad=True), torch.ones(d, V, device=device, requires_grad=True), torch.zeros(N, dtype=torch.int64, device=device)


@pytest.mark.parametrize("fn", FUNCTIONS)
def test_batched_gradients(fn, cpu_kernels):
    """is_grads_batched and vectorised jacobians hand backward a tensor without memory, of the plain type and outside functorch's transforms."""
    x, w, y = _inputs()
    dx, dw = torch.autograd.grad(_apply(fn, x, w, y), (x, w), torch.tensor([1.0, 2.0]), is_grads_batched=True)
    assert torch.equal(dx, torch.tensor([1.0, 2.0])[:, None, None].expand(2, 5, 16)) and torch.equal(dw, 5 * torch.tensor([1.0, 2.0])[:, None, None].expand(2, 16, 7))
    jac = torch.autograd.functional.jacobian(lambda t: _apply(fn, t, w, y, "none"), x, vectorize=True)
    assert torch.equal(jac, torch.eye(5)[:, :, None].expand(5, 5, 16))


@pytest.mark.parametrize("fn", FUNCTIONS)
def test_gradients_whose_memory_is_not_their_value(fn, cpu_kernels):
    x, w, y = _inputs()
    for go, value in ((torch._neg_view(torch.tensor(2.0)), -2.0), (torch._efficientzerotensor(()), 0.0)):
        (dx,) = torch.autograd.grad(_apply(fn, x, w, y), x, go)
        assert torch.equal(dx, torch.full((5, 16), value))


@pytest.mark.parametrize("offsets,keep", [(1, False), (1, True), (3, True)])
@pytest.mark.parametrize("fn", FUNCTIONS)
def test_meta_tensors(fn, offsets, keep):
    """Shapes and types of a step, from the operators' fake implementations."""
    x, w, y = _inputs("meta")
    x, mtp = x.detach().bfloat16().requires_grad_(True), torch.ones(offsets, device="meta") if offsets > 1 else None
    rest = (None, keep) if fn is ck.FusedNormSoftcappedCrossEntropy else (keep,)
    loss = fn.apply(x, y, mtp, w, 0.02, 0.02, 1.0, 1.0, 15.0, "none", *rest)
    assert loss.is_meta and loss.shape == (5,) and loss.dtype == torch.float32
    loss.mean().backward()
    assert x.grad.is_meta and x.grad.shape == x.shape and x.grad.dtype == torch.bfloat16
    assert w.grad.is_meta and w.grad.shape == w.shape and w.grad.dtype == torch.float32
    if offsets == 1:
        assert fn.apply(x, y, None, w, 0.02, 0.02, 1.0, 1.0, 15.0, "mean", *rest).shape == ()


@pytest.mark.parametrize("fn", FUNCTIONS)
def test_execution_trace_without_the_profiler(fn, cpu_kernels, tmp_path):
    path = str(tmp_path / "trace.json")
    observer = torch.profiler.ExecutionTraceObserver().register_callback(path)
    observer.start()
    x, w, y = _inputs()
    _apply(fn, x, w, y).backward()
    observer.stop()
    observer.unregister_callback()
    with open(path) as f:
        names = [node["name"] for node in json.load(f)["nodes"]]
    prefix = "slowrun_amd::norm_ce_" if fn is ck.FusedNormSoftcappedCrossEntropy else "slowrun_amd::ce_"
    assert names.count(prefix + "forward") == 1 and names.count(prefix + "backward") == 1


@pytest.mark.gpu
@pytest.mark.parametrize("fn", FUNCTIONS)
def test_batched_gradients_on_the_gpu(fn):
    x, w = torch.randn(300, 64, device="cuda").bfloat16().requires_grad_(True), torch.randn(64, 500, device="cuda").bfloat16().requires_grad_(True)
    y = torch.randint(0, 500, (300,), device="cuda")
    with torch.no_grad():
        assert not ck._seen_as_op(x.detach(), w.detach(), y, None)
    out = _apply(fn, x, w, y, "none")
    go = torch.randn(3, 300, device="cuda")
    batched = torch.autograd.grad(out, (x, w), go, is_grads_batched=True, retain_graph=True)
    for k in range(3):
        assert all(torch.equal(b[k], one) for b, one in zip(batched, torch.autograd.grad(out, (x, w), go[k], retain_graph=True)))
    (dx,) = torch.autograd.grad(out, x, torch._neg_view(go[0]))
    assert torch.equal(dx, -batched[0][0])


@pytest.mark.gpu
@pytest.mark.parametrize("fn", [ck.FusedSoftcappedCrossEntropy, ck.FusedNormSoftcappedCrossEntropy])
def test_both_ways_give_the_same_and_modes_see_the_operator(fn):
    x = torch.randn(300, 64, device="cuda").bfloat16()
    w = torch.randn(64, 500, device="cuda").bfloat16()
    y = torch.randint(0, 500, (300,), device="cuda")

    def step():
        a, b = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
        loss = fn.apply(a, y, None, b, 0.02, 0.02, 1.0, 1.0, 15.0, "mean")
        loss.backward()
        return loss.detach(), a.grad, b.grad

    plain = step()
    with _Names() as names:
        a, b = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
        loss = fn.apply(a, y, None, b, 0.02, 0.02, 1.0, 1.0, 15.0, "mean")
    assert any("ce_forward" in n for n in names.seen)
    loss.backward()
    with torch.autograd.profiler.profile(use_device=None):
        profiled = step()
    for other in ((loss.detach(), a.grad, b.grad), profiled):
        assert all(torch.equal(p, q) for p, q in zip(plain, other))
    # differentiating the backward pass stays an error
    a = x.clone().requires_grad_(True)
    loss = fn.apply(a, y, None, w, 0.02, 0.02, 1.0, 1.0, 15.0, "mean")
    with pytest.raises(RuntimeError):
        (g,) = torch.autograd.grad(loss, a, torch.ones((), device="cuda", requires_grad=True), create_graph=True)
        g.sum().backward()
