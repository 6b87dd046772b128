"""When the autograd functions call the loss head as an operator and when they call its body: whatever traces, records or transforms
operator calls still meets the operator."""
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
