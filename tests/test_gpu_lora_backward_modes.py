"""The LoRA linear's backward in contexts that its forward did not see, on the
GPU, by the native node and by the Python function: inside autocast (the
gradients of the backward outside it, in the operands' dtype), with batched
gradients, and under a dispatch mode or a profiler entered after the forward
(which see the operator)."""

from __future__ import annotations

import pytest
import torch

from cuda_force_amd import ops
from cuda_force_amd.autograd import lora_linear_autograd

from torch.utils._python_dispatch import TorchDispatchMode

from . import gpu_util as g

pytestmark = pytest.mark.gpu


def _operands(dtype, rows=70, k=64, n=40, rank=8):
    gen = torch.Generator(device="cuda").manual_seed(0)
    shapes = ((rows, k), (k, n), (k, rank), (rank, n))
    return [torch.randn(s, generator=gen, device="cuda").to(dtype) for s in shapes]


@pytest.mark.parametrize("linear", [ops.lora_linear, lora_linear_autograd])
@pytest.mark.parametrize("dtype,auto", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float16)])
def test_backward_inside_autocast_equals_the_one_outside(linear, dtype, auto):
    g.announce(f"LoRA backward inside autocast, {dtype} operands, autocast {auto}")
    operands = _operands(dtype)
    grads = []
    for inside in (False, True):
        x, w, a, b = (t.clone() for t in operands)
        leaves = [x.requires_grad_(), a.requires_grad_(), b.requires_grad_()]
        y = linear(x, w, a, b, 0.5)
        with torch.autocast("cuda", dtype=auto, enabled=inside):
            grads.append(torch.autograd.grad(y, leaves, torch.ones_like(y)))
    for u, v in zip(*grads):
        assert u.dtype == dtype
        assert torch.equal(u, v)


@pytest.mark.parametrize("linear", [ops.lora_linear, lora_linear_autograd])
@pytest.mark.parametrize("needed", [(0, 2, 3), (2, 3), (0, 1, 2, 3)])
def test_batched_gradients_equal_one_at_a_time(linear, needed):
    g.announce(f"LoRA backward with batched gradients, operands {needed}")
    operands = _operands(torch.float32)
    leaves = [operands[i].requires_grad_() for i in needed]
    y = linear(*operands, 0.5)
    dy = torch.randn(3, *y.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    batched = torch.autograd.grad(y, leaves, dy, is_grads_batched=True, retain_graph=True)
    singly = [torch.autograd.grad(y, leaves, row, retain_graph=True) for row in dy]
    for got, want in zip(batched, (torch.stack(t) for t in zip(*singly))):
        # The same fp32 products, the weights' in one batched GEMM: sums of at
        # most 70 terms in another order.
        torch.testing.assert_close(got, want, rtol=1e-5, atol=70 * 2.0**-24 * want.abs().max().item())


def test_modes_and_profilers_entered_before_the_backward_see_the_operator():
    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(func.name())
            return func(*args, **(kwargs or {}))

    x, w, a, b = _operands(torch.bfloat16)
    leaves = [t.requires_grad_() for t in (x, a, b)]
    y = ops.lora_linear(x, w, a, b, 0.5)
    dy = torch.ones_like(y)
    plain = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    with Seen() as mode:
        seen = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    assert "cudaforge::lora_linear_bwd_input" in mode.names
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        profiled = torch.autograd.grad(y, leaves, dy)
    assert any(e.name == "cudaforge::lora_linear_bwd_input" for e in prof.events())
    for u, v, p in zip(plain, seen, profiled):
        assert torch.equal(u, v) and torch.equal(u, p)


@pytest.mark.parametrize("linear", [ops.lora_linear, lora_linear_autograd])
def test_a_tangent_on_the_gradient_is_refused_not_dropped(linear):
    x, w, a, b = _operands(torch.float32)
    leaves = [t.requires_grad_() for t in (x, a, b)]
    y = linear(x, w, a, b, 0.5)
    with torch.autograd.forward_ad.dual_level():
        dy = torch.autograd.forward_ad.make_dual(torch.ones_like(y), torch.ones_like(y))
        with pytest.raises(NotImplementedError, match="forward AD"):
            torch.autograd.grad(y, leaves, dy)
