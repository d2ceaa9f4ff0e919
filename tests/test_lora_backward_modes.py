"""The backward of the LoRA linear when it is called inside autocast (the same
gradients, in the operands' dtype) and with batched gradients."""

from __future__ import annotations

import pytest
import torch

import cuda_force_amd.ops  # noqa: F401  (loads torch.ops.cudaforge)
from cuda_force_amd.autograd import lora_linear_autograd

K = torch.ops.cudaforge


def _operands(dtype):
    gen = torch.Generator().manual_seed(0)
    return [torch.randn(s, generator=gen).to(dtype) for s in ((7, 24), (24, 16), (24, 3), (3, 16))]


@pytest.mark.parametrize("dtype,auto", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float16)])
def test_input_gradient_keeps_its_dtype_under_autocast(dtype, auto):
    x, w, a, b = _operands(dtype)
    dy = torch.ones(7, 16, dtype=dtype)
    xa = x.float() @ a.float()
    want = K.lora_linear_bwd_input(x, dy, w, a, b, xa, 0.5)
    with torch.autocast("cpu", dtype=auto):
        got = K.lora_linear_bwd_input(x, dy, w, a, b, xa, 0.5)
    for u, v in zip(got, want):
        assert u.dtype == dtype
        assert torch.equal(u, v)


def test_backward_inside_autocast_equals_the_one_outside():
    operands = _operands(torch.float32)
    grads = []
    for inside in (False, True):
        x, w, a, b = (t.clone() for t in operands)
        leaves = [x.requires_grad_(), a.requires_grad_(), b.requires_grad_()]
        y = lora_linear_autograd(x, w, a, b, 0.5)
        with torch.autocast("cpu", dtype=torch.bfloat16, enabled=inside):
            grads.append(torch.autograd.grad(y.square().sum(), leaves))
    for u, v in zip(*grads):
        assert torch.equal(u, v)


def test_batched_gradients_equal_one_at_a_time():
    x, w, a, b = _operands(torch.float32)
    leaves = [x.requires_grad_(), a.requires_grad_(), b.requires_grad_()]
    y = lora_linear_autograd(x, w, a, b, 0.5)
    dy = torch.randn(3, 7, 16, generator=torch.Generator().manual_seed(1))
    batched = torch.autograd.grad(y, leaves, dy, is_grads_batched=True, retain_graph=True)
    singly = [torch.autograd.grad(y, leaves, row, retain_graph=True) for row in dy]
    for got, want in zip(batched, (torch.stack(t) for t in zip(*singly))):
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-5)
