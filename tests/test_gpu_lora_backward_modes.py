"""The LoRA linear's backward inside autocast on the GPU: the gradients of the
backward outside it, in the operands' dtype, by the native node and by the
Python function."""

from __future__ import annotations

import pytest
import torch

from cuda_force_amd import ops
from cuda_force_amd.autograd import lora_linear_autograd

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
