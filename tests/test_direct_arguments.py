"""Arguments that the direct entry of ops.py does not read (scales that are
tensors, dtypes that are not torch's) reach the general way, and a
differentiable call is still one graph for torch.compile."""

from __future__ import annotations

import pytest
import torch

from cuda_force_amd import ops


def test_scale_per_column_reaches_the_composition():
    gen = torch.Generator().manual_seed(0)
    x, w, a, b = (torch.randn(s, generator=gen) for s in ((4, 8), (8, 6), (8, 2), (2, 6)))
    scale = torch.arange(6.0)
    y = ops.lora_linear(x, w, a.clone().requires_grad_(), b, scale)
    torch.testing.assert_close(y, x @ w + scale * ((x @ a) @ b))


def test_python_float_is_a_dtype_as_torch_has_it():
    assert ops.softmax_as(torch.ones(2, 3), float).dtype == torch.float64


@pytest.mark.parametrize("op", ["rmsnorm", "softmax", "silu", "lora_linear"])
def test_differentiable_calls_compile_to_one_graph(op):
    gen = torch.Generator().manual_seed(1)
    x, w, a, b = (torch.randn(s, generator=gen) for s in ((4, 8), (8, 6), (8, 2), (2, 6)))
    rest = {"rmsnorm": (torch.ones(8),), "lora_linear": (w, a, b, 2.0)}.get(op, ())
    fn = getattr(ops, op)
    x.requires_grad_()
    compiled = torch.compile(lambda t: fn(t, *rest) * 2, backend="eager", fullgraph=True)
    torch.testing.assert_close(compiled(x), fn(x, *rest) * 2)
