"""The input gradient of the LoRA linear on the training path (the plain GEMM
plus the adapter's part added in place by the HIP kernels) against float64:
every rank block count, ranks with and without whole 16-byte rows of a, row
and column remainders, the plain kernel (fp32, odd widths, rank above 64) and
the sizes at which a GEMM takes its place,
infinite gradients, more rows than one launch takes, and the composed path a
recorded backward takes."""

from __future__ import annotations

import pytest
import torch

from cuda_force_amd import ops

from . import gpu_util as g

pytestmark = pytest.mark.gpu


def _operands(m, k, n, r, dtype, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    w = (0.02 * torch.randn(k, n, generator=gen, device="cuda")).to(dtype)
    a = (torch.randn(k, r, generator=gen, device="cuda") / 8).to(dtype)
    b = (0.1 * torch.randn(r, n, generator=gen, device="cuda")).to(dtype)
    dy = torch.randn(m, n, generator=gen, device="cuda").to(dtype)
    return x, w, a, b, dy


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [
    (1, 8, 16, 1), (17, 264, 72, 4), (64, 256, 256, 16), (130, 520, 264, 24), (333, 688, 1024, 64), (65, 48, 40, 7),
    (100, 130, 70, 5), (40, 256, 136, 100), (1100, 520, 264, 24), (300, 1001, 130, 70),
], ids=str)
def test_input_gradient_matches_float64(dtype, shape):
    m, k, n, r = shape
    g.announce(f"LoRA input gradient {dtype} {shape}")
    x, w, a, b, dy = _operands(m, k, n, r, dtype, sum(shape))
    leaves = [t.clone().requires_grad_() for t in (x, a, b)]
    y = ops.lora_linear(leaves[0], w, leaves[1], leaves[2], 1.5)
    grad_x, grad_a, grad_b = torch.autograd.grad(y, leaves, dy)
    xd, wd, ad, bd, dyd = (t.double() for t in (x, w, a, b, dy))
    gd = dyd @ bd.t()
    want = {"grad_x": dyd @ wd.t() + 1.5 * (gd @ ad.t()), "grad_a": 1.5 * (xd.t() @ gd),
            "grad_b": 1.5 * ((xd @ ad).t() @ dyd)}
    # bf16: the GEMM's result, dy @ b^T and the sum are each rounded once
    # (2^-9 relative each); fp32: sums of up to 1024 products.
    rel, floor = (1e-2, 4e-3) if dtype == torch.bfloat16 else (1e-4, 2e-5)
    for name, got in (("grad_x", grad_x), ("grad_a", grad_a), ("grad_b", grad_b)):
        err = (got.double() - want[name]).abs()
        bound = rel * want[name].abs() + floor * want[name].abs().max()
        assert bool((err <= bound).all()), f"{name}: max err {err.max().item():.3e}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rank", [1, 5, 16, 17, 40, 64, 70])
def test_infinite_gradients_stay_infinite(dtype, rank):
    """dy = +-inf at a column where w, a and b are positive: every term of that
    row of grad_x is the same infinity (ranks that the kernels pad included),
    and the other rows are the ones without it."""
    g.announce(f"LoRA input gradient with infinities {dtype} rank {rank}")
    x, w, a, b, dy = _operands(70, 264, 72, rank, dtype, rank)
    w[:, 5].abs_()
    b[:, 5].abs_().clamp_(min=1e-3)
    a.abs_().clamp_(min=1e-3)
    plain = None
    for mark in (False, True):
        if mark:
            dy[3, 5], dy[64, 5] = float("inf"), float("-inf")
        leaves = [t.clone().requires_grad_() for t in (x, a, b)]
        grad_x, _, _ = torch.autograd.grad(ops.lora_linear(leaves[0], w, leaves[1], leaves[2], 1.5), leaves, dy)
        if mark:
            assert bool((grad_x[3] == float("inf")).all()) and bool((grad_x[64] == float("-inf")).all())
            rest = [i for i in range(70) if i not in (3, 64)]
            assert torch.equal(grad_x[rest], plain[rest])
        plain = grad_x


@pytest.mark.parametrize("dtype,rows,n", [(torch.float32, 524_289, 8), (torch.float32, 524_289, 6),
                                          (torch.bfloat16, 1_048_577, 8), (torch.bfloat16, 524_289, 6)])
def test_more_rows_than_one_launch_of_the_update_takes(dtype, rows, n):
    """16 or 8 rows a workgroup and 65535 workgroups in y: one row more than
    that, on each kernel (widths that are not whole vectors take the plain
    one)."""
    g.announce(f"LoRA input gradient {dtype} {rows} rows, {n} columns")
    x, w, a, b, dy = _operands(rows, 8, n, 2, dtype, rows)
    leaves = [t.clone().requires_grad_() for t in (x, a, b)]
    grads = torch.autograd.grad(ops.lora_linear(leaves[0], w, leaves[1], leaves[2], 1.5), leaves, dy)
    for at in (slice(0, 64), slice(rows - 64, rows)):
        want = dy[at].double() @ (w.double() + 1.5 * (a.double() @ b.double())).t()
        rel, floor = (1e-2, 4e-3) if dtype == torch.bfloat16 else (1e-4, 2e-5)
        err = (grads[0][at].double() - want).abs()
        assert bool((err <= rel * want.abs() + floor * want.abs().max()).all())


def test_a_recorded_backward_can_be_differentiated_again():
    """create_graph: grad_x stays a differentiable composition (here in dy)."""
    x, w, a, b, dy = _operands(32, 64, 48, 8, torch.float32, 3)
    x.requires_grad_()
    dy.requires_grad_()
    y = ops.lora_linear(x, w, a, b, 2.0)
    (grad_x,) = torch.autograd.grad(y, x, dy, create_graph=True)
    (second,) = torch.autograd.grad(grad_x.sum(), dy)
    full = w + 2.0 * (a @ b)
    torch.testing.assert_close(second, full.sum(0).expand_as(dy), rtol=1e-4, atol=1e-4)
