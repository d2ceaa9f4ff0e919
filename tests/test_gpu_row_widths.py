"""Row operators at the widths where their kernels change: ragged softmax rows
(three passes up to 383 or 511 columns, an element per lane above: the edges of
its sizes and one past the last), aligned rows of a workgroup each, with and
without the causal mask and in place, fp32 results on both sides of the size
from which their stores merge, and RMSNorm rows of a workgroup each (few rows,
and more than eight vectors per lane, on both sides of where a wave holds them). Against float64 at the tolerances of test_gpu_rowops:
1e-5 relative for fp32 results, 1e-2 for 16-bit ones."""

from __future__ import annotations

import pytest
import torch

from cuda_force_amd import ops

from . import gpu_util as g

pytestmark = pytest.mark.gpu

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _close(got, exact, dtype, what):
    rel, floor = (1e-5, 1e-7) if dtype == torch.float32 else (1e-2, 1e-6)
    bad = ~((got.double() - exact).abs() <= rel * exact.abs() + floor)
    assert not bool(bad.any()), f"{what}: {int(bad.sum())} out of tolerance"


def _normal(rows, cols, dtype, seed, std=1.0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (std * torch.randn(rows, cols, generator=gen, device="cuda")).to(dtype)


@pytest.mark.parametrize("src,dst", [("f32", "f32"), ("bf16", "f32"), ("bf16", "bf16"), ("f16", "f32"), ("f32", "f16")])
@pytest.mark.parametrize("cols", [1, 63, 257, 383, 385, 511, 513, 4095, 4097, 8191, 8193, 16383, 16385, 32767, 32769, 50257, 65535, 65537, 8200, 16384, 32000])
def test_softmax_widths(src, dst, cols):
    g.announce(f"softmax width {cols} {src} -> {dst}")
    x = _normal(5, cols, DTYPES[src], cols, 2.0)
    y = ops.softmax_as(x, DTYPES[dst])
    _close(y, torch.softmax(x.double(), -1), DTYPES[dst], f"{cols} {src}->{dst}")
    y = ops.softmax_scaled(x, 0.5, 3, DTYPES[dst])
    keep = torch.arange(cols, device="cuda")[None] <= (torch.arange(5, device="cuda") % 3)[:, None]
    exact = torch.softmax((0.5 * x.double()).masked_fill(~keep, float("-inf")), -1)
    _close(y, exact, DTYPES[dst], f"masked {cols} {src}->{dst}")


@pytest.mark.parametrize("rows,cols", [(229, 32000), (230, 32000), (224, 32768), (225, 32768), (112, 65536), (113, 65536)])
def test_fp32_results_on_both_sides_of_28_mib(rows, cols):
    """16-bit rows to fp32: streaming stores below, merged ones above, whole
    register rows and part ones."""
    g.announce(f"softmax [{rows}, {cols}] bf16 -> f32")
    x = _normal(rows, cols, torch.bfloat16, rows, 2.0)
    _close(ops.softmax_as(x, torch.float32), torch.softmax(x.double(), -1), torch.float32, f"{rows} x {cols}")


def test_ragged_softmax_unaligned_and_in_place():
    base = _normal(1, 1 + 7 * 4099, torch.bfloat16, 3)
    x = base.view(-1)[1:].view(7, 4099)  # rows start two bytes off, widths are odd
    exact = torch.softmax(x.double(), -1)
    y = g.poison_like(x.contiguous())
    g.call("cf_softmax", x.data_ptr(), g.cf("bf16"), y.data_ptr(), g.cf("bf16"), 7, 4099, g.stream())
    _close(y, exact, torch.bfloat16, "unaligned")
    g.call("cf_softmax", x.data_ptr(), g.cf("bf16"), x.data_ptr(), g.cf("bf16"), 7, 4099, g.stream())
    _close(x, exact, torch.bfloat16, "in place")
    rows = torch.full((2, 4097), float("-inf"), device="cuda")
    rows[1, 4096] = 3.0
    y = ops.softmax(rows)
    assert bool(torch.isnan(y[0]).all()) and y[1, 4096] == 1 and y[1, :4096].abs().max() == 0


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", [(1, 2056), (4, 4096), (256, 4104), (257, 4104), (300, 5120), (40, 8192), (300, 2560),
                                   (3, 16384), (700, 6712), (5, 32768), (3, 18440), (1536, 4096), (1535, 8192),
                                   (1540, 8192), (513, 4096), (2049, 4096), (1600, 5120), (1700, 10240)], ids=str)
def test_rmsnorm_row_workgroups(dtype, shape):
    rows, cols = shape
    g.announce(f"RMSNorm row workgroups {dtype} {shape}")
    t = DTYPES[dtype]
    x, r = _normal(rows, cols, t, 1), _normal(rows, cols, t, 2)
    w = (1 + _normal(1, cols, torch.float32, 3, 0.02)).view(-1).to(t)

    def norm(v):
        return v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()

    _close(ops.rmsnorm(x, w), norm(x.double()), t, "rmsnorm")
    y, h = ops.fused_residual_rmsnorm(x, r, w)
    assert torch.equal(h, x + r)
    _close(y, norm(h.double()), t, "fused residual")
    x[0, -1] = float("nan")
    y = ops.rmsnorm(x, w)
    assert bool(torch.isnan(y[0]).all()) and (rows == 1 or bool(torch.isfinite(y[1:].float()).all()))
