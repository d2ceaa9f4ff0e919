"""The bf16 adapter backward above rank 16 (rank blocks of 16, b in LDS) and
its row tiles of 128, 256 and 512 rows, against the float64 oracle: ranks at
and off the block edges, tiles of different heights in the dy and x passes
(rows past M between them), ragged rows and columns, poisoned workspace; the
same for fp32, and problems whose dy @ b^T is formed in several parts."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle

from . import gpu_util as g
from .test_gpu_lora import assert_gemm_close, rng, run_backward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    (1, 8, 8, 17), (100, 64, 11008, 32), (130, 11008, 72, 33), (333, 4096, 264, 64), (700, 264, 4096, 48),
    (1000, 1032, 2048, 24), (2000, 4096, 4096, 64), (4096, 2048, 1024, 32), (64, 688, 256, 16), (520, 256, 4104, 5),
], ids=str)
def test_backward_ranks_and_row_tiles(shape):
    m, k, n, r = shape
    g.announce(f"adapter backward bf16 {shape}")
    gen = rng(sum(shape))
    x = g.storage_bits(gen.standard_normal((m, k)).astype(np.float32), "bf16")
    dy = g.storage_bits(gen.standard_normal((m, n)).astype(np.float32), "bf16")
    b = g.storage_bits((0.02 * gen.standard_normal((r, n))).astype(np.float32), "bf16")
    xa = (gen.standard_normal((m, r)) * 0.5).astype(np.float32)
    ga, gb = run_backward(x, dy, b, xa, "bf16", 0.5)
    exact_a, exact_b = oracle.lora_backward(
        g.host_values(x, "bf16"), g.host_values(dy, "bf16"), g.host_values(b, "bf16"), xa, 0.5, True)
    assert_gemm_close(ga, exact_a, "bf16", f"grad_a {shape}")
    assert_gemm_close(gb, exact_b, "bf16", f"grad_b {shape}")


@pytest.mark.parametrize("shape", [
    (1, 4, 4, 1), (31, 132, 68, 16), (33, 128, 4096, 17), (128, 4096, 260, 16), (511, 64, 192, 32), (512, 260, 132, 33),
    (700, 1024, 516, 64), (1025, 68, 64, 8), (4097, 2052, 1924, 17), (4353, 36, 260, 33),
], ids=str)
def test_fp32_backward_tiles(shape):
    """The fp32 MFMA backward: the three row tiles with remainders, part column
    tiles, every rank block count."""
    m, k, n, r = shape
    g.announce(f"adapter backward fp32 {shape}")
    gen = rng(sum(shape))
    x, dy, b, xa = (gen.standard_normal(s).astype(np.float32) for s in ((m, k), (m, n), (r, n), (m, r)))
    ga, gb = run_backward(x, dy, b, xa, "f32", 0.5)
    exact_a, exact_b = oracle.lora_backward(x, dy, b, xa, 0.5, False)
    # fp32 sums of up to 4096 products: 1e-5 of the result's scale.
    for got, exact in ((ga, exact_a), (gb, exact_b)):
        assert (np.abs(got - exact) <= 1e-5 * np.abs(exact) + 1e-5 * np.abs(exact).max()).all()


@pytest.mark.parametrize("dtype,shape", [("f32", (8500, 64, 8192, 64))])
def test_backward_in_several_panels_of_rows(dtype, shape):
    """More partials of dy @ b^T than are held at a time: panels of rows, the
    last one short, in a workspace of the size asked for (what lies behind it
    stays)."""
    m, k, n, r = shape
    g.announce(f"adapter backward in panels {dtype} {shape}")
    gen = torch.Generator(device="cuda").manual_seed(sum(shape))
    t = g.torch_dtype(dtype)
    x, dy, b = (torch.randn(s, generator=gen, device="cuda").to(t) for s in ((m, k), (m, n), (r, n)))
    xa = torch.randn(m, r, generator=gen, device="cuda")
    grad_a, grad_b = g.empty((k, r), t), g.empty((r, n), t)
    nbytes = g.lib().cf_lora_backward_dtype_workspace_bytes(g.cf(dtype), m, k, n, r)
    ws = torch.full((nbytes + 4096,), 0xFF, dtype=torch.uint8, device="cuda")
    g.call("cf_lora_backward", x.data_ptr(), dy.data_ptr(), b.data_ptr(), xa.data_ptr(), grad_a.data_ptr(),
           grad_b.data_ptr(), g.cf(dtype), m, k, n, r, 0.5, ws.data_ptr(), nbytes, g.stream())
    assert bool((ws[nbytes:] == 0xFF).all())
    # grad_b in float64 by columns, which keeps the copies small.
    exact_g = sum(dy[:, i:i + 1024].double() @ b[:, i:i + 1024].double().t() for i in range(0, n, 1024))
    exact_b = torch.cat([xa.double().t() @ dy[:, i:i + 1024].double() for i in range(0, n, 1024)], dim=1)
    for got, exact in ((grad_a, x.double().t() @ exact_g), (grad_b, exact_b)):
        # fp32 sums of 8500 products, of factors that are sums of 8192.
        err = (got.double() - 0.5 * exact).abs()
        assert bool((err <= 2e-5 * exact.abs().max()).all()), f"max err {(err.max() / exact.abs().max()).item():.2e}"
