"""The few-row bf16 LoRA kernels (cf_lora_forward with at most 64 rows)
against the float64 oracle: one row to 64, every 16-row block count, widths
of part strips (128 columns) and part blocks (32 k), ranks that are and are
not multiples of 8 (vector and element loads of a), rank 0, one slice and
many, a poisoned workspace. The tolerance is that of the other bf16 LoRA
tests (bf16 output rounding 2^-9 relative, a floor for cancelling sums)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from cuda_force_amd import _lib

from . import gpu_util as g
from .test_gpu_lora import assert_gemm_close, make_operands

pytestmark = pytest.mark.gpu


def run_forward(x, w, a, b, scale):
    m, k = x.shape
    n, r = w.shape[1], a.shape[1]
    t = [g.to_gpu(v, "bf16") for v in (x, w, a, b)]
    y = g.empty((m, n), torch.bfloat16)
    xa = g.empty((m, max(r, 1)), torch.float32)
    nbytes = g.lib().cf_lora_forward_workspace_bytes(_lib.CF_BF16, m, k, n, r)
    ws = g.empty(max(nbytes, 16), torch.uint8)
    g.call("cf_lora_forward", t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr() if r else None,
           t[3].data_ptr() if r else None, y.data_ptr(), xa.data_ptr(), _lib.CF_BF16, m, k, n, r, scale,
           ws.data_ptr(), nbytes, g.stream())
    torch.cuda.synchronize()
    return g.to_host(y), g.to_host(xa)


@pytest.mark.parametrize("shape", [
    (1, 8, 8, 1), (1, 4096, 4096, 16), (4, 688, 256, 16), (15, 32, 128, 8), (16, 40, 136, 4), (17, 1000, 504, 12),
    (32, 512, 11008, 32), (33, 5120, 512, 8), (48, 264, 2056, 64), (63, 2048, 120, 136), (64, 4096, 1024, 16),
    (64, 128, 128, 7),
], ids=str)
@pytest.mark.parametrize("scale", [2.0, 16 / 12])
def test_few_rows_match_the_oracle(shape, scale):
    m, k, n, r = shape
    g.announce(f"few-row LoRA bf16 {shape} scale {scale:.3f}")
    x, w, a, b = make_operands(m, k, n, r, "bf16", seed=sum(shape))
    y, xa = run_forward(x, w, a, b, scale)
    xv, wv, av, bv = (g.host_values(t, "bf16") for t in (x, w, a, b))
    assert_gemm_close(y, oracle.lora_linear(xv, wv, av, bv, scale, True), "bf16", f"{shape}")
    np.testing.assert_allclose(xa, xv.astype(np.float64) @ av, rtol=1e-4, atol=1e-5 * np.abs(xv).sum(1).max())


def test_rank_zero_and_row_independence():
    """Rank 0 is x @ w, and an infinity or NaN in one row of x stays in that
    row (rows past M and k past K read as zeros, never as a neighbour)."""
    m, k, n = 5, 200, 264
    x, w, a, b = make_operands(m, k, n, 8, "bf16", seed=7)
    y, _ = run_forward(x, w, a[:, :0], b[:0], 1.0)
    exact = g.host_values(x, "bf16").astype(np.float64) @ g.host_values(w, "bf16")
    assert_gemm_close(y, exact, "bf16", "rank 0")
    x2 = x.copy()
    x2[3, k - 1] = 0x7F80
    x2[4, 0] = 0x7FC0
    y2, _ = run_forward(x2, w, a[:, :0], b[:0], 1.0)
    np.testing.assert_array_equal(y2[:3], y[:3])
    assert not np.isfinite(g.host_values(y2, "bf16")[3:]).any()
