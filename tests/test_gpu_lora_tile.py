"""The tiled bf16 LoRA kernels (cf_lora_forward above 64 rows) against the
float64 oracle: each tile shape with part tiles in both directions, K not a
multiple of the K-step, one K-step and fewer than the stages, ranks whose
rows are 16-byte pieces, pairs and single elements, adapter parts that fill
K-steps exactly and that do not, several slices, whole tiles, split tiles and
both. The tolerance is that of the other bf16 LoRA tests (one bf16
rounding 2^-9 relative, a floor for cancelling sums)."""

from __future__ import annotations

import numpy as np
import pytest

import oracle

from . import gpu_util as g
from .test_gpu_lora import assert_gemm_close, make_operands
from .test_gpu_lora_skinny import run_forward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    (65, 8, 8, 1), (65, 32, 128, 32), (100, 4096, 4096, 16), (128, 1024, 1024, 32), (129, 688, 264, 6),
    (300, 1000, 520, 7), (333, 4096, 11008, 16), (513, 264, 4096, 100), (700, 72, 136, 128), (1000, 2048, 4096, 64),
    (2100, 136, 4104, 24), (5000, 1000, 1032, 64), (90, 16, 4096, 128), (66, 544, 2048, 48),
], ids=str)
@pytest.mark.parametrize("scale", [2.0, 16 / 12])
def test_tiles_match_the_oracle(shape, scale):
    m, k, n, r = shape
    g.announce(f"tiled LoRA bf16 {shape} scale {scale:.3f}")
    x, w, a, b = make_operands(m, k, n, r, "bf16", seed=sum(shape))
    y, xa = run_forward(x, w, a, b, scale)
    xv, wv, av, bv = (g.host_values(t, "bf16") for t in (x, w, a, b))
    assert_gemm_close(y, oracle.lora_linear(xv, wv, av, bv, scale, True), "bf16", f"{shape}")
    np.testing.assert_allclose(xa, xv.astype(np.float64) @ av, rtol=1e-4, atol=1e-5 * np.abs(xv).sum(1).max())


def test_rank_zero_and_row_independence():
    """Rank 0 is x @ w; an infinity or NaN in a row of x stays in that row
    (k past K and rows past M read as zeros)."""
    m, k, n = 150, 200, 264
    x, w, a, b = make_operands(m, k, n, 24, "bf16", seed=9)
    y, _ = run_forward(x, w, a[:, :0], b[:0], 1.0)
    exact = g.host_values(x, "bf16").astype(np.float64) @ g.host_values(w, "bf16")
    assert_gemm_close(y, exact, "bf16", "rank 0")
    x2 = x.copy()
    x2[17, k - 1] = 0x7F80
    x2[149, 0] = 0x7FC0
    y2, _ = run_forward(x2, w, a[:, :0], b[:0], 1.0)
    keep = np.ones(m, dtype=bool)
    keep[[17, 149]] = False
    np.testing.assert_array_equal(y2[keep], y[keep])
    assert not np.isfinite(g.host_values(y2, "bf16")[~keep]).any()


@pytest.mark.parametrize("scale", [2.0, 1.7])
def test_infinite_adapter_intermediate(scale):
    """x @ a overflows to infinity in one row: the row is +-inf by the sign of
    b, as in fp32 arithmetic, and the other rows are zero."""
    m, k, n, r = 100, 64, 136, 16
    x, w, a, b = (np.zeros_like(t) for t in make_operands(m, k, n, r, "bf16", seed=1))
    b = make_operands(m, k, n, r, "bf16", seed=2)[3]
    x[5, 3] = 0x7F00  # 1.7e38; its square is past fp32
    a[3, 0] = 0x7F00
    y, xa = run_forward(x, w, a, b, scale)
    got = g.host_values(y, "bf16")
    assert np.isposinf(xa[5, 0])
    np.testing.assert_array_equal(got[5], np.where(g.host_values(b, "bf16")[0] > 0, np.inf, -np.inf))
    assert (np.delete(got, 5, axis=0) == 0).all()


@pytest.mark.parametrize("scale", [2.0, 0.25, 1.7])
@pytest.mark.parametrize("shape", [(100, 64, 136, 24), (300, 4096, 264, 40), (2100, 520, 136, 7)], ids=str)
def test_infinite_b_and_a_scaled_b_past_bf16(shape, scale):
    """scale * (u @ b) in fp32: an infinite b gives +-inf by the sign of u, and a
    b whose product with the scale is past the largest bf16 gives the finite
    value it has with a small u."""
    m, k, n, r = shape
    g.announce(f"tiled LoRA with infinite and largest b {shape} scale {scale}")
    x, w, a, b = make_operands(m, k, n, r, "bf16", seed=sum(shape))
    w = np.zeros_like(w)
    b[:, 3] = 0
    b[r - 1, 3] = 0x7F80  # inf
    b[:, 5] = 0
    b[0, 5] = 0x7F7F      # 3.39e38, the largest bf16
    x, a = x & 0x7FFF, a & 0x7FFF
    x[::2] |= 0x8000      # rows of either sign
    a = (0x3000 + (a & 0x7F)).astype(np.uint16)  # 2^-31 .. 2^-30: 2 u max(b) is finite
    y, xa = run_forward(x, w, a, b, scale)
    got = g.host_values(y, "bf16")
    u = g.host_values(g.storage_bits(xa, "bf16"), "bf16").astype(np.float64)
    assert (u != 0).all()
    np.testing.assert_array_equal(got[:, 3], np.where(u[:, r - 1] > 0, np.inf, -np.inf))
    np.testing.assert_allclose(got[:, 5], scale * u[:, 0] * g.host_values(b, "bf16")[0, 5], rtol=2.0**-8)
    rest = [i for i in range(n) if i not in (3, 5)]
    assert np.isfinite(got[:, rest]).all()
