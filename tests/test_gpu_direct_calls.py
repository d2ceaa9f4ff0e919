"""The direct entry of ops.py for ordinary GPU calls: the same bits as the
dispatcher's operators, and the general way for everything else (gradients,
subclasses, function modes, autocast, profiling, strided or empty inputs,
mixed dtypes), with the LoRA autograd node under saved-tensor hooks."""

from __future__ import annotations

import pytest
import torch

from cuda_force_amd import ops
from torch.overrides import TorchFunctionMode

from . import gpu_util as g

pytestmark = pytest.mark.gpu

K = torch.ops.cudaforge


def _rand(*shape, dtype=torch.bfloat16, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, generator=gen, device="cuda").to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_direct_calls_equal_the_dispatcher(dtype):
    g.announce(f"direct calls against torch.ops.cudaforge, {dtype}")
    x, r, w = _rand(3, 5, 264, dtype=dtype), _rand(15, 264, dtype=dtype, seed=1), _rand(264, dtype=dtype, seed=2)
    rows = x.view(15, 264)
    pairs = [
        (ops.rmsnorm(x, w, 1e-5), K.rmsnorm(rows, w, 1e-5).view_as(x)),
        (ops.softmax(x), K.softmax(rows).view_as(x)),
        (ops.softmax_as(x, torch.float32), K.softmax_as(rows, torch.float32).view_as(x)),
        (ops.softmax_scaled(x, 0.5, 5), K.softmax_scaled(rows, 0.5, 5, dtype).view_as(x)),
        (ops.silu(x), K.silu(x)), (ops.gelu(x), K.gelu(x)), (ops.swiglu(rows, r), K.swiglu(rows, r)),
    ]
    pairs += list(zip(ops.fused_residual_rmsnorm(rows, r, w, 1e-5), K.fused_residual_rmsnorm(rows, r, w, 1e-5)))
    q, s = ops.quantize_int8(x)
    pairs += list(zip((q, s), K.quantize_int8(x)))
    pairs += [(ops.dequantize_int8(q, s), K.dequantize_int8(q, s)),
              (ops.dequantize_int8(q, s, dtype), K.dequantize_int8_to(q, s, dtype))]
    if dtype != torch.float16:
        a, b, wt = _rand(264, 8, dtype=dtype), _rand(8, 40, dtype=dtype), _rand(264, 40, dtype=dtype)
        pairs.append((ops.lora_linear(x, wt, a, b, 2.0), K.lora_linear(rows, wt, a, b, 2.0).view(3, 5, 40)))
    if dtype == torch.bfloat16:
        qr, kr = _rand(2, 16, 128, seed=5), _rand(2, 16, 128, seed=6)
        lower = torch.ones(16, 16, dtype=torch.bool, device="cuda").tril()
        scores = ops.attention_scores_causal(qr, kr, 2)
        pairs.append((scores[..., lower], K.attention_scores_causal(qr, kr, 2)[..., lower]))
        probs = ops.softmax_scaled(scores.view(-1, 16), 0.125, 16).view_as(scores)
        pairs.append((ops.attention_pv_causal(probs, qr, 2), K.attention_pv_causal(probs, qr, 2)))
    for i, (got, want) in enumerate(pairs):
        assert got.shape == want.shape and got.dtype == want.dtype, i
        assert torch.equal(got, want), i


def test_calls_that_are_not_ordinary_take_the_general_way():
    direct = ops._DIRECT
    x, w = _rand(6, 64), _rand(64, seed=1)
    assert direct.try_rmsnorm(x, w, 1e-6) is not None
    assert direct.try_rmsnorm(x, torch.nn.Parameter(w, requires_grad=False), 1e-6) is not None

    class Sub(torch.Tensor):
        pass

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for other in (x.as_subclass(Sub), x.t().contiguous().t(), x[:0], x.double(), x.cpu(), x.float(), x[:, :32]):
        assert direct.try_rmsnorm(other, w, 1e-6) is None
    assert direct.try_rmsnorm(x.clone().requires_grad_(), w, 1e-6) is None
    with torch.no_grad():
        assert direct.try_rmsnorm(x.clone().requires_grad_(), w, 1e-6) is not None
    with Mode():
        assert direct.try_rmsnorm(x, w, 1e-6) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert direct.try_rmsnorm(x, w, 1e-6) is None
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        assert direct.try_rmsnorm(x, w, 1e-6) is None
    seen = []
    torch.func.vmap(lambda row: seen.append(direct.try_softmax(row, None)) or row)(x)
    assert seen == [None]
    with pytest.raises(ValueError, match="does not match"):
        ops.rmsnorm(x, w[:32])
    y = ops.rmsnorm(x.clone().requires_grad_(), w)
    assert y.requires_grad


def test_lora_autograd_node_keeps_hooks_and_partial_gradients():
    x, w, a, b = _rand(70, 64), _rand(64, 40, seed=1), _rand(64, 8, seed=2), _rand(8, 40, seed=3)
    dy = _rand(70, 40, seed=4)
    leaves = [t.clone().requires_grad_() for t in (x, a, b)]
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        y = ops.lora_linear(leaves[0], w, leaves[1], leaves[2], 2.0)
    assert len(packed) == 5
    got = torch.autograd.grad(y, leaves, dy)
    plain = [t.clone().requires_grad_() for t in (x, a, b)]
    want = torch.autograd.grad(ops.lora_linear(plain[0], w, plain[1], plain[2], 2.0), plain, dy)
    for u, v in zip(got, want):
        assert torch.equal(u, v)
    # w alone, x alone, one adapter factor alone.
    for i in range(4):
        args = [t.clone() for t in (x, w, a, b)]
        args[i].requires_grad_()
        (grad,) = torch.autograd.grad(ops.lora_linear(*args, 2.0), args[i], dy)
        ref = [t.double() for t in (x, w, a, b)]
        ref[i].requires_grad_()
        (exact,) = torch.autograd.grad(ref[0] @ ref[1] + 2.0 * ((ref[0] @ ref[2]) @ ref[3]), ref[i], dy.double())
        # bf16 GEMMs and one rounded intermediate: 2^-7 of the largest value.
        assert (grad.double() - exact).abs().max() <= 2.0**-7 * exact.abs().max()


def test_arguments_the_direct_entry_does_not_read():
    direct = ops._DIRECT
    x, w = _rand(6, 64), _rand(64, seed=1)
    for eps in (None, "1", True, 1j, 10**400, torch.tensor(1e-6), torch.ones(64)):
        assert direct.try_rmsnorm(x, w, eps) is None
    assert direct.try_rmsnorm(x, w, 0) is not None
    for dtype in (float, "float32", torch.float64, torch.int32):
        assert direct.try_softmax(x, dtype) is None
    for period in (True, 2**70, -1, 2.0):
        assert direct.try_softmax_scaled(x, 1.0, period, None) is None
    with pytest.raises(RuntimeError, match="Expected a value of type 'float'"):
        ops.rmsnorm(x, w, None)


def test_forward_mode_is_refused_not_dropped():
    with torch.autograd.forward_ad.dual_level():
        x = torch.autograd.forward_ad.make_dual(_rand(6, 64), _rand(6, 64, seed=1))
        with pytest.raises(NotImplementedError, match="forward AD"):
            ops.softmax(x)


def test_errors_keep_their_types():
    x = torch.zeros(1 << 24, device="cuda")
    used = torch.cuda.memory_reserved() / torch.cuda.get_device_properties(0).total_memory
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(min(1.0, used * 0.5), 0)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            kept = [ops.silu(x) for _ in range(64)]
            del kept
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, 0)

    class Stop(Exception):
        pass

    def pack(t):
        raise Stop

    operands = _rand(70, 64), _rand(64, 40, seed=1), _rand(64, 8, seed=2).requires_grad_(), _rand(8, 40, seed=3)
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t), pytest.raises(Stop):
        ops.lora_linear(*operands, 2.0)
