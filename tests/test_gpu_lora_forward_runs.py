"""The few-row and tiled bf16 LoRA kernels (cf_lora_forward with a workspace)
run more than once: the same bits every time, in a captured graph replayed on
new inputs, and on two streams at once with a workspace each. Every result is
compared bit for bit with a call of its own on the same inputs."""

from __future__ import annotations

import pytest
import torch

from cuda_force_amd import _lib

from . import gpu_util as g

pytestmark = pytest.mark.gpu

SHAPES = [
    (4, 4096, 4096, 16),      # few rows, K in slices
    (64, 1000, 504, 12),      # few rows, element loads of a
    (100, 4096, 4096, 16),    # every tile split
    (333, 4096, 11008, 16),   # a round of whole tiles, the rest split
    (300, 4096, 4096, 64),    # two adapter steps, in the first slice
]


class _Call:
    def __init__(self, shape, seed):
        m, k, n, r = self.shape = shape
        gen = torch.Generator(device="cuda").manual_seed(seed)
        self.inputs = [(s * torch.randn(d, generator=gen, device="cuda")).bfloat16()
                       for s, d in ((1.0, (m, k)), (0.02, (k, n)), (1 / 64, (k, r)), (0.02, (r, n)))]
        self.y = g.empty((m, n), torch.bfloat16)
        self.xa = g.empty((m, r), torch.float32)
        self.bytes = g.lib().cf_lora_forward_workspace_bytes(_lib.CF_BF16, m, k, n, r)
        self.workspace = torch.full((self.bytes,), 0xFF, dtype=torch.uint8, device="cuda")

    def launch(self):
        m, k, n, r = self.shape
        x, w, a, b = (t.data_ptr() for t in self.inputs)
        g.call("cf_lora_forward", x, w, a, b, self.y.data_ptr(), self.xa.data_ptr(), _lib.CF_BF16, m, k, n, r, 1.5,
               self.workspace.data_ptr(), self.bytes, torch.cuda.current_stream().cuda_stream)

    def result(self):
        self.launch()
        torch.cuda.synchronize()
        return self.y.clone(), self.xa.clone()


def _same(got, want):
    return all(torch.equal(u, v) for u, v in zip(got, want))


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_repeats_and_replays_are_bit_equal(shape):
    g.announce(f"LoRA forward {shape}: repeats and a captured graph")
    call = _Call(shape, 1)
    first = call.result()
    for _ in range(3):
        assert _same(call.result(), first)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call.launch()
    for seed in (2, 3, 4):
        other = _Call(shape, seed)
        want = other.result()
        for t, v in zip(call.inputs, other.inputs):
            t.copy_(v)
        call.y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert _same((call.y, call.xa), want), seed


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_two_streams_with_a_workspace_each(shape):
    g.announce(f"LoRA forward {shape}: two streams")
    calls = [_Call(shape, seed) for seed in (5, 6)]
    want = [call.result() for call in calls]
    for call in calls:
        call.y.zero_()
        call.xa.zero_()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in calls]
    for _ in range(8):
        for stream, call in zip(streams, calls):
            with torch.cuda.stream(stream):
                call.launch()
    torch.cuda.synchronize()
    for call, expected in zip(calls, want):
        assert _same((call.y, call.xa), expected)
