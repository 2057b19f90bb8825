"""The HIP linear layer under torch.compile and torch.export with dynamic
shapes, traced without a GPU: the choice between the products is left to the
gemm op, whose implementation falls back to the framework's product on the
CPU.
"""
from __future__ import annotations

import pytest
import torch
import torch.nn as nn

from mamba_metal_scan_amd import _native, linear as linear_mod

# 2^30 multiply-adds lie at 4096 rows of a 512 x 512 layer.
WIDTH = 512


@pytest.fixture
def layer(monkeypatch):
    """A layer whose CPU tensors pass for ROCm ones while it is traced."""
    monkeypatch.setattr(linear_mod, "_hip_device", lambda t: True)
    monkeypatch.setattr(_native, "_on_one_device", lambda what, *ts: None)
    torch._dynamo.reset()
    torch.manual_seed(0)

    class Layer(nn.Module):
        def __init__(self):
            super().__init__()
            self.proj = nn.Linear(WIDTH, WIDTH, bias=False)

        def forward(self, x):
            return linear_mod.linear(self.proj, x)
    yield Layer()
    torch._dynamo.reset()


def _ops(graph):
    return [str(n.target) for n in graph.nodes if n.op == "call_function"]


@pytest.mark.parametrize("dynamic", [None, True])
def test_compiled_at_changing_batches(layer, dynamic):
    graphs = []

    def backend(gm, example):
        graphs.append(gm)
        return gm.forward
    f = torch.compile(layer, backend=backend, dynamic=dynamic, fullgraph=True)
    for rows in (2, 3, 9, 4097):
        x = torch.randn(rows, 1, WIDTH, requires_grad=True)
        y = f(x)
        want = layer.proj(x)
        torch.testing.assert_close(y, want)
        got = torch.autograd.grad(y.square().sum(), (x, layer.proj.weight))
        for a, b in zip(got, torch.autograd.grad(want.square().sum(), (x, layer.proj.weight))):
            torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4)
    assert len(graphs) <= 2   # one, and one more for the symbolic batch


def test_static_sizes_choose_while_tracing(layer):
    """Fixed sizes below the line keep the framework's call in the graph, above
    it the op (traced without gradients, which would wrap it)."""
    for rows, op in ((64, False), (4096, True)):
        torch._dynamo.reset()
        graphs = []

        def backend(gm, example):
            graphs.append(gm)
            return gm.forward
        with torch.no_grad():
            torch.compile(layer, backend=backend, dynamic=False, fullgraph=True)(
                torch.zeros(rows, WIDTH))
        code = "\n".join(m.code for m in graphs[0].modules() if hasattr(m, "code"))
        assert ("mamba_hip.gemm" in code) == op, code


@pytest.mark.parametrize("strict", [True, False])
def test_exported_with_a_dynamic_batch(layer, strict):
    with torch.no_grad():
        ep = torch.export.export(layer, (torch.randn(4, WIDTH),), strict=strict,
                                 dynamic_shapes={"x": {0: torch.export.Dim("batch")}})
        for rows in (1, 4, 9):
            x = torch.randn(rows, WIDTH)
            torch.testing.assert_close(ep.module()(x), layer.proj(x))
