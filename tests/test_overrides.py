"""Modules whose forward (or, of a block, any method) is set on the instance,
as adapters, offloading and instrumentation do, and weights that are not plain
tensors: every path of the model that calls such a module runs its override,
and the native paths refuse it.
"""
from __future__ import annotations

import copy

import pytest
import torch
import torch.nn as nn

from helpers import assert_close
from mamba_metal_scan_amd.block import plain, plain_mods
from mamba_metal_scan_amd.linear import no_hooks
from mamba_metal_scan_amd.model import MambaBlock, MambaConfig, TinyMamba, _plain_block

DEV = "cuda"


def _model(vocab=203):
    torch.manual_seed(2)
    m = TinyMamba(MambaConfig(vocab_size=vocab, d_model=64, n_layers=2, d_ff=128,
                              scan_impl="hip"))
    with torch.no_grad():
        for b in m.blocks:
            b.dt_proj.bias.normal_()
            b.conv.bias.normal_()
    return m


# -------------------------------------------------------- the predicates (CPU)

def test_an_overridden_forward_is_not_plain():
    lin = nn.Linear(4, 4, bias=False)
    assert plain_mods((lin,), (nn.Linear,)) and no_hooks(lin)
    lin.forward = lambda x: x
    assert not plain_mods((lin,), (nn.Linear,)) and not no_hooks(lin)
    del lin.forward
    assert plain_mods((lin,), (nn.Linear,)) and no_hooks(lin)


@pytest.mark.parametrize("where", ["forward", "mix", "_step", "_scan", "norm.forward"])
def test_a_block_with_a_method_of_its_own_is_not_plain(where):
    block = _model().blocks[0]
    assert _plain_block(block)
    owner = block.norm if where.startswith("norm") else block
    setattr(owner, where.split(".")[-1], lambda *a, **k: None)
    assert not _plain_block(block)


class Doubled(torch.Tensor):
    """A wrapper without storage of its own: twice the tensor it holds, as a
    quantised weight inside a plain nn.Linear would be computed from its codes."""

    @staticmethod
    def __new__(cls, inner):
        return torch.Tensor._make_wrapper_subclass(cls, inner.shape, dtype=inner.dtype,
                                                   device=inner.device)

    def __init__(self, inner):
        self.inner = inner

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        if func is torch.ops.aten.detach.default:
            return cls(args[0].inner)
        args = torch.utils._pytree.tree_map_only(cls, lambda t: 2 * t.inner, args)
        return func(*args, **(kwargs or {}))


class Tagged(torch.Tensor):
    """A subclass with storage, whose operators double their results."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        out = super().__torch_function__(func, types, args, kwargs)
        return 2 * out.as_subclass(torch.Tensor) if func is torch.nn.functional.linear else out


def test_a_subclass_is_not_plain():
    t = torch.randn(4, 4)
    assert plain(t, t.device, t.shape) and plain(nn.Parameter(t), t.device, t.shape)
    assert not plain(Doubled(t), t.device, t.shape)
    assert not plain(t.as_subclass(Tagged), t.device, t.shape)
    assert not plain(None, t.device, t.shape)


# ------------------------------------------------------------- every path (GPU)

def _run(m, path, idx):
    """(logits, cache tensors) of one path over the tokens idx."""
    if path == "train":
        return (m(idx)[0],)
    with torch.no_grad():
        cache = {}
        logits = m(idx[:, :-1] if path == "token" else idx, cache=cache)[0]
        if path == "token":
            logits = m(idx[:, -1:], cache=cache)[0]
    return (logits, *[b[k] for b in cache["blocks"] for k in ("h", "conv")])


def _double(mod):
    """mod's forward set on the instance: twice the class's."""
    calls = []

    def forward(*args):
        calls.append(1)
        return 2 * type(mod).forward(mod, *args)
    mod.forward = forward
    return calls


# Training calls in_proj, out_proj and the head as modules, a prompt and a
# token the other projections too, a token the conv.
@pytest.mark.gpu
@pytest.mark.parametrize("path,name", [
    (p, n) for p, ns in (("train", "in_proj out_proj"),
                         ("prefill", "in_proj out_proj dt_proj B_proj C_proj"),
                         ("token", "in_proj out_proj dt_proj B_proj C_proj conv"))
    for n in ns.split()])
def test_child_forward_runs(path, name):
    print(f"[case] override {path} {name}", flush=True)
    m = _model().to(DEV)
    idx = torch.randint(0, 203, (3, 9), generator=torch.Generator().manual_seed(1)).to(DEV)
    want = copy.deepcopy(m)
    with torch.no_grad():
        for p in getattr(want.blocks[1], name).parameters():
            p.mul_(2)
    if path == "token":   # alone: both caches from the plain model's prompt
        plain = {}
        with torch.no_grad():
            m(idx[:, :-1], cache=plain)

        def step(model):
            cache = {"blocks": [{k: v.clone() for k, v in b.items()} for b in plain["blocks"]]}
            with torch.no_grad():
                logits = model(idx[:, -1:], cache=cache)[0]
            return (logits, *[b[k] for b in cache["blocks"] for k in ("h", "conv")])
        ref = step(want)
        calls = _double(getattr(m.blocks[1], name))
        got = step(m)
    else:
        ref = _run(want, path, idx)
        calls = _double(getattr(m.blocks[1], name))
        got = _run(m, path, idx)
    torch.cuda.synchronize()
    assert calls == [1]
    for i, (a, b) in enumerate(zip(got, ref)):
        assert_close(f"output {i}", a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["train", "prefill", "token"])
def test_head_and_norm_forward_run(path):
    """The head at a size the HIP product would take (512 x 32768 x 64)."""
    print(f"[case] override head, norms {path}", flush=True)
    m = _model(vocab=32768).to(DEV)
    idx = torch.randint(0, 32768, (4, 128), generator=torch.Generator().manual_seed(1)).to(DEV)
    m.head.forward = lambda x: x.sum(-1, keepdim=True)
    calls = [_double(mod) for mod in (m.ln_f, m.blocks[0].norm)]
    logits = _run(m, path, idx)[0]
    assert logits.shape == (4, 1 if path == "token" else 128, 1)
    n = 2 if path == "token" else 1
    assert [len(c) for c in calls] == [n, n]


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["train", "prefill", "token"])
@pytest.mark.parametrize("method", ["forward", "mix"])
def test_block_method_runs(path, method):
    print(f"[case] override block {method} {path}", flush=True)
    m = _model().to(DEV)
    idx = torch.randint(0, 203, (2, 9), generator=torch.Generator().manual_seed(1)).to(DEV)
    want = _run(m, path, idx)
    block, calls = m.blocks[0], []

    def own(*args):
        calls.append(1)
        return getattr(MambaBlock, method)(block, *args)
    setattr(block, method, own)
    for i, (a, b) in enumerate(zip(_run(m, path, idx), want)):
        assert_close(f"output {i}", a, b)
    assert len(calls) == (2 if path == "token" else 1)


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["train", "prefill", "token"])
@pytest.mark.parametrize("kind", [Doubled, Tagged])
def test_subclassed_weights_keep_their_operators(path, kind):
    """in_proj, out_proj and the head (512 x 32768 x 64: a size the HIP product
    would take) with weights of a subclass that stands for twice its values."""
    print(f"[case] subclassed weights {kind.__name__} {path}", flush=True)
    m = _model(vocab=32768).to(DEV)
    m.head.weight = nn.Parameter(m.head.weight.detach().clone())
    idx = torch.randint(0, 32768, (4, 128), generator=torch.Generator().manual_seed(1)).to(DEV)
    want = copy.deepcopy(m)
    for model, double in ((want, lambda w: 2 * w),
                          (m, lambda w: kind(w) if kind is Doubled else w.as_subclass(kind))):
        for mod in (model.head, model.blocks[0].in_proj, model.blocks[1].out_proj):
            w = double(mod.weight.detach())
            mod.weight = nn.Parameter(w, requires_grad=False)
            assert type(mod.weight) in (nn.Parameter, kind)
    ref = _run(want, path, idx)
    for i, (a, b) in enumerate(zip(_run(m, path, idx), ref)):
        assert_close(f"output {i}", a.as_subclass(torch.Tensor), b)
