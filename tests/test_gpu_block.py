"""GPU parity of the native block (mhs_block_fwd_f32 / _bwd_f32): a MambaBlock's
output, input gradient and every parameter gradient, and a prefill's cache,
against the float64 torch block (scan_impl 'torch', the reference's own
forward, mamba_metal/model.py:225-256).

Bar: 1e-4 max relative per tensor, the build's parity bar.
"""
from __future__ import annotations

import contextlib

import pytest
import torch

from helpers import assert_close
from mamba_metal_scan_amd import _native, block as block_mod
from mamba_metal_scan_amd.model import MambaBlock, MambaConfig, TinyMamba

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _blocks(d_model, d_inner, n=16, k=4, chunk=16):
    kw = dict(vocab_size=8, d_model=d_model, d_state=n, d_conv=k, ckpt_chunk=chunk)
    torch.manual_seed(d_model + d_inner + n)
    hip = MambaBlock(MambaConfig(scan_impl="hip", **kw), d_inner)
    with torch.no_grad():
        hip.dt_proj.bias.normal_()
        hip.D_skip.normal_()
        hip.A.normal_(0.0, 3.0)
        hip.norm.weight.normal_(1.0, 0.1)
    ref = MambaBlock(MambaConfig(scan_impl="torch", **kw), d_inner).double()
    ref.load_state_dict({k2: v.double() for k2, v in hip.state_dict().items()})
    return hip.to(DEV), ref


def _calls(monkeypatch):
    """The native forwards, by whether they kept checkpoints."""
    seen = []
    real = block_mod.block_forward

    def spy(*args):
        seen.append(args[4])
        return real(*args)
    monkeypatch.setattr(block_mod, "block_forward", spy)
    monkeypatch.setattr("mamba_metal_scan_amd.model.block_forward", spy)
    return seen


# Rows and widths below, at and above the products' tiles (64, 128), sequences
# of one step, of a chunk's remainder and in time segments, every conv length's
# ends, strides that recompute checkpoints.
@pytest.mark.parametrize("bt,t,d_model,d_inner,n,k,chunk", [
    (1, 1, 4, 4, 4, 4, 16), (2, 5, 64, 68, 16, 1, 16), (3, 65, 128, 132, 8, 8, 64),
    (2, 300, 132, 64, 64, 4, 32), (4, 129, 68, 256, 16, 2, 100)])
def test_forward_and_gradients(monkeypatch, bt, t, d_model, d_inner, n, k, chunk):
    print(f"[case] block {bt}x{t} {d_model} {d_inner} {n} {k} {chunk}", flush=True)
    hip, ref = _blocks(d_model, d_inner, n, k, chunk)
    seen = _calls(monkeypatch)
    g = torch.Generator().manual_seed(t)
    x, dy = (torch.randn(bt, t, d_model, generator=g) for _ in range(2))
    xr, xh = x.double().requires_grad_(), x.to(DEV).requires_grad_()
    yr, yh = ref(xr), hip(xh)
    yr.backward(dy.double())
    yh.backward(dy.to(DEV))
    torch.cuda.synchronize()
    assert seen == [True]
    assert_close("out", yh, yr)
    assert_close("dx", xh.grad, xr.grad)
    for (name, p), q in zip(hip.named_parameters(), ref.parameters()):
        assert_close(name, p.grad, q.grad)


@pytest.mark.parametrize("t", [1, 2, 3, 40])
def test_prefill_fills_the_cache(monkeypatch, t):
    """Prompts shorter and longer than the conv window."""
    hip, ref = _blocks(64, 96)
    seen = _calls(monkeypatch)
    x = torch.randn(3, t, 64, generator=torch.Generator().manual_seed(t))
    ch, cr = {}, {}
    with torch.no_grad():
        yh, yr = hip(x.to(DEV), ch), ref(x.double(), cr)
    torch.cuda.synchronize()
    assert seen == [False]
    assert_close("out", yh, yr)
    assert_close("h", ch["h"], cr["h"])
    assert_close("conv", ch["conv"], cr["conv"])


def test_frozen_weights_and_unused_outputs():
    """Products whose gradient nobody asks for are left out; the gradient of x
    + delta alone (the block's output unused) passes through."""
    hip, _ = _blocks(64, 96)
    x = torch.randn(2, 33, 64, generator=torch.Generator().manual_seed(0)).to(DEV)

    def run(frozen):
        for name, p in hip.named_parameters():
            p.requires_grad_(name not in frozen)
            p.grad = None
        xi = x.clone().requires_grad_()
        hip(xi).square().sum().backward()
        return xi.grad, {k: p.grad for k, p in hip.named_parameters()}
    dx, full = run(())
    for frozen in (("in_proj.weight", "out_proj.weight"), ("A", "dt_proj.weight")):
        dx2, part = run(frozen)
        assert torch.equal(dx, dx2)
        for k, v in part.items():
            assert (v is None) if k in frozen else torch.equal(v, full[k]), k
    xi = x.clone().requires_grad_()
    delta = torch.ones_like(x).requires_grad_()
    x_out, _ = hip._native(xi, delta)
    x_out.sum().backward()
    assert torch.equal(xi.grad, torch.ones_like(x)) and torch.equal(delta.grad, xi.grad)


def test_error_is_no_larger_than_the_modules():
    """The block of the 640-wide model on 4 x 130 tokens: every output's
    relative 2-norm error against float64 beside that of the same block's
    module calls (a hook on in_proj), whose products are the library's. Bar:
    1.3 times it, and 2^-23, a rounding of the result and one of its terms."""
    print("[case] block error 4x130x640", flush=True)
    hip, ref = _blocks(640, 1432)
    ref = ref.to(DEV)
    g = torch.Generator().manual_seed(3)
    x, dy = (torch.randn(4, 130, 640, generator=g).to(DEV) for _ in range(2))

    def run(block, dtype):
        xi = x.to(dtype).requires_grad_()
        out = block(xi)
        grads = torch.autograd.grad(out, [xi, *block.parameters()], dy.to(dtype))
        return [out.detach().double(), *[v.double() for v in grads]]
    want = run(ref, torch.float64)
    native = run(hip, torch.float32)
    handle = hip.in_proj.register_forward_hook(lambda m, i, o: None)
    modules = run(hip, torch.float32)
    handle.remove()
    names = ["out", "dx"] + [k for k, _ in hip.named_parameters()]
    for name, a, b, w in zip(names, native, modules, want):
        ea, eb = ((v - w).norm() / w.norm() for v in (a, b))
        assert ea <= 1.3 * eb + 2.0 ** -23, (name, ea.item(), eb.item())


@pytest.mark.parametrize("with_delta", [False, True])
def test_gradients_of_gradients_as_the_module_path_leaves_them(with_delta):
    """create_graph: first-order gradients equal, and a penalty on the
    projections' weight gradients has the gradients that the module path (a
    hook on in_proj) gives it."""
    print(f"[case] create_graph block delta {with_delta}", flush=True)
    m = TinyMamba(MambaConfig(vocab_size=50, d_model=64, n_layers=2, d_ff=128,
                              scan_impl="hip")).to(DEV)
    block = m.blocks[1] if with_delta else m.blocks[0]
    idx = torch.randint(0, 50, (2, 20), generator=torch.Generator().manual_seed(0)).to(DEV)
    x = torch.randn(2, 20, 64, generator=torch.Generator().manual_seed(1)).to(DEV)
    weights = (block.in_proj.weight, block.out_proj.weight)

    def run():
        loss = m(idx, idx)[1] if with_delta else block(x).square().mean()
        first = torch.autograd.grad(loss, weights, create_graph=True)
        penalty = sum(g.square().sum() for g in first)
        second = torch.autograd.grad(penalty, weights, allow_unused=True)
        return [*first, *[torch.zeros_like(w) if v is None else v
                          for v, w in zip(second, weights)]]
    native = run()
    handles = [b.in_proj.register_forward_hook(lambda mod, i, o: None) for b in m.blocks]
    modules = run()
    for h in handles:
        h.remove()
    for i, (a, b) in enumerate(zip(native, modules)):
        assert_close(f"gradient {i}", a, b, tol=2e-5)
    assert native[2].abs().max() > 0


def test_frozen_blocks_keep_no_checkpoints(monkeypatch):
    """With autograd on and nothing to differentiate, as with it off: no
    checkpoints are written, nothing is saved."""
    hip, ref = _blocks(64, 96)
    hip.requires_grad_(False)
    seen = _calls(monkeypatch)
    x = torch.randn(2, 33, 64, generator=torch.Generator().manual_seed(0))
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(packed.append, lambda t: t):
        out = hip(x.to(DEV))
    assert seen == [False] and packed == [] and not out.requires_grad
    assert_close("out", out, ref(x.double()))
    hip(x.to(DEV).requires_grad_())
    assert seen == [False, True]


@pytest.mark.parametrize("form", ["cpu", "strided", "offset", "bf16"])
def test_saved_tensor_hooks(form):
    """Hooks that move what the forward saved, give it back in another layout
    or at another alignment, or keep it in bf16 (whatever is saved, floating
    point or not, must survive as numbers)."""
    print(f"[case] saved-tensor hooks {form}", flush=True)
    hip, _ = _blocks(64, 96)
    x = torch.randn(2, 33, 64, generator=torch.Generator().manual_seed(0)).to(DEV)
    packed = []

    def pack(t):
        packed.append(t.dtype)
        return t.to(torch.bfloat16) if form == "bf16" else t.cpu()

    def unpack(t):
        t = t.float().to(DEV)
        if form == "strided":
            return torch.stack([t, t], -1)[..., 0]
        if form == "offset":
            return torch.cat([t.new_zeros(5), t.flatten()])[5:].view(t.shape)
        return t

    def run(ctx):
        xi = x.clone().requires_grad_()
        hip.zero_grad(set_to_none=True)
        with ctx:
            out = hip(xi)
        out.square().sum().backward()
        return [out.detach(), xi.grad, *[p.grad for p in hip.parameters()]]
    want = run(contextlib.nullcontext())
    got = run(torch.autograd.graph.saved_tensors_hooks(pack, unpack))
    assert packed and set(packed) == {torch.float32}
    for i, (a, b) in enumerate(zip(got, want)):
        if form == "bf16":
            assert_close(f"output {i}", a, b, tol=0.1)
        else:
            assert torch.equal(a, b), i


def test_hooks_subclasses_and_offset_views_take_the_module_path(monkeypatch):
    hip, ref = _blocks(64, 96)
    seen = _calls(monkeypatch)
    x = torch.randn(2, 20, 64, generator=torch.Generator().manual_seed(5))
    want = ref(x.double())
    ran = []
    h = hip.out_proj.register_forward_hook(lambda m, i, o: ran.append(1))
    assert_close("hook", hip(x.to(DEV)), want)
    h.remove()
    assert ran == [1] and seen == []

    class Doubled(MambaBlock):
        def mix(self, h, cache=None):
            return 2 * super().mix(h, cache)
    hip.__class__ = Doubled
    assert_close("subclass", hip(x.to(DEV)) - x.to(DEV), 2 * (want - x.double()))
    hip.__class__ = MambaBlock
    assert seen == []
    buf = torch.empty(x.numel() + 1, device=DEV)   # x 4 bytes into its storage: copied
    view = buf[1:].view(x.shape).copy_(x.to(DEV))
    assert_close("offset view", hip(view), want)
    assert seen == [True]


def test_model_gradients_equal_the_module_path():
    """A TinyMamba's loss and gradients through the native blocks against the
    same model with a hook on every in_proj (the module path)."""
    torch.manual_seed(0)
    m = TinyMamba(MambaConfig(vocab_size=203, d_model=64, n_layers=3, d_ff=128,
                              scan_impl="hip")).to(DEV)
    idx = torch.randint(0, 203, (3, 50), generator=torch.Generator().manual_seed(2)).to(DEV)

    def grads():
        m.zero_grad(set_to_none=True)
        _, loss = m(idx[:, :-1], idx[:, 1:])
        loss.backward()
        return loss.detach(), {k: p.grad.clone() for k, p in m.named_parameters()}
    loss, native = grads()
    handles = [b.in_proj.register_forward_hook(lambda mod, i, o: None) for b in m.blocks]
    loss2, module = grads()
    for h in handles:
        h.remove()
    assert_close("loss", loss, loss2, tol=1e-6)
    for k in native:
        assert_close(k, native[k], module[k], tol=2e-5)


def test_forward_and_gradients_replay_from_a_hip_graph():
    """The native block's launches captured once and replayed three times, with
    eager work between: every replay equals the eager result."""
    hip, _ = _blocks(64, 96)
    g = torch.Generator().manual_seed(4)
    x = torch.randn(2, 65, 64, generator=g).to(DEV).requires_grad_()
    dy = torch.randn(2, 65, 64, generator=g).to(DEV)
    leaves = [x] + list(hip.parameters())

    def step(inputs):
        out = hip(inputs[0])
        return (out,) + torch.autograd.grad(out, inputs, dy)
    _native.set_reduction(_native.REDUCTION_FIXED)
    try:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            ref = [v.detach().clone() for v in step(leaves)]
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = step(leaves)
        for rep in range(3):
            torch.randn(1 << 20, device=DEV).sum().item()   # eager work between replays
            graph.replay()
            torch.cuda.synchronize()
            for i, (a, b) in enumerate(zip(outs, ref)):
                assert torch.equal(a, b), f"replay {rep}: output {i} differs"
    finally:
        _native.set_reduction(_native.REDUCTION_AUTO)
