"""GPU parity of the native one-token step of a TinyMamba (mhs_decode_f32):
logits, states and conv windows against the float64 step of the torch model
(scan_impl 'torch', the reference's own update, mamba_metal/model.py:228-256),
over several tokens.

Bar: 1e-4 max relative per tensor, the build's parity bar.
"""
from __future__ import annotations

import pytest
import torch

from helpers import assert_close
from mamba_metal_scan_amd import decode
from mamba_metal_scan_amd.model import MambaConfig, TinyMamba

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _models(**over):
    kw = dict(vocab_size=203, d_model=64, n_layers=2, d_ff=128, max_seq_len=64, d_state=16,
              d_conv=4)
    kw.update(over)
    torch.manual_seed(3)
    hip = TinyMamba(MambaConfig(scan_impl="hip", **kw))
    with torch.no_grad():   # not the initial zeros and ones
        for b in hip.blocks:
            b.dt_proj.bias.normal_()
            b.D_skip.normal_()
            b.A.normal_(0.0, 4.0)   # softplus on both sides of 0
            b.norm.weight.normal_(1.0, 0.1)
        hip.ln_f.weight.normal_(1.0, 0.1)
    ref = TinyMamba(MambaConfig(scan_impl="torch", **kw)).double()
    ref.load_state_dict({k: v.double() for k, v in hip.state_dict().items()})
    return hip.to(DEV), ref


def _native_calls(monkeypatch):
    seen = []
    real = decode.decode_step

    def spy(*args):
        out = real(*args)
        seen.append(out is not None)
        return out
    monkeypatch.setattr("mamba_metal_scan_amd.model.decode_step", spy)
    return seen


# Batches around the kernels' 1, 2, 4 and 8 rows; widths whose K / 4 is below,
# at and above one pass (128 lanes' loads); states of the 4-lane and the
# 1-lane kernel, odd ones; the shortest and longest conv.
@pytest.mark.parametrize("batch,over", [
    (1, {}), (2, dict(d_model=128, d_inner=516)), (3, dict(d_state=5)), (4, dict(d_state=64)),
    (5, dict(d_state=3, d_conv=2)), (8, dict(d_model=512, d_inner=512, d_conv=8)),
    (9, dict(d_state=1, vocab_size=17)), (17, dict(d_model=516, d_inner=4, n_layers=1))])
def test_token_matches_float64(monkeypatch, batch, over):
    print(f"[case] decode batch {batch} {over}", flush=True)
    hip, ref = _models(**over)
    seen = _native_calls(monkeypatch)
    vocab = hip.cfg.vocab_size
    idx = torch.randint(0, vocab, (batch, 9), generator=torch.Generator().manual_seed(batch))
    ch, cr = {}, {}
    with torch.no_grad():
        hip(idx[:, :6].to(DEV), cache=ch)
        ref(idx[:, :6], cache=cr)
        for t in range(6, 9):
            lh, _ = hip(idx[:, t:t + 1].to(DEV), cache=ch)
            lr, _ = ref(idx[:, t:t + 1], cache=cr)
            torch.cuda.synchronize()
            assert_close("logits", lh, lr)
            for bh, br in zip(ch["blocks"], cr["blocks"]):
                assert_close("h", bh["h"], br["h"])
                assert_close("conv", bh["conv"], br["conv"])
    assert seen == [True] * 3


@pytest.mark.parametrize("batch,shift", [(4, 0.0), (8, -8.0)])
def test_error_is_no_larger_than_the_modules(monkeypatch, batch, shift):
    """A token of a 640-wide block from a given cache: the relative 2-norm
    error of its logits, state and window against float64 beside that of the
    module calls, which use the framework's softplus, sigmoid and exp and the
    library's products. Bar: 1.2 times it (measured 0.5 to 1.0 of it)."""
    print(f"[case] decode error batch {batch}", flush=True)
    hip, ref = _models(d_model=640, d_inner=1432, n_layers=1)
    with torch.no_grad():
        for m in (hip, ref):
            m.blocks[0].A.add_(shift)
    ref = ref.to(DEV)
    g = torch.Generator().manual_seed(batch)
    start = {"h": torch.randn(batch, 1432, 16, generator=g).to(DEV),
             "conv": torch.randn(batch, 1432, 3, generator=g).to(DEV)}
    tok = torch.randint(0, 203, (batch, 1), generator=g).to(DEV)

    def run(model, dtype):
        cache = {"blocks": [{k: v.to(dtype, copy=True) for k, v in start.items()}]}
        with torch.no_grad():
            logits = model(tok, cache=cache)[0]
        return [v.double() for v in (logits, cache["blocks"][0]["h"], cache["blocks"][0]["conv"])]
    want = run(ref, torch.float64)
    seen = _native_calls(monkeypatch)
    native = run(hip, torch.float32)
    assert seen == [True]
    monkeypatch.setattr("mamba_metal_scan_amd.model.decode_step", lambda *a: None)
    for name, a, b, w in zip(("logits", "h", "conv"), native, run(hip, torch.float32), want):
        ea, eb = ((v - w).norm() / w.norm() for v in (a, b))
        assert ea <= 1.2 * eb, (name, ea.item(), eb.item())


def test_batches_on_both_sides_of_the_limit(monkeypatch):
    """The largest batch of the native token and the next, which takes the
    module calls; both follow the float64 step."""
    hip, ref = _models(n_layers=1)
    limit = decode.batch_limit(64, hip.d_inner, 16, 1, 203, False)
    assert 8 < limit < 1024
    seen = _native_calls(monkeypatch)
    for batch, native in ((limit, True), (limit + 1, False)):
        idx = torch.randint(0, 203, (batch, 4), generator=torch.Generator().manual_seed(batch))
        ch, cr = {}, {}
        with torch.no_grad():
            hip(idx[:, :3].to(DEV), cache=ch)
            ref(idx[:, :3], cache=cr)
            lh, _ = hip(idx[:, 3:].to(DEV), cache=ch)
            lr, _ = ref(idx[:, 3:], cache=cr)
        assert_close("logits", lh, lr)
        assert_close("h", ch["blocks"][0]["h"], cr["blocks"][0]["h"])
        assert seen.pop() is native
    # in a HIP graph the modules' launches cost less: the line is lower
    low = decode.batch_limit(64, hip.d_inner, 16, 1, 203, True)
    assert 8 <= low < limit
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    for batch, native in ((low, True), (low + 1, False)):
        cache, idx = {}, torch.zeros((batch, 2), dtype=torch.int64, device=DEV)
        with torch.no_grad():
            hip(idx, cache=cache)
            hip(idx[:, :1], cache=cache)
        assert seen.pop() is native


def test_other_forms_take_the_general_step(monkeypatch):
    """A hook inside a block and autograd keep the module calls, with the same
    results; so does autocast, which their step kernel refuses."""
    hip, ref = _models()
    seen = _native_calls(monkeypatch)
    idx = torch.randint(0, 203, (2, 8), generator=torch.Generator().manual_seed(1)).to(DEV)

    def step(ctx, prepare=lambda: None):
        cache = {}
        with torch.no_grad():
            hip(idx[:, :-1], cache=cache)
        prepare()
        with ctx:
            return hip(idx[:, -1:], cache=cache)[0].detach().float()

    want = step(torch.no_grad())
    assert seen == [True]
    assert_close("autograd", step(torch.enable_grad()), want)
    assert len(seen) == 1    # not asked
    hook = []
    handles = []
    got = step(torch.no_grad(), lambda: handles.append(
        hip.blocks[1].in_proj.register_forward_hook(lambda m, i, o: hook.append(1))))
    handles[0].remove()
    assert hook == [1] and seen == [True, False]
    assert_close("hook", got, want)
    with torch.autocast("cuda", dtype=torch.bfloat16), pytest.raises(RuntimeError,
                                                                     match="fp32-only"):
        step(torch.no_grad())    # refused by the general step
    assert seen == [True, False, False]


def test_windows_of_earlier_steps_are_kept():
    """A cache's conv window is replaced, not written: a copy of the cache
    dicts (with h cloned) resumes from where it was taken."""
    hip, _ = _models()
    idx = torch.randint(0, 203, (2, 8), generator=torch.Generator().manual_seed(2)).to(DEV)
    cache = {}
    with torch.no_grad():
        hip(idx[:, :6], cache=cache)
        hip(idx[:, 6:7], cache=cache)
        snap = {"blocks": [dict(b, h=b["h"].clone()) for b in cache["blocks"]]}
        first, _ = hip(idx[:, 7:8], cache=cache)
        again, _ = hip(idx[:, 7:8], cache=snap)
    assert torch.equal(first, again)


def test_token_replays_from_a_hip_graph():
    """One captured token (the cache it reads written back in place between
    replays): three replays, with eager work between, equal the eager token."""
    hip, _ = _models()
    idx = torch.randint(0, hip.cfg.vocab_size, (2, 7), generator=torch.Generator().manual_seed(2))
    idx = idx.to(DEV)
    with torch.no_grad():
        cache = {}
        hip(idx[:, :6], cache=cache)
        saved = [{k: v.clone() for k, v in b.items()} for b in cache["blocks"]]

        def token():
            c = {"blocks": [dict(b) for b in start]}
            return hip(idx[:, 6:], cache=c)[0]
        start = [{k: v.clone() for k, v in b.items()} for b in saved]

        def restore():
            for b, s in zip(start, saved):
                for k in s:
                    b[k].copy_(s[k])
        ref = token().clone()
        restore()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            token()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = token()
        for rep in range(3):
            restore()
            torch.randn(1 << 20, device=DEV).sum().item()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref), f"replay {rep}"
