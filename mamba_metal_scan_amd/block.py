"""A MambaBlock's forward and backward as one native call each.

The block (mamba_metal/model.py:225-256) is a norm, three products, a conv, a
scan and a gate: through the framework, a dozen calls and three autograd
Functions per direction, whose host time (about 250 us a direction) exceeds
the GPU's for small batches. ``BlockHIP`` hands it to ``mhs_block_fwd_f32`` /
``mhs_block_bwd_f32``, which launch the same kernels from native code.
"""
from __future__ import annotations

import struct
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _native
from .fused import mamba_inner
from .linear import PLAIN
from .norm import rms_norm_residual

_WEIGHTS = struct.Struct("11Q4f")      # mhs_block_weights
_GRADS = struct.Struct("10Q")          # mhs_block_grads
_f32 = torch.float32


def plain(t: Optional[torch.Tensor], dev: torch.device, shape: tuple) -> bool:
    """Whether t is a plain tensor, fp32 of that shape, contiguous, on dev."""
    return (type(t) in PLAIN and t.dtype is _f32 and t.shape == shape and t.device == dev
            and t.is_contiguous())


def plain_mods(mods, kinds) -> bool:
    """Whether each module is of exactly its kind, without hooks or a forward
    of its own."""
    for mod, kind in zip(mods, kinds):
        if (type(mod) is not kind or mod._forward_hooks or mod._forward_pre_hooks
                or mod._backward_hooks or mod._backward_pre_hooks or "forward" in mod.__dict__):
            return False
    return True


def block_params(block: nn.Module, x: torch.Tensor, strict: bool) -> Optional[tuple]:
    """The block's parameters in mhs_block_weights' order where the native
    block takes them and x (batch, T, d_model), else None: plain modules
    without hooks or a forward of their own (strict: those too that the
    block's fused path never calls), plain fp32 contiguous 16-byte aligned
    parameters of the block's shapes, sizes that are multiples of 4. The
    caller has checked the global hooks, autocast, tracing and that x is an
    fp32 ROCm tensor."""
    m, p = block._modules, block._parameters
    try:
        norm, in_proj, conv, dt_proj, b_proj, c_proj, out_proj = mods = (
            m["norm"], m["in_proj"], m["conv"], m["dt_proj"], m["B_proj"], m["C_proj"],
            m["out_proj"])
        if not plain_mods((in_proj, out_proj), (nn.Linear, nn.Linear)):
            return None
        if strict and not plain_mods(mods[2:6], (nn.Conv1d, nn.Linear, nn.Linear, nn.Linear)):
            return None
        w_conv, w_dt = conv._parameters, dt_proj._parameters
        params = (norm._parameters["weight"], in_proj._parameters["weight"], w_conv["weight"],
                  w_conv["bias"], w_dt["weight"], w_dt["bias"], p["A"],
                  b_proj._parameters["weight"], c_proj._parameters["weight"], p["D_skip"],
                  out_proj._parameters["weight"])
        if (in_proj._parameters["bias"] is not None or b_proj._parameters["bias"] is not None
                or c_proj._parameters["bias"] is not None
                or out_proj._parameters["bias"] is not None):
            return None
    except (KeyError, AttributeError):
        return None
    dm, dev, a = x.shape[2], x.device, params[6]
    if a is None or a.dim() != 2 or params[2] is None or params[2].dim() != 3:
        return None
    d, n = a.shape
    taps = params[2].shape[2]
    if (dm % 4 or not 4 <= dm <= _native.NORM_MAX_COLS or d % 4 or n % 4 or not 4 <= n <= 64
            or not 1 <= taps <= 8 or 2 * d >= 1 << 22 or x.shape[0] > 65535
            or not block.dt_min < block.dt_max or block.ckpt_chunk < 1):
        return None
    bits = 0
    for t, shape in zip(params, ((dm,), (2 * d, dm), (d, 1, taps), (d,), (d, d), (d,), (d, n),
                                 (n, d), (n, d), (d,), (dm, d))):
        if not plain(t, dev, shape):
            return None
        bits |= t.data_ptr()
    return None if bits & 15 else params


def _sizes(x: torch.Tensor, params: tuple) -> tuple:
    d, n = params[6].shape
    return (*x.shape, d, n, params[2].shape[2])


def _pack(params: tuple, consts: tuple) -> bytes:
    return _WEIGHTS.pack(*[t.data_ptr() for t in params], *consts[:3], 0.0)


def block_forward(x: torch.Tensor, delta: Optional[torch.Tensor], params: tuple, consts: tuple,
                  with_ckpt: bool, want_state: bool) -> tuple:
    """(x + delta (or x), out, xz, saved, h_last): see mhs_block_fwd_f32.
    consts: (eps, dt_min, dt_max, chunk)."""
    bt, t_len, dm, d, n, taps = sizes = _sizes(x, params)
    lib = _native.library()
    dev = x.device
    out = torch.empty_like(x)
    x_out = torch.empty_like(x) if delta is not None else x
    xz = x.new_empty((bt, t_len, 2 * d))
    h_last = x.new_empty((bt, d, n)) if want_state else None
    # (fp32, as its contents: saved-tensor hooks may convert what they pack)
    saved = x.new_empty(lib.mhs_block_saved_bytes(*sizes, consts[3], with_ckpt) // 4)
    nbytes = lib.mhs_block_fwd_workspace_bytes(*sizes)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    with _native._on(dev):
        rc = lib.mhs_block_fwd_f32(
            _pack(params, consts), x.data_ptr(), _native._ptr(delta), x_out.data_ptr(),
            out.data_ptr(), xz.data_ptr(), saved.data_ptr(), _native._ptr(h_last), *sizes,
            consts[3], with_ckpt, ws.data_ptr(), nbytes, _native._stream(dev))
    _native._check(rc, "mhs_block_fwd_f32")
    return x_out, out, xz, saved, h_last


def _restored(t: torch.Tensor, align: int) -> torch.Tensor:
    """A saved tensor as the kernels read it, whatever layout a saved-tensor
    hook gave it back in."""
    if t.dtype is not _f32:
        raise TypeError(f"the block's saved tensors are float32; a saved-tensor hook returned "
                        f"{t.dtype}")
    t = t.contiguous()
    return t.clone() if t.data_ptr() % align else t


def _module_gradients(ctx, x: torch.Tensor, params: list, g_x, g_out) -> tuple:
    """The backward's gradients by way of the functions of the module path run
    again, for a caller that differentiates them: a graph over the products,
    as that path's own backward leaves it (the kernels' Functions are first
    order). Differentiated by aliases: x is an output of this node itself where
    a delta was added, and the way to the weights must not lead through it."""
    leaves = [t.view_as(t) for t in (x, *params)]
    x, *params = leaves
    norm_w, in_w, conv_w, conv_b, dt_w, dt_b, a, b_w, c_w, d_skip, out_w = params
    eps, dt_min, dt_max, chunk = ctx.consts
    res, h = rms_norm_residual(x, norm_w, eps)
    out = F.linear(mamba_inner(F.linear(h, in_w), conv_w, conv_b, dt_w, dt_b, b_w, c_w, a, d_skip,
                               dt_min, dt_max, chunk=chunk), out_w)
    need = [i for i, t in enumerate(leaves) if t.requires_grad]
    pairs = [(o, g) for o, g in ((res, g_x), (out, g_out)) if g is not None]
    got = torch.autograd.grad([o for o, _ in pairs], [leaves[i] for i in need],
                              [g for _, g in pairs], create_graph=True, allow_unused=True)
    grads = [None] * len(leaves)
    for i, g in zip(need, got):
        grads[i] = g
    return (grads[0], grads[0] if ctx.has_delta else None, None, *grads[1:])


class BlockHIP(torch.autograd.Function):
    """(x + delta, out) of a block; delta None: (x, out). The gradients of both
    outputs reach x and delta in the norm's backward kernel."""

    @staticmethod
    def forward(ctx, x, delta, consts, *params):
        need = any(ctx.needs_input_grad)   # (a frozen block keeps nothing)
        x_out, out, xz, saved, _ = block_forward(x, delta, params, consts, need, False)
        if need:
            ctx.save_for_backward(x_out, xz, saved, *params)
        ctx.consts = consts
        ctx.has_delta = delta is not None
        ctx.set_materialize_grads(False)
        return x_out, out

    @staticmethod
    def backward(ctx, g_x, g_out):
        x, xz, saved, *params = ctx.saved_tensors
        x, xz, *params = (_restored(t, 16) for t in (x, xz, *params))
        if torch.is_grad_enabled():   # create_graph
            return _module_gradients(ctx, x, params, g_x, g_out)
        saved = _restored(saved, 256)
        need = ctx.needs_input_grad
        if g_out is None:
            g_out = torch.zeros_like(x)
        g_out = g_out.contiguous()
        if g_out.data_ptr() & 15:
            g_out = g_out.clone()
        if g_x is not None:
            g_x = g_x.contiguous()
            if g_x.data_ptr() & 15:
                g_x = g_x.clone()
        sizes = _sizes(x, params)
        d, n = params[6].shape
        norm_w, in_w, conv_w, conv_b, dt_w, dt_b, a, _, _, d_skip, out_w = params
        dx = torch.empty_like(x)
        d_norm, d_conv_w = torch.empty_like(norm_w), torch.empty_like(conv_w)
        d_conv_b, d_dt_b = torch.empty_like(conv_b), torch.empty_like(dt_b)
        d_a, dd = torch.empty_like(a), torch.empty_like(d_skip)
        d_in = torch.empty_like(in_w) if need[4] else None
        d_out = torch.empty_like(out_w) if need[13] else None
        d_proj = dt_w.new_empty((d + 2 * n, d))
        grads = [dx, d_norm, d_in, d_conv_w, d_conv_b, d_proj, d_dt_b, d_a, dd, d_out]
        lib = _native.library()
        dev = x.device
        with _native._bwd_reduction(), _native._on(dev):
            nbytes = lib.mhs_block_bwd_workspace_bytes(*sizes, ctx.consts[3])
            ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
            rc = lib.mhs_block_bwd_f32(
                _pack(params, ctx.consts), x.data_ptr(), xz.data_ptr(), saved.data_ptr(),
                g_out.data_ptr(), _native._ptr(g_x),
                _GRADS.pack(*[0 if t is None else t.data_ptr() for t in grads]), *sizes,
                ctx.consts[3], ws.data_ptr(), nbytes, _native._stream(dev))
        _native._check(rc, "mhs_block_bwd_f32")
        return (dx, dx if ctx.has_delta else None, None, d_norm, d_in, d_conv_w, d_conv_b,
                d_proj[:d], d_dt_b, d_a, d_proj[d:d + n], d_proj[d + n:], dd, d_out)
