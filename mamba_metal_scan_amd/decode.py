"""One recurrent token of a TinyMamba as a single native call.

The reference's step (mamba_metal/model.py:228-256, :289-298) is about twenty
framework calls a block; at one token per sequence each is a launch that costs
more than its work (80M model, batch 4: 231 launches, 4.0 ms for 314 MB of
weights). ``decode_step`` hands the weights, the cache and the embedded token
to ``mhs_decode_f32``, which launches four kernels a block.
"""
from __future__ import annotations

import struct
from typing import Optional

import torch
import torch.nn as nn

from . import _native
from .linear import no_hooks

# mhs_decode_layer: 13 pointers, the conv window's strides, the next window,
# eps, dt_min, dt_max, unused.
_LAYER = struct.Struct("13Q3qQ4f")


def _weight(mod: Optional[nn.Module], kind: type, dev: torch.device, shape: tuple
            ) -> Optional[torch.Tensor]:
    """mod's weight where mod is a plain module of that type without hooks and
    the weight is fp32 of that shape, contiguous, on dev; else None."""
    if type(mod) is not kind or not no_hooks(mod):
        return None
    return _param(mod._parameters.get("weight"), dev, shape)


def _param(p: Optional[torch.Tensor], dev: torch.device, shape: tuple) -> Optional[torch.Tensor]:
    if (p is None or p.dtype != torch.float32 or p.device != dev or p.shape != shape
            or not p.is_contiguous()):
        return None
    return p


def _layer(block: nn.Module, bc: dict, dev: torch.device, sizes: tuple, norm_type: type,
           conv_next: torch.Tensor) -> Optional[bytes]:
    """The block's mhs_decode_layer, or None where the native step does not
    take it."""
    batch, d_model, d, n, taps = sizes
    m, p = block._modules, block._parameters
    norm, conv, dt_proj = m.get("norm"), m.get("conv"), m.get("dt_proj")
    h, win = bc.get("h"), bc.get("conv")
    weights = (
        _weight(norm, norm_type, dev, (d_model,)),
        _weight(m.get("in_proj"), nn.Linear, dev, (2 * d, d_model)),
        _weight(conv, nn.Conv1d, dev, (d, 1, taps)),
        _param(conv._parameters.get("bias"), dev, (d,)) if conv is not None else None,
        _weight(dt_proj, nn.Linear, dev, (d, d)),
        _param(dt_proj._parameters.get("bias"), dev, (d,)) if dt_proj is not None else None,
        _param(p.get("A"), dev, (d, n)),
        _weight(m.get("B_proj"), nn.Linear, dev, (n, d)),
        _weight(m.get("C_proj"), nn.Linear, dev, (n, d)),
        _param(p.get("D_skip"), dev, (d,)),
        _weight(m.get("out_proj"), nn.Linear, dev, (d_model, d)),
        _param(h, dev, (batch, d, n)),
    )
    if (any(t is None for t in weights) or win is None or win.dtype != torch.float32
            or win.device != dev or win.shape != (batch, d, taps - 1) or not norm.hip
            or block.scan_impl == "torch" or not block.dt_min < block.dt_max
            or any(m[k]._parameters.get("bias") is not None
                   for k in ("in_proj", "B_proj", "C_proj", "out_proj"))):
        return None
    ptrs = [t.data_ptr() for t in weights]
    # The products read 16 bytes at a time.
    if (ptrs[0] | ptrs[1] | ptrs[4] | ptrs[7] | ptrs[8] | ptrs[10]) & 15:
        return None
    return _LAYER.pack(*ptrs, win.data_ptr(), *win.stride(), conv_next.data_ptr(), norm.eps,
                       block.dt_min, block.dt_max, 0.0)


def decode_step(model: nn.Module, x: torch.Tensor, cache: dict) -> Optional[torch.Tensor]:
    """The logits (batch, 1, vocab) of one embedded token per sequence, x
    (batch, 1, d_model), against a filled cache, which is advanced (each
    block's h in place, its conv window replaced). None (and nothing changed)
    where the native step does not apply: modules with hooks or of other
    types, other dtypes or layouts, autocast, or a cache that no prefill
    filled. The caller has checked that autograd is off and that every block
    is a plain MambaBlock."""
    blocks, states, head, ln_f = model.blocks, cache["blocks"], model.head, model.ln_f
    if (torch.is_autocast_enabled() or torch.compiler.is_compiling() or x.dim() != 3
            or x.dtype != torch.float32 or x.numel() == 0 or len(blocks) == 0
            or len(states) != len(blocks)):
        return None
    first = blocks[0]
    if type(first.conv) is not nn.Conv1d or type(head) is not nn.Linear:
        return None
    batch, _, d_model = x.shape
    d, n, taps = first.d_inner, first.A.shape[1], first.conv.kernel_size[0]
    dev = x.device
    head_w = _weight(head, nn.Linear, dev, (head.out_features, d_model))
    norm_w = _weight(ln_f, type(first.norm), dev, (d_model,))
    x = x.contiguous()
    if (head_w is None or norm_w is None or head.bias is not None or not ln_f.hip
            or d_model % 4 or d % 4 or not 2 <= taps <= 8 or not 1 <= n <= 64
            or batch > 65535 or (head_w.data_ptr() | norm_w.data_ptr() | x.data_ptr()) & 15):
        return None
    windows = torch.empty((len(blocks), batch, d, taps - 1), dtype=torch.float32,
                          device=dev).unbind(0)
    sizes = (batch, d_model, d, n, taps)
    layers = []
    for block, bc, nxt in zip(blocks, states, windows):
        packed = _layer(block, bc, dev, sizes, type(first.norm), nxt)
        if packed is None:
            return None
        layers.append(packed)
    logits = x.new_empty((batch, 1, head_w.shape[0]))
    lib = _native.library()
    nbytes = int(lib.mhs_decode_workspace_bytes(batch, d_model, d, n))
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    with _native._on(dev):
        rc = lib.mhs_decode_f32(b"".join(layers), len(layers), x.data_ptr(), norm_w.data_ptr(),
                                ln_f.eps, head_w.data_ptr(), logits.data_ptr(), batch,
                                d_model, d, n, taps, head_w.shape[0], ws.data_ptr(), nbytes,
                                _native._stream(dev))
    _native._check(rc, "mhs_decode_f32")
    for bc, nxt in zip(states, windows):
        bc["conv"] = nxt
    return logits
