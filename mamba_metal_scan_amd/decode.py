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
from .block import plain, plain_mods
from .linear import PLAIN, no_hooks

# mhs_decode_layer: 13 pointers, the conv window's strides, the next window,
# eps, dt_min, dt_max, unused.
_LAYER = struct.Struct("13Q3qQ4f")


_f32 = torch.float32


def _layer(block: nn.Module, bc: dict, dev: torch.device, shapes: tuple, kinds: tuple,
           conv_next: torch.Tensor) -> Optional[bytes]:
    """The block's mhs_decode_layer, or None where the native step does not
    take it: a module of another type, with hooks or with a forward of its
    own, a weight that is not a plain fp32 parameter of its shape, a state or
    window that is not the cache's own form."""
    m, p = block._modules, block._parameters
    try:
        norm, in_proj, conv, dt_proj, b_proj, c_proj, out_proj = mods = (
            m["norm"], m["in_proj"], m["conv"], m["dt_proj"], m["B_proj"], m["C_proj"],
            m["out_proj"])
        h, win = bc["h"], bc["conv"]
        if not plain_mods(mods, kinds):
            return None
        w_dt, w_conv = dt_proj._parameters, conv._parameters
        weights = (norm._parameters["weight"], in_proj._parameters["weight"], w_conv["weight"],
                   w_conv["bias"], w_dt["weight"], w_dt["bias"], p["A"],
                   b_proj._parameters["weight"], c_proj._parameters["weight"], p["D_skip"],
                   out_proj._parameters["weight"], h)
        biases = (in_proj._parameters["bias"], b_proj._parameters["bias"],
                  c_proj._parameters["bias"], out_proj._parameters["bias"])
    except (KeyError, AttributeError):
        return None
    for t, shape in zip(weights, shapes):
        if not plain(t, dev, shape):
            return None
    if (any(v is not None for v in biases) or type(win) not in PLAIN or win.dtype is not _f32
            or win.shape != shapes[12] or win.device != dev or not norm.hip
            or block.scan_impl == "torch" or not block.dt_min < block.dt_max):
        return None
    ptrs = [t.data_ptr() for t in weights]
    # The products read 16 bytes at a time.
    if (ptrs[0] | ptrs[1] | ptrs[4] | ptrs[7] | ptrs[8] | ptrs[10]) & 15:
        return None
    return _LAYER.pack(*ptrs, win.data_ptr(), *win.stride(), conv_next.data_ptr(), norm.eps,
                       block.dt_min, block.dt_max, 0.0)


def batch_limit(d_model: int, d_inner: int, d_state: int, n_layers: int, vocab: int,
                captured: bool) -> int:
    """The largest batch that the native token takes.

    Its products pass over their weights, 512 columns at a time, again for
    every 8 rows, with VALU fmas: a layer (with its share of the head) costs
    about 0.7 us a row and 0.136 us a row and million of weights so padded, on
    top of reading them once. The module calls reuse tiles in the library's
    products, on top of their launches: 280 us and more a layer from Python; in
    a HIP graph what those cost beyond the native token's, less what its
    slower rows lose, comes to 100 us for every layer but one. us a token,
    native / modules, at the last batch won and the first lost, and the line,
    from Python and in a graph (vocabulary 32768; 200 at d_model 64, 1024 and
    2048, 5000 at 516):
      d_model 64, d_inner 88, 4 layers
        188: 557 / 5020,  585: 1628 / 1340, 384;   64: 219 / 264,   188: 555 / 460,   102
      128, 272, 2 layers
        128: 450 / 705,   256: 868 / 703,   143;   24: 114 / 136,    32: 143 / 142,   26
      384, 856, 10 layers
        256: 2711 / 3409, 512: 5313 / 3262, 226;  192: 2016 / 2153, 256: 2702 / 2405, 73
      516, 1152, 3 layers
        206: 1000 / 1081,                   171;   64: 350 / 365,   206: 1006 / 619,  41
      640, 1432, 12 layers
        128: 2632 / 4045, 256: 5008 / 4045, 143;   96: 2031 / 2276, 128: 2617 / 2454, 47
      1024, 2312, 24 layers
        64: 4393 / 7596,  128: 8205 / 7996, 108;   64: 4363 / 4943,  96: 6252 / 5809, 38
      1536, 3472, 8 layers
        32: 1633 / 2573,   64: 2921 / 2712, 47;    24: 1302 / 1406,  32: 1635 / 1588, 16
      2048, 4640, 4 layers
        16: 717 / 1339,    36: 1457 / 1356, 31;    16: 718 / 804,    36: 1456 / 1227, 9
    Up to 8 rows the weights are read once, as any product must."""
    def padded(k: int) -> int:
        return (k + 511) // 512 * 512
    weights = 2 * d_inner * padded(d_model) + (d_inner + 2 * d_state + d_model) * padded(d_inner)
    weights += vocab * padded(d_model) / n_layers
    budget = 100.0 - 100.0 / n_layers if captured else 280.0 - 0.6e-6 * weights
    return max(8, int(budget / (0.7 + 0.136e-6 * weights)))


def decode_step(model: nn.Module, x: torch.Tensor, cache: dict) -> Optional[torch.Tensor]:
    """The logits (batch, 1, vocab) of one embedded token per sequence, x
    (batch, 1, d_model), against a filled cache, which is advanced (each
    block's h in place, its conv window replaced). None (and nothing changed)
    where the native step does not apply: modules with hooks, with a forward
    set on the instance or of other types, tensors of subclasses, other
    dtypes or layouts, autocast, a cache that no prefill filled, or a batch
    above batch_limit, where the modules are the faster. The caller has
    checked that autograd is off and that every block is a plain
    MambaBlock."""
    blocks, states, head, ln_f = model.blocks, cache["blocks"], model.head, model.ln_f
    if (torch.is_autocast_enabled() or torch.compiler.is_compiling() or x.dim() != 3
            or type(x) not in PLAIN or x.dtype != torch.float32 or x.numel() == 0
            or len(blocks) == 0 or len(states) != len(blocks)):
        return None
    first = blocks[0]
    if type(first.conv) is not nn.Conv1d or type(head) is not nn.Linear:
        return None
    batch, _, d_model = x.shape
    d, n, taps = first.d_inner, first.A.shape[1], first.conv.kernel_size[0]
    dev = x.device
    x = x.contiguous()
    if (not no_hooks(head) or not no_hooks(ln_f) or type(ln_f) is not type(first.norm)
            or head.bias is not None or not ln_f.hip
            or d_model % 4 or d % 4 or not 2 <= taps <= 8 or not 1 <= n <= 64
            or batch > 8 and batch > batch_limit(d_model, d, n, len(blocks), head.out_features,
                                                 torch.cuda.is_current_stream_capturing())):
        return None
    head_w, norm_w = head._parameters.get("weight"), ln_f._parameters.get("weight")
    if (not plain(norm_w, dev, (d_model,)) or not plain(head_w, dev, (head.out_features, d_model))
            or (head_w.data_ptr() | norm_w.data_ptr() | x.data_ptr()) & 15):
        return None
    windows = torch.empty((len(blocks), batch, d, taps - 1), dtype=torch.float32,
                          device=dev).unbind(0)
    # In mhs_decode_layer's order; then the conv window.
    shapes = ((d_model,), (2 * d, d_model), (d, 1, taps), (d,), (d, d), (d,), (d, n), (n, d),
              (n, d), (d,), (d_model, d), (batch, d, n), (batch, d, taps - 1))
    kinds = (type(ln_f), nn.Linear, nn.Conv1d, nn.Linear, nn.Linear, nn.Linear, nn.Linear)
    layers = []
    for block, bc, nxt in zip(blocks, states, windows):
        packed = _layer(block, bc, dev, shapes, kinds, nxt)
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
