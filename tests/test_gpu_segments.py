"""The automatic split of sparse grids into many time segments: outputs and
gradients against the same kernels unsegmented, over the forms the entry
points take (d_state of each plan, strides that walk, sweep or recompute, bf16,
the gated scan with strided projections and a bias, a final-state gradient).

Bar: 1e-5 max relative per tensor (fp32 sums in another order; a segment's
start state is folded from its predecessors' instead of walked), bf16 outputs
1e-2 (their rounding).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from helpers import rel_err
from mamba_metal_scan_amd import _native, selective_scan_gated, selective_scan_hip
from oracle import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _grads(out, leaves, seed):
    g = torch.Generator().manual_seed(seed)
    outs = [o for o in out if o is not None]
    ups = [torch.randn(o.shape, generator=g).to(DEV, o.dtype) for o in outs]
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, leaves, ups))


def _both(run):
    auto = run()
    _native.set_time_segments(1)
    try:
        return auto, run()
    finally:
        _native.set_time_segments(0)


def _compare(auto, one, bf16):
    for i, (a, b) in enumerate(zip(auto, one)):
        tol = 1e-2 if bf16 and a.dtype == torch.bfloat16 else 1e-5
        assert rel_err(a.float(), b.float()) <= tol, i


def _more_workspace(bt, t, d, n):
    """The split the shape gets is automatic and not the unsegmented one."""
    need = _native.library().mhs_scan_fwd_workspace_bytes(bt, t, d, n)
    assert 0 < need <= _native.NOALLOC_SCRATCH_BYTES
    return need


@pytest.mark.parametrize("bt,t,d,n,chunk,bf16", [
    (1, 577, 64, 16, 16, False), (2, 1000, 40, 5, 32, False), (1, 3001, 33, 64, 100, False),
    (1, 4099, 70, 16, 64, True), (3, 333, 96, 4, 16, True), (1, 2048, 512, 32, 48, False),
    (4, 1024, 1024, 64, 16, False)])
def test_many_segments_equal_one(bt, t, d, n, chunk, bf16):
    print(f"[case] segments {bt}x{t}x{d}x{n} chunk {chunk} bf16 {bf16}", flush=True)
    assert _more_workspace(bt, t, d, n) > 0
    g = torch.Generator().manual_seed(t + d + n)
    dtype = torch.bfloat16 if bf16 else torch.float32

    def rand(*s):
        return torch.randn(*s, generator=g)
    leaves = [rand(bt, t, d).to(DEV, dtype), F.softplus(rand(bt, t, d) - 4).to(DEV, dtype),
              (0.05 + torch.rand(d, n, generator=g)).to(DEV), rand(bt, t, n).to(DEV, dtype),
              rand(bt, t, n).to(DEV, dtype)]   # slow decays: carries matter
    leaves = [v.requires_grad_() for v in leaves]

    def run():
        return _grads(selective_scan_hip(*leaves, chunk=chunk, return_state=True), leaves, 1)
    _compare(*_both(run), bf16)


def test_gated_scan_in_many_segments():
    bt, t, d, n = 1, 1500, 68, 16
    print(f"[case] gated segments {bt}x{t}x{d}x{n}", flush=True)
    assert _more_workspace(bt, t, d, n) > 0
    g = torch.Generator().manual_seed(3)
    proj = torch.randn(bt, t, d + 2 * n, generator=g).to(DEV).requires_grad_()
    x = torch.randn(bt, t, d, generator=g).to(DEV).requires_grad_()
    a = torch.randn(d, n, generator=g).to(DEV).requires_grad_()
    bias = torch.randn(d, generator=g).to(DEV).requires_grad_()
    leaves = [x, proj, a, bias]

    def run():
        out = selective_scan_gated(x, proj[..., :d], a, proj[..., d:d + n], proj[..., d + n:],
                                   0.001, 0.1, return_state=True, dt_bias=bias)
        return _grads(out, leaves, 2)
    _compare(*_both(run), False)


@pytest.mark.parametrize("bt,t,d,n,chunk", [
    (6, 500, 1100, 4, 16), (5, 700, 1000, 12, 100), (7, 333, 1000, 16, 32), (7, 400, 1000, 24, 16),
    (10, 300, 1000, 40, 64), (13, 250, 1200, 64, 16), (13, 250, 1200, 20, 48)])
def test_middle_grids_equal_one_segment(bt, t, d, n, chunk):
    """From two fifths of a block per CU to just under two, at each plan."""
    print(f"[case] middle {bt}x{t}x{d}x{n} chunk {chunk}", flush=True)
    g = torch.Generator().manual_seed(t + d + n)

    def rand(*s):
        return torch.randn(*s, generator=g).to(DEV)
    leaves = [v.requires_grad_() for v in (rand(bt, t, d), F.softplus(rand(bt, t, d) - 4),
                                           rand(d, n).abs(), rand(bt, t, n), rand(bt, t, n))]
    auto, one = _both(lambda: _grads(
        selective_scan_hip(*leaves, chunk=chunk, return_state=True), leaves, 1))
    _compare(auto, one, False)


@pytest.mark.parametrize("n,chunk,gated", [(17, 16, False), (24, 32, False), (25, 64, True),
                                           (32, 16, True), (32, 32, True), (32, 48, False)])
def test_dense_gradients_of_middle_states_equal_two_states_per_lane(n, chunk, gated):
    """d_state 17..32 on a grid of a block per CU or more: four states per lane
    in the gradient pass against two in every pass."""
    bt, t, d = 8, 100, 1000 + 4 * (n % 2)
    print(f"[case] dense {bt}x{t}x{d}x{n} chunk {chunk} gated {gated}", flush=True)
    assert bt * ((d + 31) // 32) >= _native.library().mhs_cu_count()
    g = torch.Generator().manual_seed(n + chunk)

    def rand(*s):
        return torch.randn(*s, generator=g).to(DEV)
    leaves = [v.requires_grad_() for v in (rand(bt, t, d), F.softplus(rand(bt, t, d) - 4),
                                           rand(d, n).abs(), rand(bt, t, n), rand(bt, t, n))]

    def run():
        out = (selective_scan_gated(*leaves, 0.001, 0.1, chunk=chunk, return_state=True) if gated
               else selective_scan_hip(*leaves, chunk=chunk, return_state=True))
        return _grads(out, leaves, 1)
    auto = run()
    _native.set_variant(2)
    try:
        two = run()
    finally:
        _native.set_variant(0)
    _compare(auto, two, False)


@pytest.mark.parametrize("bt,t,d,n,eighth", [(4, 512, 1536, 32, 8), (2, 2048, 1792, 16, 19),
                                            (4, 1024, 1024, 64, 11)])
def test_long_segments_do_not_add_error(bt, t, d, n, eighth):
    """dAneg's error against float64 where the automatic split takes fewer
    segments than those of `eighth` chunks each that the grid's
    blocks per CU would give. Bar (relative 2-norm): a chain of m = 16 eighth
    additions of terms of any sign rounds each by about 0.4 2^-24 of a running
    sum that grows as the root of its length, 0.4 2^-24 sqrt(m / 2) in all,
    and 2 2^-24 for the terms: 3.1e-7, 4.1e-7, 3.4e-7. (One chain over the
    longer segments: 4.6e-7, 4.5e-7, 4.7e-7.)"""
    print(f"[case] dAneg error {bt}x{t}x{d}x{n}", flush=True)
    arrs = oracle.make_inputs(bt, t, d, n, seed=1, style="bench")
    dy = np.random.default_rng(2).standard_normal((bt, t, d), dtype=np.float32)
    leaves = [torch.from_numpy(a).to(DEV).requires_grad_() for a in arrs]
    y = selective_scan_hip(*leaves, chunk=16)
    da = torch.autograd.grad(y, leaves[2], torch.from_numpy(dy).to(DEV))[0]
    ref = oracle.scan_bwd(*arrs, dy)[2]
    rel = np.linalg.norm(da.cpu().double().numpy() - ref) / np.linalg.norm(ref)
    assert rel <= 2.0 ** -24 * (0.4 * (16 * eighth / 2) ** 0.5 + 2), rel
