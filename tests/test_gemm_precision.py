"""The fp32 products on the bf16 matrix cores hold fp32's precision: operands
of which one partial product alone decides the result (exact, so that no
partial product can be missing anywhere), and the error and bias of long sums
beside the library's fp32 product of the same operands.
"""
from __future__ import annotations

import pytest
import torch

from mamba_metal_scan_amd import _native

DEV = "cuda"
FORMS = {"nt": _native.GEMM_NT, "nn": _native.GEMM_NN, "tn": _native.GEMM_TN}
KEPT = [(0, 0), (1, 0), (0, 1), (2, 0), (1, 1), (0, 2)]   # parts of a, of b


def isolating(i, j, m, n, k, seed=0):
    """a (m, k), b (n, k) and a b^T, where the products of a's part i with b's
    part j make up the whole result: groups of 4 k's whose other partial
    products cancel exactly. u has the parts 1, e and e^2, e = 2^-10."""
    e = 2.0 ** -10
    u = [1.0, 1.0 + e, 1.0 + e + e * e]
    g = torch.Generator().manual_seed(seed + 3 * i + j)
    sign = (torch.randint(0, 2, (n, k // 4), generator=g) * 2 - 1).double()
    row = 2.0 ** torch.randint(-3, 4, (m, 1), generator=g).double()

    def quads(i_first, second):
        """4 k's: the value with part i, and the one without it, negated."""
        hi = u[i_first]
        lo = u[i_first - 1] if i_first else 0.0
        return [hi, -lo, -hi, lo] if not second else [hi, hi, lo, lo]
    a = (row * torch.tensor(quads(i, False)).double().repeat(k // 4))
    b = torch.tensor(quads(j, True)).double().repeat(k // 4) * sign.repeat_interleave(4, 1)
    return a.float(), b.float(), a @ b.t()


def emulated(a, b, kept):
    """a b^T in 64 bits from the products `kept` of the bf16 parts."""
    def parts(x):
        out = []
        for _ in range(3):
            out.append(x.to(torch.bfloat16).float())
            x = x - out[-1]
        return [p.double() for p in out]
    pa, pb = parts(a), parts(b)
    return sum(pa[i] @ pb[j].t() for i, j in kept)


@pytest.mark.parametrize("i,j", KEPT)
def test_isolating_operands_need_their_product(i, j):
    """On the CPU: the six products give the exact result, five without (i, j)
    do not."""
    a, b, want = isolating(i, j, 6, 5, 48)
    assert want.abs().max() > 0 and torch.equal(a.double() @ b.double().t(), want)
    assert torch.equal(emulated(a, b, KEPT), want)
    less = emulated(a, b, [p for p in KEPT if p != (i, j)])
    assert (less - want).norm() >= 0.9 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("m,n", [(40, 36), (2048, 1024)])   # small and large tiles
def test_every_partial_product(form, m, n):
    """K 208: 13 tiles, in both LDS buffers and both signs."""
    print(f"[case] partial products {form} {m}x{n}", flush=True)
    f = FORMS[form]
    for i, j in KEPT:
        a, b, want = isolating(i, j, m, n, 208)
        a, b = a.to(DEV), b.to(DEV)
        x = a.t().contiguous() if f == _native.GEMM_TN else a
        y = b if f == _native.GEMM_NT else b.t().contiguous()
        assert torch.equal(product(x, y, f).double().cpu(), want), (i, j)


def product(a, b, form):
    """The C entry at any size (the Python layer sends small ones elsewhere)."""
    lib = _native.library()
    m, n, k = _native._gemm_sizes(a, b, form)
    out = torch.full((m, n), float("nan"), device=DEV)
    need = lib.mhs_gemm_workspace_bytes(m, n, k)
    ws = torch.empty(max(need, 256), dtype=torch.uint8, device=DEV)
    rc = lib.mhs_gemm_f32(form, a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0),
                          out.data_ptr(), n, m, n, k, 0, ws.data_ptr(), need,
                          torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.mhs_last_error()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("m,n,k", [(1024, 1024, 256), (2048, 1464, 1432), (2048, 2048, 8192)])
@pytest.mark.parametrize("positive", [False, True])
def test_error_and_bias_of_long_sums(form, m, n, k, positive):
    """Relative 2-norm error against float64 no larger than 1.1 times the
    library product's (measured 0.3 to 0.9 of it: 2e-7 to 1e-6; one bf16 part
    of each operand would have 2e-3, two 4e-6), and a mean error below 3e-8 of
    the rms (measured up to 3e-9). Sums that round down without the
    alternation of signs are low by about (6 K / 16) 2^-24 / 4 of a same-sign
    sum, 8e-6 at K 1432."""
    print(f"[case] product error {form} {m}x{n}x{k} positive {positive}", flush=True)
    f = FORMS[form]
    g = torch.Generator(DEV).manual_seed(k)
    a = torch.randn((k, m) if f == _native.GEMM_TN else (m, k), device=DEV, generator=g)
    b = torch.randn((n, k) if f == _native.GEMM_NT else (k, n), device=DEV, generator=g)
    if positive:
        a, b = a.abs(), b.abs()
    ad, bd = a.double(), b.double()
    ref = (ad.t() if f == _native.GEMM_TN else ad) @ (bd.t() if f == _native.GEMM_NT else bd)
    err = product(a, b, f).double() - ref
    lib = _native._mm(a, b, f).double() - ref
    assert err.norm() <= 1.1 * lib.norm(), (err.norm() / ref.norm(), lib.norm() / ref.norm())
    assert err.mean().abs() <= 3e-8 * ref.square().mean().sqrt(), err.mean()
