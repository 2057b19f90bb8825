"""GPU parity of the fp32 matrix products on the bf16 matrix cores with
float64, at the edges of their tiles (128 x 128, 16 deep) and of the split
over k.

Bar, per element: |got - ref| <= (6 K / 16 + S + 8) 2^-23 sum_k |a_k b_k|: the
product of a k tile is six additions to the sum, each rounding (or
truncating) by at most 2^-23 of the running sum, which sum_k |a_k b_k| bounds;
S more additions sum the splits, and the dropped parts and the parts' own
roundings stay below the 8.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

from mamba_metal_scan_amd import _native
from mamba_metal_scan_amd._native import GEMM_NN, GEMM_NT, GEMM_TN
from mamba_metal_scan_amd.linear import LinearHIP

pytestmark = pytest.mark.gpu
DEV = "cuda"
FORMS = {"nt": GEMM_NT, "nn": GEMM_NN, "tn": GEMM_TN}


def _operands(form, m, n, k, seed=0, pad=0):
    g = torch.Generator().manual_seed(seed + m * 7 + n * 3 + k)

    def mat(r, c):
        return torch.randn(r, c + pad, generator=g).to(DEV)[:, :c]
    return (mat(k, m) if form == GEMM_TN else mat(m, k),
            mat(n, k) if form == GEMM_NT else mat(k, n))


def _ref(a, b, form):
    a = a.t() if form == GEMM_TN else a
    return a @ (b.t() if form == GEMM_NT else b)


def _call(a, b, form, out, accumulate=False):
    """The C entry at any size (the Python layer sends small ones elsewhere)."""
    lib = _native.library()
    m, n, k = _native._gemm_sizes(a, b, form)
    need = lib.mhs_gemm_workspace_bytes(m, n, k)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
    rc = lib.mhs_gemm_f32(form, a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0),
                          out.data_ptr(), out.stride(0), m, n, k, accumulate, ws.data_ptr(),
                          need, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.mhs_last_error()
    torch.cuda.synchronize()
    return need


def _assert_bounded(got, a, b, form, k, extra=0):
    ref = _ref(a.double(), b.double(), form)
    bound = (6 * k / 16 + 32 + 8) * 2.0 ** -23 * _ref(a.double().abs(), b.double().abs(), form)
    bad = ((got.double() - extra - ref).abs() > bound + 2.0 ** -22 * abs(extra)).sum().item()
    assert bad == 0, f"{bad} elements off"


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("m,n,k", [(1, 4, 4), (128, 128, 16), (129, 132, 20), (127, 260, 1432),
                                   (300, 8, 36), (257, 128, 8192)])
def test_products_match_float64(form, m, n, k):
    print(f"[case] gemm {form} {m}x{n}x{k}", flush=True)
    f = FORMS[form]
    for pad in (0, 4):
        a, b = _operands(f, m, n, k, pad=pad)
        out = torch.full((m, n), float("nan"), device=DEV)
        _call(a, b, f, out)
        _assert_bounded(out, a, b, f, k)
        _call(a, b, f, out.fill_(0.5), accumulate=True)
        _assert_bounded(out, a, b, f, k, extra=0.5)


@pytest.mark.parametrize("form,m,n,k", [("nn", 33, 7, 64), ("tn", 33, 7, 37), ("nt", 33, 7, 64)])
def test_widths_that_are_no_multiple_of_four(form, m, n, k):
    f = FORMS[form]
    a, b = _operands(f, m, n, k)
    out = torch.full((m, n), float("nan"), device=DEV)
    assert _call(a, b, f, out) == 0   # never split
    _assert_bounded(out, a, b, f, k)


@pytest.mark.parametrize("form,m,n,k", [("nt", 33, 7, 8192), ("nn", 129, 131, 9000),
                                        ("tn", 130, 642, 9001), ("tn", 64, 64, 20000)])
def test_long_sums_of_any_width_are_split(form, m, n, k):
    """More than 4096 k's are summed in several chains at any width and row
    stride of c: the error stays below a plain fp32 product's (one chain of
    MFMA additions of 32768 has 1.5 times it)."""
    print(f"[case] gemm {form} {m}x{n}x{k}", flush=True)
    f = FORMS[form]
    a, b = _operands(f, m, n, k)
    ref = _ref(a.double(), b.double(), f)
    lib = (_native._mm(a, b, f).double() - ref).norm() / ref.norm()
    for pad in (0, 1):
        out = torch.full((m, n + pad), float("nan"), device=DEV)[:, :n]
        assert _call(a, b, f, out) >= 2 * m * n * 4
        _assert_bounded(out, a, b, f, k)
        rel = (out.double() - ref).norm() / ref.norm()
        assert rel <= 1.1 * lib, (rel.item(), lib.item())
        _call(a, b, f, out.fill_(0.5), accumulate=True)
        _assert_bounded(out, a, b, f, k, extra=0.5)


def test_infinities_and_nan_come_out_as_in_fp32():
    a, b = _operands(GEMM_NT, 200, 140, 64)
    a[3, 5], a[7, 9], b[11, 2], a[20, 1] = float("inf"), float("nan"), -float("inf"), 3.4e38
    a[21], b[30] = 1e30, 1e30
    ref = _ref(a, b, GEMM_NT)
    out = torch.empty(200, 140, device=DEV)
    _call(a, b, GEMM_NT, out)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(out), inf) and torch.equal(out[inf], ref[inf])


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("m,n,k", [(33, 36, 20), (129, 132, 100), (257, 128, 8192)])
def test_non_finite_elements_of_every_form(form, m, n, k):
    """Infinities, NaN and values whose parts overflow, in tiles with edges and
    a split of k: the other elements keep their values."""
    print(f"[case] non-finite gemm {form} {m}x{n}x{k}", flush=True)
    f = FORMS[form]
    a, b = _operands(f, m, n, k)
    ka, kb = (a.t() if f == GEMM_TN else a), (b if f == GEMM_NT else b.t())   # rows by k
    ka[m - 1, k - 1], ka[2, 0], kb[n - 2, k // 2] = float("nan"), float("inf"), -float("inf")
    ka[5, 1], ka[6] = 3.4e38, 0.0
    kb[:, 1] *= 1e-3
    ref = _ref(a.double(), b.double(), f)
    out = torch.empty(m, n, device=DEV)
    _call(a, b, f, out)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(out), inf) and torch.equal(out.double()[inf], ref[inf])
    fin = torch.isfinite(ref)
    bound = (6 * k / 16 + 40) * 2.0 ** -23 * _ref(a.double().abs(), b.double().abs(), f)
    assert ((out.double() - ref).abs() <= bound)[fin].all()


def test_non_finite_products_stay_fast():
    """All NaN: the recomputation is bound by the fp32 matrix rate, a few times
    the finite product (and not the hundreds of a loop per element)."""
    a, b = _operands(GEMM_NT, 2048, 1464, 1432)
    out = torch.empty(2048, 1464, device=DEV)
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    times = []
    for x in (a, torch.full_like(a, float("nan"))):
        _call(x, b, GEMM_NT, out)
        start.record()
        for _ in range(3):
            _call(x, b, GEMM_NT, out)
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end))
    assert torch.isnan(out).all()
    assert times[1] < 15 * times[0], times


@pytest.mark.parametrize("scale", [1e-12, 1e-19, 1e15])
def test_scales(scale):
    a, b = (v * scale for v in _operands(GEMM_NT, 130, 128, 256))
    out = torch.empty(130, 128, device=DEV)
    _call(a, b, GEMM_NT, out)
    _assert_bounded(out, a, b, GEMM_NT, 256)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("m,n,k", [(33, 36, 20), (200, 132, 300), (257, 128, 8192)])
@pytest.mark.parametrize("scale", [1e-30, 1e-34, 1e-37])
def test_small_operands_keep_their_bits(form, m, n, k, scale):
    """Rows of one operand whose bf16 parts would run into the subnormals (the
    other operand large, so that the results do not): all rows, and one. The
    bar is that of the plain fp32 products which such tiles take: a sum of k
    terms in any order, sqrt(k) / 2 roundings of at most 2^-24, with a margin
    of 2, relative to the 2-norm."""
    f = FORMS[form]
    for which in ("a", "b"):
        for rows in (slice(None), slice(3, 4)):
            a, b = _operands(f, m, n, k)
            ka, kb = (a.t() if f == GEMM_TN else a), (b if f == GEMM_NT else b.t())
            small, large = (ka, kb) if which == "a" else (kb, ka)
            small[rows] *= scale
            large *= 1e20
            out = torch.empty(m, n, device=DEV)
            _call(a, b, f, out)
            got, ref = out.double(), _ref(a.double(), b.double(), f)
            if which == "b":
                got, ref = got.t(), ref.t()
            rel = (got - ref)[rows].norm() / ref[rows].norm()
            assert rel <= k ** 0.5 * 2.0 ** -24 + 2.0 ** -23, (which, rows, rel.item())


def test_linear_gradients():
    """A layer large enough for the HIP products in every direction."""
    rows, k, n = 2048, 640, 1464
    assert _native.gemm_preferred(rows, n, k)
    g = torch.Generator().manual_seed(1)
    x = torch.randn(rows, k, generator=g).to(DEV).requires_grad_()
    w = torch.randn(n, k, generator=g).to(DEV).requires_grad_()
    dy = torch.randn(rows, n, generator=g).to(DEV)
    y = LinearHIP.apply(x, w)
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    _assert_bounded(y.detach(), x.detach(), w.detach(), GEMM_NT, k)
    _assert_bounded(dx, dy, w.detach(), GEMM_NN, n)
    _assert_bounded(dw, dy, x.detach(), GEMM_TN, rows)
