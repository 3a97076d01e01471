"""FP32 products as BF16 terms (the default it_gemm FP32 path) at the edges of their tiles and on
operands the split has to hand over to the FP32 units.

Bound per element, against the float64 product of the same operands: an element split into three
BF16 terms keeps 24 significand bits, the left-out term products are below 2^-24 of a product, and
the running sums round once per 8 products, so |error| <= (K / 8 + 16) 2^-23 (|A|.|B|)_ij.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from irontensor_amd import _lib, profiler, synth
from tests.numerics import op

pytestmark = pytest.mark.gpu

LAYOUTS = [(0, 0), (0, 1), (1, 0), (1, 1)]


def _operands(seed, m, n, k, ta, tb):
    a = synth.normal(seed, (k, m) if ta else (m, k))
    b = synth.normal(seed + 1, (n, k) if tb else (k, n), std=0.02)
    return a, b


def _check(got, a, b, ta, tb, k, extra=0.0):
    A, B = op(a, ta).astype(np.float64), op(b, tb).astype(np.float64)
    bound = (k / 8 + 16) * 2.0 ** -23 * (np.abs(A) @ np.abs(B)) + 1e-30
    worst = float(np.max(np.abs(got - (A @ B + extra)) / bound))
    assert worst <= 1.0, f"error {worst:.2f} times its bound"


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 768, 256), (63, 65, 31), (64, 32, 33), (65, 33, 32), (129, 127, 97),
                                   (300, 701, 1000), (128, 128, 64), (1025, 515, 70), (257, 40, 3000)])
def test_layouts_and_edges(it, m, n, k, ta, tb):
    a, b = _operands(m + 7 * n + k, m, n, k, ta, tb)
    c = it.gemm(it.Tensor.from_f32_slice(a, a.shape), it.Tensor.from_f32_slice(b, b.shape), trans_a=bool(ta),
                trans_b=bool(tb))
    _check(c.numpy(), a, b, ta, tb, k)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(512, 384, 4096), (640, 1152, 96), (192, 200, 40)])
def test_strided_unaligned_operands(it, m, n, k, ta, tb):
    """Rows at any element alignment: operands and output inside wider buffers, starting at odd columns,
    whose surrounding elements are NaN (they may be read past K and past an edge, never used) or must
    stay untouched."""
    a, b = _operands(31 + m, m, n, k, ta, tb)
    ctx = it.Context.global_()

    def wide(x, fill):
        w = np.full((x.shape[0] + 2, x.shape[1] + 7), fill, np.float32)
        w[1:-1, 3:-4] = x
        return it.Tensor.from_f32_slice(w, list(w.shape)), w.shape[1]

    (A, lda), (B, ldb) = wide(a, np.nan), wide(b, np.nan)
    Cw, ldc = wide(np.zeros((m, n), np.float32), 7.0)
    ptr = lambda t, ld: C.c_void_p(t.ptr + 4 * (ld + 3))
    st = ctx.lib.it_gemm(ctx.handle, 0, 0, ta, tb, m, n, k, 1.0, ptr(A, lda), lda, 0, ptr(B, ldb), ldb, 0, 0.0,
                         ptr(Cw, ldc), ldc, 0, 1, None)
    assert st == 0
    got = Cw.numpy()
    _check(got[1:-1, 3:-4], a, b, ta, tb, k)
    edge = got.copy()
    edge[1:-1, 3:-4] = 7.0
    assert np.all(edge == 7.0)


@pytest.mark.parametrize("ta,tb", [(0, 1), (1, 0)])
@pytest.mark.parametrize("m,n,k", [(70, 66, 80), (300, 260, 520)])
def test_nonfinite_and_extreme_operands(it, m, n, k, ta, tb):
    """An infinity, a NaN, the type's largest value and subnormals give what the FP32 units give: the
    same non-finite elements, and the finite ones within the bound."""
    a, b = _operands(5, m, n, k, ta, tb)
    big = np.finfo(np.float32).max
    va, vb = op(a, ta), op(b, tb)  # views
    va[3, 5] = np.inf
    va[17, 2] = -np.inf
    va[40, k - 1] = np.nan
    va[50, 7] = big
    va[51, 7] = -big
    vb[9, 11] = np.inf
    va[60, :] = 1e-40
    A, B = it.Tensor.from_f32_slice(a, a.shape), it.Tensor.from_f32_slice(b, b.shape)
    got = it.gemm(A, B, trans_a=bool(ta), trans_b=bool(tb)).numpy()
    units = it.Tensor.empty([m, n])
    epi = _lib.Epilogue(flags=_lib.IT_EPI_F32_UNITS)
    st = A.ctx.lib.it_gemm(A.ctx.handle, 0, 0, ta, tb, m, n, k, 1.0, C.c_void_p(A.ptr), a.shape[1], 0,
                           C.c_void_p(B.ptr), b.shape[1], 0, 0.0, C.c_void_p(units.ptr), n, 0, 1, C.byref(epi))
    assert st == 0
    ref = units.numpy()
    fine = np.isfinite(ref)
    assert np.array_equal(fine, np.isfinite(got)) and np.array_equal(np.isnan(ref), np.isnan(got))
    assert np.array_equal(ref[~fine & ~np.isnan(ref)], got[~fine & ~np.isnan(ref)])
    with np.errstate(all="ignore"):
        A64, B64 = va.astype(np.float64), vb.astype(np.float64)
        exact, size = A64 @ B64, np.abs(A64) @ np.abs(B64)
        err = np.abs(got.astype(np.float64) - exact)[fine]
    # (sums of subnormal results round to FP32's smallest step, 2^-149, once per product)
    assert np.all(err <= (k / 8 + 16) * 2.0 ** -23 * size[fine] + 2.0 ** -140)


@pytest.mark.parametrize("rows,h,f", [(65, 33, 49), (200, 256, 688), (1024, 128, 2048)])
def test_swiglu_and_bias(it, rows, h, f):
    x, wg, wu = synth.normal(1, (rows, h)), synth.normal(2, (f, h), std=0.05), synth.normal(3, (f, h), std=0.05)
    bias = synth.normal(4, (2 * f,), std=0.1)
    T = it.Tensor.from_f32_slice
    hh, g, u = it.swiglu_up(T(x, x.shape), T(wg, wg.shape), T(wu, wu.shape), bias=T(bias, [2 * f]))
    _check(g.numpy(), x, wg, 0, 1, h, bias[None, :f].astype(np.float64))
    _check(u.numpy(), x, wu, 0, 1, h, bias[None, f:].astype(np.float64))
    gate, up = g.numpy().astype(np.float64), u.numpy().astype(np.float64)
    ref = gate / (1 + np.exp(-gate)) * up
    assert np.max(np.abs(hh.numpy() - ref)) <= 4e-6 * np.max(np.abs(ref))


def test_training_step_on_the_fp32_units_or_terms(it):
    """f32_units=False takes the terms: the first step's gradients agree to FP32 rounding."""
    from irontensor_amd.step import ModelShape
    from irontensor_amd.train import TrainStep

    shape = ModelShape("small", 2, 128, 2, 64, 176, 1000, 2, 64)
    grads = []
    for units in (True, False):
        st = TrainStep(shape, seed=5, f32_units=units)
        st.step()
        grads.append([t.numpy().astype(np.float64) for t in st.grads])
    for x, y in zip(*grads):
        assert np.linalg.norm(x - y) <= 2e-5 * np.linalg.norm(x)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(70, 66, 80), (192, 200, 40), (640, 1152, 96), (512, 300, 4096)])
@pytest.mark.parametrize("a_exp,b_exp", [(-110, 90), (-118, 100), (-126, 100), (-140, 120), (100, -125), (113, -60),
                                         (70, 30)])
def test_small_and_large_operands(it, ta, tb, m, n, k, a_exp, b_exp):
    """Operands near either end of FP32's range keep their 24 bits: below 2^-110 the last of three unscaled
    terms would lose its own (2^-126: all but 8 bits of an element), and subnormal operands have no more
    bits than they show. Elements of 2^113 or sums above 2^96 leave the scaled terms' range."""
    a, b = _operands(3, m, n, k, ta, tb)
    a, b = np.ldexp(a, a_exp).astype(np.float32), np.ldexp(b / np.float32(0.02), b_exp).astype(np.float32)
    c = it.gemm(it.Tensor.from_f32_slice(a, a.shape), it.Tensor.from_f32_slice(b, b.shape), trans_a=bool(ta),
                trans_b=bool(tb))
    _check(c.numpy(), a, b, ta, tb, k)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(300, 260, 520), (1100, 1500, 333), (4100, 2300, 130), (520, 260, 4099)])
def test_infinities_in_every_wave(it, ta, tb, m, n, k):
    """An infinity in every 13th row of A (at another k each) sends every wave's tile to the second
    computation: those rows are the infinities of B's signs, the others finite and within the bound."""
    a, b = _operands(11, m, n, k, ta, tb)
    va, vb = op(a, ta), op(b, tb)  # views
    rows = np.arange(0, m, 13)
    cols = (rows * 7 + 3) % k
    va[rows, cols] = np.inf
    got = it.gemm(it.Tensor.from_f32_slice(a, a.shape), it.Tensor.from_f32_slice(b, b.shape), trans_a=bool(ta),
                  trans_b=bool(tb)).numpy()
    assert np.array_equal(got[rows], np.where(vb[cols] > 0, np.inf, -np.inf).astype(np.float32))
    rest = np.delete(np.arange(m), rows)
    _check(got[rest], np.ascontiguousarray(va[rest]), np.ascontiguousarray(vb), 0, 0, k)


def _keys(it, fn):
    ctx = it.Context.global_()
    profiler.reset(ctx)
    profiler.enable(ctx)
    assert fn() == 0
    keys = list(profiler.stats(ctx))
    profiler.enable(ctx, False)
    return keys


@pytest.mark.parametrize("tile,splits,ta,tb,m,n,k", [
    ("256x128", 1, 0, 0, 1510, 2863, 1283), ("256x128", 1, 0, 1, 1410, 2803, 1241), ("256x128", 8, 0, 0, 837, 971, 3202),
    ("256x128", 2, 0, 1, 2281, 1353, 1104), ("128x128", 1, 1, 1, 1985, 1681, 226), ("128x128", 3, 1, 0, 1766, 1293, 1585),
    ("128x128", 3, 0, 0, 1221, 1000, 1087), ("128x128", 1, 0, 1, 1173, 2713, 283), ("128x128", 6, 0, 1, 772, 1345, 1666),
    ("64x64", 1, 1, 0, 291, 246, 21), ("64x64", 3, 0, 0, 2154, 226, 1390), ("64x64", 5, 0, 1, 149, 1887, 2467),
    ("64x64", 8, 1, 0, 307, 220, 1007), ("64x64", 12, 1, 1, 655, 37, 1435), ("64x64", 1, 0, 1, 1470, 390, 17),
    ("64x32", 1, 0, 0, 28, 594, 22), ("64x32", 5, 1, 1, 31, 355, 557), ("64x32", 12, 0, 1, 212, 126, 1830),
    ("64x32", 3, 0, 0, 77, 1203, 821), ("64x32", 24, 1, 0, 96, 35, 2973)])
def test_every_tile_at_its_edges(it, tile, splits, ta, tb, m, n, k):
    """Each tile shape and layout at sizes it does not divide, operands and output at odd columns of wider
    buffers whose other elements are NaN (the output's: untouched). Gaussian data against float64: every
    element within the bound, and the whole within 4e-7, where losing one of the 2^-16 term products
    (each operand's terms are 2^-9 / sqrt(3) of the one before in the mean) would show 7e-7."""
    a, b = _operands(41, m, n, k, ta, tb)
    ctx = it.Context.global_()

    def wide(x, fill):
        w = np.full((x.shape[0] + 2, x.shape[1] + 7), fill, np.float32)
        w[1:-1, 3:-4] = x
        return it.Tensor.from_f32_slice(w, list(w.shape)), w.shape[1]

    (A, lda), (B, ldb) = wide(a, np.nan), wide(b, np.nan)
    Cw, ldc = wide(np.zeros((m, n), np.float32), 7.0)
    ptr = lambda t, ld: C.c_void_p(t.ptr + 4 * (ld + 3))
    keys = _keys(it, lambda: ctx.lib.it_gemm(ctx.handle, 0, 0, ta, tb, m, n, k, 1.0, ptr(A, lda), lda, 0, ptr(B, ldb), ldb,
                                             0, 0.0, ptr(Cw, ldc), ldc, 0, 1, None))
    assert keys == [f"gemm_f32_{'NT'[ta]}{'NT'[tb]}_{tile}|[{m},{n},{k}]x1 s{splits}"], keys
    got = Cw.numpy()
    y = got[1:-1, 3:-4].astype(np.float64)
    _check(y, a, b, ta, tb, k)
    exact = op(a, ta).astype(np.float64) @ op(b, tb).astype(np.float64)
    assert np.linalg.norm(y - exact) <= 4e-7 * np.linalg.norm(exact)
    got[1:-1, 3:-4] = 7.0
    assert np.all(got == 7.0)
