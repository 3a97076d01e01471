"""FP32 products that ask for the FP32 units (IT_EPI_F32_UNITS, the training step's default): the tiles
that other FP32 products reach only with few rows.

Bound per element, against the float64 product of the same operands: K products and sums, each rounded
once, in any order, so |error| <= (K + 2) 2^-24 (|A|.|B|)_ij.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from irontensor_amd import _lib, profiler, synth
from tests.numerics import op

pytestmark = pytest.mark.gpu


def _within(got, a, b, extra=0.0):
    """a.b^T in float64 against got."""
    A, B = a.astype(np.float64), b.astype(np.float64)
    bound = (a.shape[1] + 2) * 2.0 ** -24 * (np.abs(A) @ np.abs(B).T) + 2.0 ** -23 * np.abs(extra)
    worst = float(np.max(np.abs(got - (A @ B.T + extra)) / bound))
    assert worst <= 1.0, f"error {worst:.2f} times its bound"


@pytest.mark.parametrize("rows,h,f", [(65, 64, 52), (200, 256, 688), (4096, 256, 688), (130, 32, 36), (64, 96, 4),
                                      (1000, 36, 700), (129, 35, 33), (256, 128, 2048)])
def test_swiglu_weights_inside_nan(it, rows, h, f):
    """Widths that no tile divides: the rows past X, past the gate and past the up weight are NaN and
    reach no result. Descriptor loads where h is a multiple of 32 (200 x 256 x 688), masked and
    bounds-checked ones elsewhere, plain ones on whole tiles."""
    print(f"[units swiglu] {rows}x{h}x{f}", flush=True)
    x, wg, wu = synth.normal(1, (rows, h)), synth.normal(2, (f, h), std=0.05), synth.normal(3, (f, h), std=0.05)
    bias = synth.normal(4, (2 * f,), std=0.1)
    gap = np.full((70, h), np.nan, np.float32)
    X = it.Tensor.from_f32_slice(np.concatenate([x, gap]), [rows + 70, h])
    W = it.Tensor.from_f32_slice(np.concatenate([gap, wg, gap, wu, gap]), [2 * f + 210, h])
    Bias = it.Tensor.from_f32_slice(bias, [2 * f])
    outs = [it.Tensor.from_f32_slice(np.full((rows + 2, f), 7.0, np.float32), [rows + 2, f]) for _ in range(3)]
    inner = [t.ptr + 4 * f for t in outs]
    epi = _lib.Epilogue(flags=_lib.IT_EPI_SWIGLU | _lib.IT_EPI_BIAS | _lib.IT_EPI_F32_UNITS, bias=Bias.ptr,
                        B2=W.ptr + 4 * h * (f + 140), gate_out=inner[1], up_out=inner[2])
    st = X.ctx.lib.it_gemm(X.ctx.handle, 0, 0, 0, 1, rows, f, h, 1.0, C.c_void_p(X.ptr), h, 0,
                           C.c_void_p(W.ptr + 4 * h * 70), h, 0, 0.0, C.c_void_p(inner[0]), f, 0, 1, C.byref(epi))
    assert st == 0
    hh, g, u = (t.numpy() for t in outs)
    for t in (hh, g, u):
        assert np.all(t[0] == 7.0) and np.all(t[-1] == 7.0)
    _within(g[1:-1], x, wg, bias[None, :f].astype(np.float64))
    _within(u[1:-1], x, wu, bias[None, f:].astype(np.float64))
    gate, up = g[1:-1].astype(np.float64), u[1:-1].astype(np.float64)
    ref = gate / (1 + np.exp(-gate)) * up
    assert np.max(np.abs(hh[1:-1] - ref)) <= 4e-6 * np.max(np.abs(ref))


@pytest.mark.parametrize("units", [False, True])
@pytest.mark.parametrize("tokens,vocab,h", [(4096, 16384, 256), (129, 1001, 65), (70, 34, 33), (333, 5003, 300)])
def test_cross_entropy_operand(it, units, tokens, vocab, h):
    """dh = G.E and dE = G^T.h with G = (softmax - onehot) / T rebuilt from the logits, on the terms and on the
    FP32 units, against float64; an infinity in the other operand reaches its own column alone (the
    terms' second computation rebuilds G as well)."""
    from irontensor_amd import train_ops
    logits = synth.normal(1, (tokens, vocab), std=3.0)
    hid, emb = synth.normal(2, (tokens, h)), synth.normal(3, (vocab, h), std=0.02)
    tg = synth.tokens(4, tokens, vocab)
    hid[min(40, tokens - 1), h - 1] = np.inf
    emb[min(40, vocab - 1), 0] = np.inf
    T = it.Tensor.from_f32_slice
    L, Hd, E = T(logits, logits.shape), T(hid, hid.shape), T(emb, emb.shape)
    _, _, stats = train_ops.cross_entropy_stats(L, tg)
    ids = train_ops.upload_ids(tg, vocab)
    epi = _lib.Epilogue(flags=_lib.IT_EPI_XENT_A | (_lib.IT_EPI_F32_UNITS if units else 0), xent_stats=stats.ptr,
                        xent_targets=ids.ptr, xent_scale=1.0 / tokens)
    dh, de = it.Tensor.empty([tokens, h]), it.Tensor.empty([vocab, h])
    ctx = L.ctx
    for ta, a, b, c, m, k in ((0, L, E, dh, tokens, vocab), (1, L, Hd, de, vocab, tokens)):
        st = ctx.lib.it_gemm(ctx.handle, 0, 0, ta, 0, m, h, k, 1.0, C.c_void_p(a.ptr), vocab, 0, C.c_void_p(b.ptr), h,
                             0, 0.0, C.c_void_p(c.ptr), h, 0, 1, C.byref(epi))
        assert st == 0
    x = logits.astype(np.float64)
    p = np.exp(x - x.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    p[np.arange(tokens), tg] -= 1.0
    p /= tokens
    # The sums' bound, and the rebuilt element's own: exp2 of a rounded argument, about 1e-6 of it.
    for got, A, B, bad in ((dh.numpy(), p, emb, 0), (de.numpy(), p.T, hid, h - 1)):
        assert not np.isfinite(got[:, bad]).any()
        fine = np.arange(h) != bad
        A, B = np.ascontiguousarray(A), B[:, fine].astype(np.float64)
        n = A.shape[1]
        assert np.all(np.abs(got[:, fine] - A @ B) <= ((n + 2) * 2.0 ** -24 + 3e-6) * (np.abs(A) @ np.abs(B)))


def _keys(it, fn):
    ctx = it.Context.global_()
    profiler.reset(ctx)
    profiler.enable(ctx)
    assert fn() == 0
    keys = list(profiler.stats(ctx))
    profiler.enable(ctx, False)
    return keys


@pytest.mark.parametrize("tile,ta,tb,m,n,k", [
    ("256x128", 0, 0, 4096, 256, 16384), ("256x128", 0, 1, 4096, 256, 16384), ("128x128", 0, 1, 2279, 2554, 22),
    ("128x128", 1, 0, 2356, 1812, 32), ("128x128", 0, 0, 2462, 2470, 17), ("128x128", 1, 1, 2021, 2978, 39),
    ("64x64", 0, 1, 4096, 768, 256), ("64x64", 1, 0, 307, 220, 1007), ("64x64", 0, 0, 2225, 47, 491),
    ("64x64", 1, 1, 1354, 515, 19), ("64x64", 0, 1, 129, 2868, 2781), ("64x64", 0, 0, 932, 44, 1592),
    ("64x32", 0, 0, 4096, 256, 1376), ("64x32", 0, 1, 4096, 256, 688), ("64x32", 0, 1, 4000, 250, 700),
    ("64x32", 1, 0, 4000, 250, 700), ("64x32", 0, 0, 1000, 90, 300), ("64x32", 1, 1, 609, 128, 1079),
    ("64x32", 1, 0, 288, 28, 2208)])
def test_every_tile_exact(it, tile, ta, tb, m, n, k):
    """Every tile, whole and at sizes it does not divide (descriptor, masked and bounds-checked loads), with
    alpha, beta and a bias: exact on small integers, whose sums are integers below 2^24."""
    a = synth.small_ints(51, (k, m) if ta else (m, k), -3, 3)
    b = synth.small_ints(52, (n, k) if tb else (k, n), -3, 3)
    bias, c0 = synth.small_ints(53, (n,), -4, 4), synth.small_ints(54, (m, n), -4, 4)
    T = it.Tensor.from_f32_slice
    A, B, out, Bias = T(a, list(a.shape)), T(b, list(b.shape)), T(c0, [m, n]), T(bias, [n])
    epi = _lib.Epilogue(flags=_lib.IT_EPI_BIAS | _lib.IT_EPI_F32_UNITS, bias=Bias.ptr)
    keys = _keys(it, lambda: A.ctx.lib.it_gemm(A.ctx.handle, 0, 0, ta, tb, m, n, k, 2.0, C.c_void_p(A.ptr), a.shape[1], 0,
                                               C.c_void_p(B.ptr), b.shape[1], 0, 3.0, C.c_void_p(out.ptr), n, 0, 1,
                                               C.byref(epi)))
    assert len(keys) == 1 and keys[0].startswith(f"gemm_f32_{'NT'[ta]}{'NT'[tb]}_{tile}|units:"), keys
    ref = op(a, ta).astype(np.float64) @ op(b, tb).astype(np.float64)
    assert np.array_equal(out.numpy(), (2 * ref + 3 * c0 + bias).astype(np.float32))


@pytest.mark.parametrize("bt,m,n,k,shared", [(3, 65, 40, 96, False), (5, 200, 130, 37, True), (2, 300, 300, 128, False)])
def test_batches_and_causal_outputs(it, bt, m, n, k, shared):
    """Strided and shared operands of a batch, plain and with the causal mask (-inf above the diagonal)."""
    a, b = synth.small_ints(61, (bt, m, k), -3, 3), synth.small_ints(62, (1 if shared else bt, n, k), -3, 3)
    A, B = it.Tensor.from_f32_slice(a, list(a.shape)), it.Tensor.from_f32_slice(b, list(b.shape))
    exact = np.matmul(a.astype(np.float64), np.swapaxes(b.astype(np.float64), 1, 2))
    above = np.triu(np.ones((m, n), bool), 1)
    for causal in (0, _lib.IT_EPI_CAUSAL):
        out = it.Tensor.empty([bt, m, n])
        epi = _lib.Epilogue(flags=_lib.IT_EPI_F32_UNITS | causal)
        keys = _keys(it, lambda: A.ctx.lib.it_gemm(A.ctx.handle, 0, 0, 0, 1, m, n, k, 1.0, C.c_void_p(A.ptr), k, m * k,
                                                   C.c_void_p(B.ptr), k, 0 if shared else n * k, 0.0, C.c_void_p(out.ptr), n,
                                                   m * n, bt, C.byref(epi)))
        assert "|units:" in keys[0], keys
        want = np.where(above, -np.inf, exact) if causal else exact
        assert np.array_equal(out.numpy(), want.astype(np.float32))


@pytest.mark.parametrize("dims,k", [([(1376, 256), (256, 688), (768, 256), (256, 256)], 4096),
                                    ([(100, 300), (301, 500), (65, 64)], 3001), ([(128, 128), (130, 132)], 100)])
def test_group_exact(it, dims, k):
    """Weight gradients as one grouped launch on the FP32 units, whole and ragged."""
    T = it.Tensor.from_f32_slice
    data = [(synth.small_ints(71 + i, (k, m), -2, 2), synth.small_ints(81 + i, (k, n), -2, 2)) for i, (m, n) in enumerate(dims)]
    ops = [(T(x, list(x.shape)), T(y, list(y.shape)), it.Tensor.empty([m, n])) for (x, y), (m, n) in zip(data, dims)]
    epi = _lib.Epilogue(flags=_lib.IT_EPI_F32_UNITS)
    calls = (_lib.GemmCall * len(dims))(*[
        _lib.GemmCall(1, 0, m, n, k, 1.0, x.ptr, m, 0, y.ptr, n, 0, 0.0, o.ptr, n, 0, 1, C.pointer(epi))
        for (x, y, o), (m, n) in zip(ops, dims)])
    ctx = ops[0][0].ctx
    keys = _keys(it, lambda: ctx.lib.it_gemm_group(ctx.handle, 0, 0, len(dims), calls))
    print(f"[units group] {keys}", flush=True)
    assert len(keys) == 1 and keys[0].startswith("gemm_f32_TN_64x64_group|units:"), keys
    for (x, y), (_, _, o) in zip(data, ops):
        assert np.array_equal(o.numpy(), (x.T.astype(np.float64) @ y.astype(np.float64)).astype(np.float32))
