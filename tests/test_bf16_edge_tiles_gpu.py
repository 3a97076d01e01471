"""BF16 products that no whole-tile kernel takes, on the direct-to-LDS tiles (padded copies of operands
that cannot be read in place, bounds-checked edge tiles): exact on small integers, whose sums are
integers below 2^24, against a float64 product."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from irontensor_amd import _lib, profiler, synth
from tests.numerics import op

pytestmark = pytest.mark.gpu


def _bf16(it, x):
    return it.Tensor.from_f32_as_bf16(x, list(x.shape))


def _keys(it, fn):
    ctx = it.Context.global_()
    profiler.reset(ctx)
    profiler.enable(ctx)
    fn()
    keys = list(profiler.stats(ctx))
    profiler.enable(ctx, False)
    return keys


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(1999, 3001, 1237), (511, 513, 640), (1000, 2048, 1111), (257, 1025, 128),
                                   (2100, 2000, 3000), (130, 8190, 2049)])
def test_exact_in_every_layout(it, m, n, k, ta, tb):
    a = synth.small_ints(m + k, (k, m) if ta else (m, k), -3, 3)
    b = synth.small_ints(n + k, (n, k) if tb else (k, n), -3, 3)
    out = it.Tensor.empty([m, n], it.Precision.FP32)
    keys = _keys(it, lambda: it.gemm(_bf16(it, a), _bf16(it, b), trans_a=bool(ta), trans_b=bool(tb), out=out))
    print(f"[bf16 edge] {m}x{n}x{k} {keys}", flush=True)
    assert len(keys) == 1 and ("_dtl_edge|" in keys[0] or m * n < 300000), keys
    ref = op(a, ta).astype(np.float64) @ op(b, tb).astype(np.float64)
    assert np.array_equal(out.numpy(), ref.astype(np.float32))


def test_batched_bias_alpha_beta_and_bf16_output(it):
    """A ragged batch that is priced onto the plain tiles (test_batched_epilogues_on_edge_tiles has the others)."""
    bt, m, n, k = 3, 301, 517, 200
    a, b = synth.small_ints(1, (bt, m, k), -3, 3), synth.small_ints(2, (n, k), -3, 3)
    bias, c0 = synth.small_ints(3, (n,), -4, 4), synth.small_ints(4, (bt, m, n), -4, 4)
    out = it.Tensor.from_f32_slice(c0, list(c0.shape))
    it.gemm(_bf16(it, a), _bf16(it, b), trans_b=True, alpha=2.0, beta=3.0, out=out,
            bias=it.Tensor.from_f32_slice(bias, [n]))
    prod = a.astype(np.float64) @ b.astype(np.float64).T
    assert np.array_equal(out.numpy(), (2 * prod + 3 * c0 + bias).astype(np.float32))
    got = it.gemm(_bf16(it, a), _bf16(it, b), trans_b=True, out_precision=it.Precision.BF16)
    assert np.array_equal(got.as_bf16_slice().reshape(bt, m, n), it.f32_to_bf16(prod.astype(np.float32)))


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
def test_strided_operands_inside_nan(it, ta, tb):
    """Operands and output inside wider buffers at odd columns: the surrounding NaN never reach a
    result and nothing outside the output is written."""
    m, n, k = 700, 900, 450
    a = synth.small_ints(7, (k, m) if ta else (m, k), -3, 3)
    b = synth.small_ints(8, (n, k) if tb else (k, n), -3, 3)
    ctx = it.Context.global_()

    def wide(x):
        w = np.full((x.shape[0] + 2, x.shape[1] + 7), np.nan, np.float32)
        w[1:-1, 3:-4] = x
        return _bf16(it, w), w.shape[1]

    (A, lda), (B, ldb) = wide(a), wide(b)
    ldc = n + 7
    Cw = it.Tensor.from_f32_slice(np.full((m + 2, ldc), 7.0, np.float32), [m + 2, ldc])
    st = ctx.lib.it_gemm(ctx.handle, 2, 0, ta, tb, m, n, k, 1.0, C.c_void_p(A.ptr + 2 * (lda + 3)), lda, 0,
                         C.c_void_p(B.ptr + 2 * (ldb + 3)), ldb, 0, 0.0, C.c_void_p(Cw.ptr + 4 * (ldc + 3)), ldc, 0,
                         1, None)
    assert st == 0
    got = Cw.numpy()
    ref = op(a, ta).astype(np.float64) @ op(b, tb).astype(np.float64)
    assert np.array_equal(got[1:-1, 3:-4], ref.astype(np.float32))
    got[1:-1, 3:-4] = 7.0
    assert np.all(got == 7.0)


def test_capture_without_scratch_takes_the_plain_tiles(it):
    """A capture may not allocate: on a fresh context the product captures on the plain tiles, and its
    replays give the same results."""
    m, n, k = 600, 700, 333
    ctx = it.Context(0)
    a, b = synth.small_ints(11, (m, k), -3, 3), synth.small_ints(12, (n, k), -3, 3)
    A = it.Tensor.from_bf16_slice(it.f32_to_bf16(a), [m, k], ctx)
    B = it.Tensor.from_bf16_slice(it.f32_to_bf16(b), [n, k], ctx)
    out = it.Tensor.zeros([m, n], it.Precision.FP32, ctx)
    g = C.c_void_p()
    assert ctx.lib.it_capture_begin(ctx.handle) == 0
    it.gemm(A, B, trans_b=True, out=out)
    assert ctx.lib.it_capture_end(ctx.handle, C.byref(g)) == 0
    ref = (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.float32)
    for _ in range(3):
        assert ctx.lib.it_zero(ctx.handle, C.c_void_p(out.ptr), out.byte_size()) == 0
        assert ctx.lib.it_graph_launch(ctx.handle, g) == 0
        assert np.array_equal(out.numpy(), ref)
    assert ctx.lib.it_graph_destroy(g) == 0


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("shared", [False, True])
def test_batched_epilogues_on_edge_tiles(it, ta, tb, shared):
    """A batch on padded copies and edge tiles, B its own or shared by the items: alpha, beta and a bias
    into FP32 and BF16 outputs of odd rows (8-byte stores at 2-byte alignment)."""
    bt, m, n, k = 3, 700, 901, 333
    a = synth.small_ints(21, (bt, k, m) if ta else (bt, m, k), -2, 2)
    b = synth.small_ints(22, ((1,) if shared else (bt,)) + ((n, k) if tb else (k, n)), -2, 2)
    bias, c0 = synth.small_ints(23, (n,), -4, 4), synth.small_ints(24, (bt, m, n), -4, 4)
    A, B, Bias = _bf16(it, a), _bf16(it, b), it.Tensor.from_f32_slice(bias, [n])
    ctx = it.Context.global_()
    exact = 2 * (np.matmul(op(a, ta).astype(np.float64), op(b, tb).astype(np.float64))) + bias
    for bf16 in (False, True):
        beta = 0.0 if bf16 else 3.0
        out = _bf16(it, c0) if bf16 else it.Tensor.from_f32_slice(c0, list(c0.shape))
        epi = _lib.Epilogue(flags=_lib.IT_EPI_BIAS, bias=Bias.ptr)
        keys = _keys(it, lambda: ctx.lib.it_gemm(
            ctx.handle, 2, 2 if bf16 else 0, ta, tb, m, n, k, 2.0, C.c_void_p(A.ptr), m if ta else k, m * k,
            C.c_void_p(B.ptr), k if tb else n, 0 if shared else n * k, beta, C.c_void_p(out.ptr), n, m * n, bt, C.byref(epi)))
        assert len(keys) == 1 and "_dtl_edge|" in keys[0], keys
        want = (exact + beta * c0).astype(np.float32)
        got = out.as_bf16_slice().reshape(want.shape) if bf16 else out.numpy()
        assert np.array_equal(got, it.f32_to_bf16(want) if bf16 else want)


@pytest.mark.parametrize("ta,tb,m,n,k", [(0, 0, 246, 656, 9110), (1, 1, 529, 210, 6306), (0, 1, 995, 2294, 4345),
                                         (1, 0, 991, 1358, 10784)])
def test_split_k_on_edge_tiles(it, ta, tb, m, n, k):
    """Few tiles and a long ragged k: the edge tiles' partial sums and their reduction."""
    a = synth.small_ints(31, (k, m) if ta else (m, k), -2, 2)
    b = synth.small_ints(32, (n, k) if tb else (k, n), -2, 2)
    out = it.Tensor.empty([m, n], it.Precision.FP32)
    keys = _keys(it, lambda: it.gemm(_bf16(it, a), _bf16(it, b), trans_a=bool(ta), trans_b=bool(tb), out=out))
    print(f"[bf16 edge split] {keys}", flush=True)
    assert "_dtl_edge|" in keys[0] and not keys[0].endswith(" s1"), keys
    assert np.array_equal(out.numpy(), (op(a, ta).astype(np.float64) @ op(b, tb).astype(np.float64)).astype(np.float32))
