"""FP32 decode products (X.W^T, at most 16 rows) on gemv_nt: the edges of its 16-column blocks, of a
wave's k range and of the row counts, against float64."""
import numpy as np
import pytest

from irontensor_amd import profiler, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def it():
    import irontensor_amd
    return irontensor_amd


def _keys(it, call):
    ctx = it.Context.global_()
    profiler.reset(ctx)
    profiler.enable(ctx)
    out = call()
    keys = list(profiler.stats(ctx))
    profiler.enable(ctx, False)
    return out, keys


@pytest.mark.parametrize("bt,m,k,n", [(1, 1, 4, 1), (1, 1, 256, 768), (1, 8, 100, 33), (1, 9, 516, 2050), (1, 16, 60, 17),
                                      (1, 16, 1028, 64), (3, 5, 264, 40), (2, 13, 68, 15)])
def test_f32_decode(it, bt, m, k, n):
    print(f"[f32 decode] {bt}x{m}x{k}x{n}", flush=True)
    a, b = synth.small_ints(1, (bt, m, k), -3, 3), synth.small_ints(2, (bt, n, k), -3, 3)
    sa, sb, sc = (list(s) if bt > 1 else list(s[1:]) for s in ((bt, m, k), (bt, n, k), (bt, m, n)))
    A, B = it.Tensor.from_f32_slice(a, sa), it.Tensor.from_f32_slice(b, sb)
    c, keys = _keys(it, lambda: it.gemm(A, B, trans_b=True))
    assert any(key.startswith("gemv_f32_NT") for key in keys), keys
    exact = np.matmul(a.astype(np.float64), np.swapaxes(b, 1, 2).astype(np.float64))
    assert np.array_equal(c.numpy().reshape(exact.shape), exact)  # small integers: sums are exact
    if bt == 1:
        bias, c0 = synth.small_ints(3, (n,), -4, 4), synth.small_ints(4, (m, n), -4, 4)
        out = it.Tensor.from_f32_slice(c0, [m, n])
        it.gemm(A, B, trans_b=True, alpha=2.0, beta=1.0, out=out, bias=it.Tensor.from_f32_slice(bias, [n]))
        assert np.array_equal(out.numpy(), (2.0 * exact[0] + c0 + bias).astype(np.float32))
    # normal values: at most k rounded sums of |a||b| each
    x, w = synth.normal(5, (m, k)), synth.normal(6, (n, k), std=0.02)
    got = it.gemm(it.Tensor.from_f32_slice(x, [m, k]), it.Tensor.from_f32_slice(w, [n, k]), trans_b=True).numpy()
    ref, mag = x.astype(np.float64) @ w.astype(np.float64).T, np.abs(x).astype(np.float64) @ np.abs(w).T
    assert np.all(np.abs(got - ref) <= (k + 2) * 2.0 ** -24 * mag)


def test_f32_decode_infinity_and_nan(it):
    """An infinite weight gives its column an infinity, a NaN row of X stays that row's; nothing spreads through
    the rows that fill the operand up."""
    x, w = synth.normal(7, (3, 36)), synth.normal(8, (20, 36))
    x[1, 5], w[19, 0] = np.nan, np.inf
    got = it.gemm(it.Tensor.from_f32_slice(x, [3, 36]), it.Tensor.from_f32_slice(w, [20, 36]), trans_b=True).numpy()
    assert np.isnan(got[1]).all()
    assert np.isfinite(got[[0, 2], :19]).all() and np.isinf(got[[0, 2], 19]).all()


def test_f32_decode_odd_k_keeps_the_tiles(it):
    A, B = (it.Tensor.from_f32_slice(synth.normal(9 + i, s), list(s)) for i, s in enumerate(((4, 37), (24, 37))))
    c, keys = _keys(it, lambda: it.gemm(A, B, trans_b=True))
    assert not any(key.startswith("gemv") for key in keys), keys
    assert np.isfinite(c.numpy()).all()
