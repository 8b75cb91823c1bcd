"""The wide linear's two-part f16 products (csrc/split_f16.h): every value range
and the edges of its tiles and K stages.

The bound is the one of an f32 dot product: with u = 2^-24 and s = sum_k |x_k
w_k|, |got - exact| <= 2 sqrt(K) u s + u |exact|.  (The split adds at most
2^-23 per factor and 2^-22 per left-out product, rms 2^-25 each, which stay
below u s; rows whose values are all tiny, or that hold a value f16 cannot,
run on F32 matrix instructions.)
"""
import numpy as np
import pytest

from test_gpu_patch_block import normals

pytestmark = pytest.mark.gpu

vh = pytest.importorskip("vestra_hip")

U = 2.0 ** -24


def _linear(rt, x, w, b):
    m, (k, n) = x.shape[0], w.shape
    out = rt.alloc_f32(m * n)
    rt.prepare_linear_f32(k, n, w, b).run_into(rt.upload_f32(x), m, out)
    return out.numpy().reshape(m, n)


def _check(got, x, w, b, label, floor=0.0):
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    ref = x64 @ w64 + b
    tol = (2 * np.sqrt(x.shape[1]) * U * (np.abs(x64) @ np.abs(w64)) + U * np.abs(ref)
           + U * np.abs(b) + 2.0 ** -149 + floor * np.abs(w64).sum(axis=0))
    bad = np.abs(got - ref) > tol
    assert not bad.any(), f"{label}: {int(bad.sum())} off, worst {np.max(np.abs(got - ref) / tol)}"


# tiles 128 x 256 (10392 x 64 -> 768, 4000 x 1024 -> 1028), 64 x 64 (2 stages a barrier: odd counts, tails), 64 x 128, 128 x 128,
# rows and columns one past a tile, split runs, K below one stage
@pytest.mark.parametrize("m,k,n", [(1, 4, 4), (63, 28, 60), (65, 96, 68), (64, 100, 64),
                                   (130, 3072, 132), (1500, 160, 2304), (10392, 64, 768),
                                   (4097, 132, 1540), (4000, 1024, 1028)])
def test_shapes(rt, rng, m, k, n):
    x, w, b = normals(rng, m, k), normals(rng, k, n, scale=0.02), normals(rng, n, scale=0.02)
    _check(_linear(rt, x, w, b), x, w, b, f"{m}x{k}->{n}")


@pytest.mark.parametrize("m,k,n", [(130, 768, 192), (1500, 768, 2304), (10392, 128, 768)])
@pytest.mark.parametrize("xs,ws", [(1e-6, 1.0), (1e-3, 1e-20), (1e5, 1e-3), (1e25, 1e-30),
                                   (1e-30, 1e10), (3e4, 1.0)])
def test_value_ranges(rt, rng, m, k, n, xs, ws):
    """Whole inputs and weights of unusual sizes, and one such row and column
    among ordinary ones."""
    x, w = normals(rng, m, k), normals(rng, k, n)
    b = np.zeros(n, np.float32)
    xa, wa = (x * xs).astype(np.float32), (w * ws).astype(np.float32)
    _check(_linear(rt, xa, wa, b), xa, wa, b, "all rows")
    xa, wa = x.copy(), w.copy()
    xa[m // 2] *= np.float32(xs)
    wa[:, n // 2] *= np.float32(ws)
    _check(_linear(rt, xa, wa, b), xa, wa, b, "one row")


def test_zero_rows_and_columns(rt, rng):
    x, w, b = normals(rng, 130, 96), normals(rng, 96, 192), normals(rng, 192)
    x[5], w[:, 7] = 0, 0
    got = _linear(rt, x, w, b)
    assert np.array_equal(got[5], b) and np.all(got[:, 7] == b[7])
    _check(got, x, w, b, "zeros")


@pytest.mark.parametrize("m,k,n", [(70, 96, 128), (130, 3072, 132), (5000, 64, 768)])
def test_infinities_and_nan_stay_in_their_rows_and_columns(rt, rng, m, k, n):
    x, w, b = normals(rng, m, k), normals(rng, k, n, scale=0.02), np.zeros(n, np.float32)
    x[3, 5], x[4, k - 1], x[m - 1, 0] = np.inf, np.nan, -np.inf
    x[10, 1] = 3.0e38
    w[2, 9], w[k - 1, n - 1] = np.inf, np.nan
    got = _linear(rt, x, w, b)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = (x.astype(np.float64) @ w.astype(np.float64)).astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref) & ~np.isnan(ref)
    assert np.array_equal(got[inf], ref[inf])
    rows = [r for r in range(m) if r not in (3, 4, m - 1)]
    cols = [c for c in range(n) if c not in (9, n - 1)]
    _check(got[np.ix_(rows, cols)], x[rows], w[:, cols], b[cols], "finite part")


@pytest.mark.parametrize("m,k,n", [(70, 96, 128), (130, 3072, 132), (1500, 768, 2304),
                                   (5000, 64, 768), (4000, 1024, 1028)])
@pytest.mark.parametrize("wide_range", [False, True])
def test_f16_stored_weights_are_the_f32_preparation(rt, rng, m, k, n, wide_range):
    """Weights stored as f16 take one part and two products, unless a column's
    range needs the second part (f16's largest value beside subnormals): the
    bits of the f32 preparation of the same values either way."""
    x, b = normals(rng, m, k), normals(rng, n, scale=0.02)
    w = normals(rng, k, n, scale=0.02).astype(np.float16)
    if wide_range:
        w[0, :] = 60000.0
        w[1:3, :] = np.float16(2.0 ** -24) * 3
        x[:, 0] *= np.float32(1e-6)
    out = rt.alloc_f32(m * n)
    rt.prepare_linear_w16(k, n, w, b).run_into(rt.upload_f32(x), m, out)
    assert np.array_equal(out.numpy().reshape(m, n), _linear(rt, x, w.astype(np.float32), b))
    # the split of x has a floor of 2^-36 of 1, which weights of 60000 against
    # values of 1e-6 (where they give 0.06) make visible: 2^-36 sum_k |w_k|
    _check(out.numpy().reshape(m, n), x, w.astype(np.float32), b, "f16 weights",
           floor=2.0 ** -36 if wide_range else 0.0)
