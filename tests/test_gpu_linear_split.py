"""The wide linear's two-part f16 products (csrc/split_f16.h): every value range
and the edges of its tiles and K stages.

The bound is the one of an f32 dot product: with u = 2^-24 and s = sum_k |x_k
w_k|, |got - exact| <= 2 sqrt(K) u s + u |exact|.  The split holds a factor to
2^-23 = 2u (rms u/2) and leaves out a product of at most 2^-22 = 4u (rms u/2)
of the term; over K terms of random sign that is below sqrt(K) u s.  Whatever it
holds less well (values beyond f16, tiny ones beside large ones, sums of few
terms) is an F32 sum, so there is no floor: the bound is one of the sum's own
terms, whatever else the row, the column and the tile hold.
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


def _check(got, x, w, b, label, terms=None):
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    ref = x64 @ w64 + b
    tol = ((terms or 2 * np.sqrt(x.shape[1])) * U * (np.abs(x64) @ np.abs(w64)) + U * np.abs(ref)
           + U * np.abs(b) + 2.0 ** -149)
    bad = np.abs(got - ref) > tol
    assert not bad.any(), f"{label}: {int(bad.sum())} off, worst {np.max(np.abs(got - ref) / tol)}"


# tails of rows, columns and K on every tile; K below one stage; odd counts of 32 k
# on tiles of two a barrier
SHAPE_FORM = {(1, 4, 4): (64, 64, 1), (63, 28, 60): (64, 64, 1), (65, 96, 68): (64, 64, 1),
              (64, 100, 64): (64, 64, 1), (130, 3072, 132): (64, 64, 8),
              (1500, 160, 2304): (64, 128, 1), (4000, 1024, 1028): (64, 128, 1),
              (10392, 64, 768): (128, 128, 1), (4097, 132, 1540): (128, 128, 1),
              (10392, 768, 768): (128, 256, 1), (10300, 804, 764): (128, 256, 1),
              (2600, 3072, 772): (128, 256, 3)}


@pytest.mark.parametrize("m,k,n", list(SHAPE_FORM))
def test_shapes(rt, rng, m, k, n):
    x, w, b = normals(rng, m, k), normals(rng, k, n, scale=0.02), normals(rng, n, scale=0.02)
    _check(_linear(rt, x, w, b), x, w, b, f"{m}x{k}->{n}")


@pytest.mark.parametrize("m,k,n", [(130, 768, 192), (1500, 768, 2304), (10392, 128, 768),
                                   (10392, 768, 768), (70, 20, 64), (300, 48, 128)])
@pytest.mark.parametrize("xs,ws", [(1e-6, 1.0), (1e-3, 1e-20), (1e5, 1e-3), (1e25, 1e-30),
                                   (1e-30, 1e10), (3e4, 1.0), (1e-38, 1.0)])
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


@pytest.mark.parametrize("m,k,n", [(70, 96, 128), (130, 3072, 132), (5000, 64, 768),
                                   (2600, 3072, 772)])
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
                                   (5000, 64, 768), (4000, 1024, 1028), (10392, 768, 768)])
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
    _check(out.numpy().reshape(m, n), x, w.astype(np.float32), b, "f16 weights")


# rows, k, columns of one shape for each tile, and its (rows, columns, splits) on 256
# compute units (test_plans.py holds the table to the rules)
FORM_OF = {(130, 768, 192): (64, 64, 6), (1500, 768, 2304): (64, 128, 1),
           (10392, 128, 768): (128, 128, 1), (10392, 768, 768): (128, 256, 1),
           (2600, 3072, 768): (128, 256, 4)}
FORMS = list(FORM_OF)


@pytest.mark.parametrize("m,k,n", FORMS)
@pytest.mark.parametrize("small", [1e-4, 1e-6, 1e-8, 1e-11, 1e-20])
def test_mixed_sizes_within_a_row_and_a_column(rt, rng, m, k, n, small):
    """Channels `small` times the others, read by columns that read no other
    (and by ordinary ones); weights `small` times the others, met by rows that
    meet no other.  One large channel or weight, or an eighth of them.  Where one
    term stands far above the others its sum is cut to the same bits at each of
    K / 4 steps of an F32 product: (K / 4 + 4) u s."""
    b, cut = np.zeros(n, np.float32), k / 4 + 4
    for large in (1, k // 8):
        x, w = normals(rng, m, k), normals(rng, k, n, scale=0.02)
        x[::2, large:] *= np.float32(small)
        w[:large, ::2] = 0
        got = _linear(rt, x, w, b)
        _check(got, x, w, b, f"row, {large} large", cut)
        _check(got[::2, ::2], x[::2], w[:, ::2], b[::2], f"row, read alone, {large} large")
        x, w = normals(rng, m, k), normals(rng, k, n, scale=0.02)
        w[large:, ::2] *= np.float32(small)
        x[::2, :large] = 0
        got = _linear(rt, x, w, b)
        _check(got, x, w, b, f"column, {large} large", cut)
        _check(got[::2, ::2], x[::2], w[:, ::2], b[::2], f"column, met alone, {large} large")


@pytest.mark.parametrize("m,k", [(130, 192), (1500, 768), (10392, 128), (4100, 1024), (70, 16),
                                 (300, 48)])
def test_selecting_weights_copy(rt, rng, m, k):
    """A column with a single weight of 1 returns its channel's bits; a row with
    a single 1 the weights of that channel."""
    x, w = ((normals(rng, r, k) * 10.0 ** rng.integers(-9, 9, (r, k))).astype(np.float32)
            for r in (m, k))
    zero = np.zeros(k, np.float32)
    assert np.array_equal(_linear(rt, x, np.eye(k, dtype=np.float32), zero), x)
    rows = np.zeros((m, k), np.float32)
    pick = rng.integers(0, k, m)
    rows[np.arange(m), pick] = 1
    assert np.array_equal(_linear(rt, rows, w, zero), w[pick])


@pytest.mark.parametrize("m,k,n", FORMS)
def test_an_output_depends_on_its_row_and_column_alone(rt, rng, m, k, n):
    """Rows and columns that the split does not hold change no other output."""
    x, w, b = normals(rng, m, k), normals(rng, k, n, scale=0.02), normals(rng, n)
    good = _linear(rt, x, w, b)
    x2, w2 = x.copy(), w.copy()
    x2[3], x2[m // 2, 1:], x2[m - 2] = 0, 0, np.nan
    x2[5, k - 1], x2[6, 0], x2[7, 1:] = np.inf, 3e38, x[7, 1:] * np.float32(1e-9)
    w2[1, 4], w2[:, 9], w2[1:, n - 2], w2[0, n // 2] = np.inf, 0, 0, 1e30
    got = _linear(rt, x2, w2, b)
    rows = [r for r in range(m) if r not in (3, 5, 6, 7, m // 2, m - 2)]
    cols = [c for c in range(n) if c not in (4, 9, n // 2, n - 2)]
    assert np.array_equal(got[np.ix_(rows, cols)], good[np.ix_(rows, cols)])


# one image's 64 x 64 tiles, twelve views' 128 x 256 and a 64 x 128 form
@pytest.mark.parametrize("views,gh,gw", [(1, 24, 36), (12, 24, 36), (2, 24, 36)])
def test_fused_forms_of_outputs_taken_again(rt, rng, views, gh, gw):
    """Inputs with rows and weights that the split does not hold, through the
    head-major forms, the Q/K epilogue, the residual and its LayerNorm: the bits
    of the plain linear followed by the separate operations."""
    heads, d = 12, 768
    m = views * (1 + gh * gw)
    b = normals(rng, 3 * d)
    x, w = normals(rng, m, d), normals(rng, d, 3 * d, scale=0.02)
    x[5, 1:] *= np.float32(1e-12)
    x[70, 3], x[m - 1] = 1e30, x[m - 1] * np.float32(1e-38)
    w[:, 7], w[1:, 800], w[3, 1700] = 0, 0, 1e30
    lin, xt = rt.prepare_linear_f32(d, 3 * d, w, b), rt.upload_f32(x)
    plain = rt.alloc_f32(m * 3 * d)
    lin.run_into(xt, m, plain)
    q, k, v = rt.split_qkv_hnd_f32(plain, m, heads, 64)
    got = [rt.alloc_f32(m * d) for _ in range(3)]
    par = [rt.upload_f32(a) for a in (normals(rng, 64, shift=1), normals(rng, 64),
                                      normals(rng, 64, shift=1), normals(rng, 64))]
    lin.run_qkv_hnd_norm_rope(xt, m, heads, *got, *par, 1, gh, gw, views, False, 100.0, 1e-5)
    rt.qk_norm_rope_grid_f32(q, k, *par, heads, 64, 1, gh, gw, views, False,
                             vh.VK_QK_HEADS_OUTER, 100.0, 1e-5)
    for name, a, e in zip("qkv", got, (q, k, v)):
        assert np.array_equal(a.numpy(), e.numpy(), equal_nan=True), name

    hnd = rt.upload_f32(np.ascontiguousarray(x.reshape(m, heads, 64).transpose(1, 0, 2)))
    proj = rt.prepare_linear_f32(d, d, np.ascontiguousarray(w[:, :d]), b[:d], normals(rng, d))
    res = normals(rng, m, d)
    want, fused = rt.alloc_f32(m * d), rt.upload_f32(res)
    proj.run_into(xt, m, want)
    proj.run_hnd_residual(hnd, m, heads, fused)
    with np.errstate(over="ignore", invalid="ignore"):
        assert np.array_equal(fused.numpy().reshape(m, d), res + want.numpy().reshape(m, d),
                              equal_nan=True)
