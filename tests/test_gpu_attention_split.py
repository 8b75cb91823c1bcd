"""The attention kernel's two-part f16 products (csrc/attention.hip): tile and
key-block edges, both workgroup sizes with and without key splits, and every
value range, with the bound of test_gpu_attention (F32 products and sums)
against float64.

What the split adds to that bound is at most 2^-34 of the largest |v| of the
output's channel (FLOOR below, twice that: the weights' floor is of the same
size), however small the output is; a channel that is small as a whole, or a
query whose 64 outputs are, has none.
"""
import numpy as np
import pytest

from conftest import record_margin
from test_gpu_attention import _reference_and_bound, _run
from test_gpu_patch_block import normals

pytestmark = pytest.mark.gpu

vh = pytest.importorskip("vestra_hip")

FLOOR = 2.0 ** -33

# sequences and rows of one shape for each kernel form, and its (waves, key splits) on
# 256 compute units (test_plans.py holds the tables to the rules)
FORM_OF = {(250, 300): (4, 1), (40, 800): (8, 1), (12, 866): (4, 3), (2, 1000): (4, 8),
           (12, 1732): (8, 3)}
FORMS = list(FORM_OF)
# one block and one past it, 128- and 256-query tiles and one past each
SIZE_FORM = {(2, 63): (4, 1), (3, 66): (4, 1), (2, 127): (4, 1), (2, 128): (4, 1),
             (12, 190): (4, 1), (2, 513): (4, 5), (130, 129): (8, 1), (250, 257): (4, 1),
             (250, 320): (4, 1), (40, 800): (8, 1), (12, 1740): (8, 3)}


def _assert_close(got, q, k, v, label, channel_floor=FLOOR):
    ref, bound = _reference_and_bound(q, k, v)
    tol = bound + 2.0 ** -23 * np.abs(ref) + channel_floor * np.abs(v).max(axis=0) + 2.0 ** -149
    record_margin("attention split", got, ref, tol=tol, label=label)
    off = np.abs(got.astype(np.float64) - ref)
    assert np.all(off <= tol), f"{label}: {np.sum(~(off <= tol))} off, worst {np.max(off / tol)}"


def _check(rt, q, k, v, label, seqs=None, channel_floor=FLOOR):
    s, n, _ = q.shape
    got = _run(rt, q, k, v, s, n)
    for i in (range(s) if seqs is None else seqs):
        _assert_close(got[i], q[i], k[i], v[i], f"{label} seq {i}", channel_floor)


def _some(s):
    return range(0, s, max(1, s // 3))


@pytest.mark.parametrize("s,n", list(SIZE_FORM))
def test_sizes(rt, rng, s, n):
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    _check(rt, q, k, v, f"n={n}", _some(s))


@pytest.mark.parametrize("s,n", FORMS)
@pytest.mark.parametrize("qs,ks,vs", [(1, 1, 1e-5), (1, 1, 1e4), (1e-4, 1e4, 1), (1e4, 1e-4, 1),
                                      (1e-20, 1, 1e-30), (1, 300, 1), (1, 1e-6, 1e-3)])
def test_value_ranges(rt, rng, s, n, qs, ks, vs):
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    _check(rt, (q * qs).astype(np.float32), (k * ks).astype(np.float32),
           (v * vs).astype(np.float32), f"{qs} {ks} {vs}", _some(s))


@pytest.mark.parametrize("s,n", FORMS)
@pytest.mark.parametrize("least,most", [(-30, 30), (-12, 1)])
def test_channels_of_different_sizes(rt, rng, s, n, least, most):
    """Every channel of V to its own size, and some of zeros throughout or in the
    first key blocks."""
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    v *= (10.0 ** np.linspace(least, most, 64)).astype(np.float32)
    v[0, :, 5], v[0, :, 40] = 0, 0
    v[1, :n // 2, 7], v[1, :70, 30] = 0, 0
    v[1, 70, 31] *= 1e-12
    _check(rt, q, k, v, "channels", {0, 1, s - 1})


@pytest.mark.parametrize("s,n", FORMS)
@pytest.mark.parametrize("small", [1e-4, 1e-7, 1e-12, 0.0])
def test_queries_that_attend_to_small_rows(rt, rng, s, n, small):
    """Two keys that some queries attend to alone, with rows of V `small` times the
    others: relative to the row they return."""
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    keys, own = [n // 2, n - 1], slice(3, n, 5)
    k[:, :, 0] = 0
    k[:, keys, 0], q[:, own, 0] = 100.0, 20.0
    v[:, keys] *= np.float32(small)
    got = _run(rt, q, k, v, s, n)
    for i in _some(s):
        ref, bound = _reference_and_bound(q[i], k[i], v[i])
        off = np.abs(got[i].astype(np.float64) - ref)
        tol = bound + 2.0 ** -22 * np.abs(ref).max(axis=1, keepdims=True) + 2.0 ** -149
        assert np.all(off[own] <= tol[own]), np.max((off / tol)[own])
        _assert_close(got[i], q[i], k[i], v[i], f"seq {i}")


@pytest.mark.parametrize("s,n", FORMS + [(4, 10392)])
def test_even_attention_beside_a_few_large_rows(rt, rng, s, n):
    """Weights all alike and three first keys with V a hundred times the others':
    outputs far below V's largest values."""
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    v[:, :3] *= 100
    v -= v.mean(axis=1, keepdims=True)
    _check(rt, q * np.float32(0.01), k, v, "even", [0, s - 1])


def test_growing_maximum_and_flat_tails(rt, rng):
    """Scores that rise block after block (the running maximum moves each
    time), in steps below the slack, and thousands of weights far below one."""
    n = 2048
    q, k, v = (normals(rng, 2, n, 64) * np.float32(0.1) for _ in range(3))
    q[..., 0] = 8.0
    k[0, :, 0] = np.arange(n) // 64 * 0.9   # 0.9 a block: within the slack
    k[1, :, 0] = np.arange(n) // 64 * 8.0   # 8 a block: beyond it
    _check(rt, q, k, v, "rising")
    k[0, :, 0], k[1, :, 0] = 0.0, -12.0
    k[:, 5, 0] = 6.0                         # one key far above all others
    _check(rt, q, k, v, "flat tail")


@pytest.mark.parametrize("s,n", FORMS)
def test_infinities_and_nan_stay_in_their_sequence(rt, rng, s, n):
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    good = _run(rt, q, k, v, s, n)
    q2, k2, v2 = q.copy(), k.copy(), v.copy()
    v2[0, 7, 3] = np.nan
    k2[1, n - 70, 5] = np.inf
    got = _run(rt, q2, k2, v2, s, n)
    assert np.isnan(got[0, :, 3]).all() and np.isnan(got[1]).any()
    others = [d for d in range(64) if d != 3]
    ref, bound = _reference_and_bound(q[0], k[0], v[0])
    off = np.abs(got[0][:, others] - ref[:, others])
    assert np.all(off <= (bound + 2.0 ** -23 * np.abs(ref) + FLOOR * np.abs(v[0]).max(axis=0))[:, others])
    assert np.array_equal(got[2:], good[2:])


@pytest.mark.parametrize("s,n", FORMS)
def test_a_query_depends_on_its_own_row(rt, rng, s, n):
    """Queries that are computed again change no other query's bits."""
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    good = _run(rt, q, k, v, s, n)
    odd = [1, 40, 190, n - 1]
    q2 = q.copy()
    q2[:, 1], q2[:, 40], q2[:, 190], q2[:, n - 1] = 1000, np.nan, -400, np.inf
    got = _run(rt, q2, k, v, s, n)
    rest = [i for i in range(n) if i not in odd]
    assert np.array_equal(got[:, rest], good[:, rest])
    for i in _some(s):
        ref, bound = _reference_and_bound(q2[i, [1, 190]], k[i], v[i])
        off = np.abs(got[i, [1, 190]] - ref)
        assert np.all(off <= bound + 2.0 ** -23 * np.abs(ref) + FLOOR * np.abs(v[i]).max(axis=0))


@pytest.mark.parametrize("s,n", FORMS)
def test_a_neighbours_growing_maximum_changes_no_bits(rt, rng, s, n):
    """A query's running maximum moves by its own scores alone."""
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    k[:, n // 2:, 0] *= 3
    good = _run(rt, q, k, v, s, n)
    q2 = q.copy()
    q2[:, 41], q2[:, 190] = 0, 60
    got = _run(rt, q2, k, v, s, n)
    rest = [i for i in range(n) if i not in (41, 190)]
    assert np.array_equal(got[:, rest], good[:, rest])
