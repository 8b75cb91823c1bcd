"""The attention kernel's two-part f16 products (csrc/attention.hip): tile and
key-block edges, both workgroup sizes, and every value range, with the bound of
test_gpu_attention (F32 products and sums) against float64.
"""
import numpy as np
import pytest

from test_gpu_attention import _assert_attention, _reference_and_bound, _run
from test_gpu_patch_block import normals

pytestmark = pytest.mark.gpu

vh = pytest.importorskip("vestra_hip")


def _check(rt, q, k, v, label, seqs=None):
    s, n, _ = q.shape
    got = _run(rt, q, k, v, s, n)
    for i in (range(s) if seqs is None else seqs):
        ref, bound = _reference_and_bound(q[i], k[i], v[i])
        _assert_attention(got[i], ref.astype(np.float32), bound, f"{label} seq {i}")


# one block and one past it, 128- and 256-query tiles and one past each, key
# splits (12 x 190, 2 x 513), unsplit four waves (130 x 129) and eight (250 x 257)
@pytest.mark.parametrize("s,n", [(2, 63), (3, 66), (2, 127), (2, 128), (12, 190), (2, 513),
                                 (130, 129), (250, 257), (250, 320)])
def test_sizes(rt, rng, s, n):
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    _check(rt, q, k, v, f"n={n}", range(0, s, max(1, s // 5)))


@pytest.mark.parametrize("s,n", [(2, 150), (250, 300)])
@pytest.mark.parametrize("qs,ks,vs", [(1, 1, 1e-5), (1, 1, 1e4), (1e-4, 1e4, 1), (1e4, 1e-4, 1),
                                      (1e-20, 1, 1e-30), (1, 300, 1), (1, 1e-6, 1e-3)])
def test_value_ranges(rt, rng, s, n, qs, ks, vs):
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    _check(rt, (q * qs).astype(np.float32), (k * ks).astype(np.float32),
           (v * vs).astype(np.float32), f"{qs} {ks} {vs}", range(0, s, max(1, s // 4)))


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


@pytest.mark.parametrize("s,n", [(2, 150), (250, 300)])
def test_infinities_and_nan_stay_in_their_sequence(rt, rng, s, n):
    q, k, v = (normals(rng, s, n, 64) for _ in range(3))
    good = _run(rt, q, k, v, s, n)
    q2, k2, v2 = q.copy(), k.copy(), v.copy()
    v2[0, 7, 3] = np.nan
    k2[1, 70, 5] = np.inf
    got = _run(rt, q2, k2, v2, s, n)
    assert np.isnan(got[0, :, 3]).all() and np.isnan(got[1]).any()
    others = [d for d in range(64) if d != 3]
    ref, bound = _reference_and_bound(q[0], k[0], v[0])
    _assert_attention(got[0][:, others], ref[:, others].astype(np.float32), bound[:, others],
                      "columns beside a NaN")
    if s > 2:
        assert np.array_equal(got[2:], good[2:])


# four waves unsplit, eight waves unsplit, four waves in three key splits, eight in three
@pytest.mark.parametrize("s,n", [(250, 300), (40, 800), (12, 866), (12, 1732)])
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
