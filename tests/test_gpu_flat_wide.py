"""GPU parity of the flat search's ranking kernel above k 32 (six keys per lane
list) and above 128 dimensions, against the oracle's brute force
(src/distance.rs:78-109): ids equal, float32 distances bit-identical.  Sizes at
the edges of a lane list (7 tiles in one slice), of a 32-dimension step, of a
query block and of a pass, crowded lane lists, rows and queries that are not
finite."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(ids, dists, oids, odists):
    assert ids.shape == oids.shape
    assert np.array_equal(ids, oids)
    assert dists.tobytes() == odists.tobytes()


def _index(d, metric, base):
    from vicinity_amd import FlatIndex

    fx = FlatIndex(d, "l2" if metric == 0 else "cosine")
    fx.add(base)
    return fx


@pytest.mark.parametrize("n,d,nq,k", [
    (97, 7, 3, 112),          # 7 tiles in two slices: no list fills, all 97 rows are returned
    (176, 16, 5, 112),        # 11 tiles in two slices of six: lists exactly full
    (3600, 20, 9, 112),       # slices of eight tiles: more tiles than keys in a list
    (1000, 129, 129, 33),     # k just past 32, five steps, one dimension of the last
    (3001, 256, 40, 112),     # the largest d and k
    (9000, 160, 33, 1),       # wide rows, few keys
    (17_000, 128, 260, 100),  # three query blocks
    (20_011, 200, 70, 100),   # seven steps, ragged n
    (40_000, 25, 300, 64),
    (300, 8, 40_970, 40),     # two passes
])
@pytest.mark.parametrize("metric", [0, 1])
def test_flat_wide_shapes(oracle, n, d, nq, k, metric):
    print(f"[case] flat wide n={n} d={d} nq={nq} k={k} metric={metric}", flush=True)
    rng = np.random.default_rng(n + d + k + metric)
    base = rng.standard_normal((n, d)).astype(np.float32)
    q = rng.standard_normal((nq, d)).astype(np.float32)
    if metric == 1:
        base, q = oracle.normalize_rows(base), oracle.normalize_rows(q)
    ids, dists = _index(d, metric, base).search(q, k)
    _check(ids, dists, *oracle.flat_search(base, q, k, metric=metric))


@pytest.mark.parametrize("d,k", [(64, 100), (200, 10)])
def test_flat_wide_crowded_lanes_and_ties(oracle, d, k):
    """Nine near-copies in one lane of one slice, more than a lane list keeps, and
    700 exact copies, more than the merge rescores: each ends in the exhaustive
    fallback by itself, ordinary queries do not."""
    print(f"[case] flat wide crowded d={d} k={k}", flush=True)
    rng = np.random.default_rng(d + k)
    base = rng.standard_normal((20_000, d)).astype(np.float32)
    v, w = base[17].copy(), base[18].copy()
    base[(100 + np.arange(9)) * 16 + 5] = v + 1e-4 * rng.standard_normal((9, d)).astype(np.float32)
    base[5000:5700] = w
    crowded = v + 1e-3 * rng.standard_normal((300, d)).astype(np.float32)
    ties = w + 1e-3 * rng.standard_normal((5, d)).astype(np.float32)
    rest = np.concatenate([rng.standard_normal((20, d)).astype(np.float32), np.zeros((1, d), np.float32)])
    fx = _index(d, 0, base)
    for q, least, most in [(crowded, 300, 300), (ties, 5, 5), (rest, 0, 2),
                           (np.concatenate([crowded, ties, rest]), 305, 307)]:
        ids, dists = fx.search(q, k)
        _check(ids, dists, *oracle.flat_search(base, q, k, metric=0))
        assert least <= fx.last_fallbacks() <= most, (len(q), fx.last_fallbacks())


@pytest.mark.parametrize("bad", [np.inf, 1e18])
def test_flat_wide_rows_far_from_finite(oracle, bad):
    """Infinite rows, and rows whose squares overflow float32: the fp32 path."""
    print(f"[case] flat wide bad rows {bad}", flush=True)
    rng = np.random.default_rng(5)
    base = rng.standard_normal((3000, 48)).astype(np.float32)
    base[7, 3] = bad
    base[2000] = bad
    q = rng.standard_normal((30, 48)).astype(np.float32)
    ids, dists = _index(48, 0, base).search(q, 100)
    _check(ids, dists, *oracle.flat_search(base, q, 100, metric=0))


def test_flat_wide_query_that_is_not_finite(oracle):
    """A NaN query and one whose squares overflow, beside ordinary ones: each
    gets k rows, and the others' results do not change."""
    import torch

    print("[case] flat wide NaN query", flush=True)
    rng = np.random.default_rng(6)
    n, d, k = 5000, 64, 100
    base = rng.standard_normal((n, d)).astype(np.float32)
    q = rng.standard_normal((20, d)).astype(np.float32)
    oids, odists = oracle.flat_search(base, q, k, metric=0)
    bad = q.copy()
    bad[3, 5], bad[11] = np.nan, 1e19
    ids = torch.empty((20, k), dtype=torch.int64, device="cuda:0")
    dists = torch.empty((20, k), dtype=torch.float32, device="cuda:0")
    fx = _index(d, 0, base)
    fx.search_device(torch.from_numpy(bad).to("cuda:0"), k, ids, dists)
    ids, dists = ids.cpu().numpy(), dists.cpu().numpy()
    rest = np.delete(np.arange(20), [3, 11])
    _check(ids[rest], dists[rest], oids[rest], odists[rest])
    assert np.isnan(dists[3]).all() and np.unique(ids[3]).size == k
    assert np.isinf(dists[11]).all() and np.array_equal(ids[11], np.arange(k))


@pytest.mark.parametrize("offset,metric,lost", [(0.5, 0, False), (3.0, 0, True), (30.0, 0, False), (12.0, 1, True)])
def test_flat_wide_rows_far_from_the_origin(oracle, offset, metric, lost):
    """Rows whose common offset swallows the ranking path's bound but not the
    fp32 path's (lost): the fp32 path, which proves nearly every query; the
    ranking path's exhaustive fallback had all of them."""
    print(f"[case] flat wide offset {offset} metric {metric}", flush=True)
    rng = np.random.default_rng(11)
    n, d, k = 6000, 200, 10
    c = rng.standard_normal((20, d))
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    base = (c[rng.integers(0, 20, n)] + 0.05 * rng.standard_normal((n, d)) + offset).astype(np.float32)
    q = (c[rng.integers(0, 20, 200)] + 0.05 * rng.standard_normal((200, d)) + offset).astype(np.float32)
    fx = _index(d, metric, base)
    _check(*fx.search(q, k), *oracle.flat_search(base, q, k, metric=metric))
    if lost:
        assert fx.last_fallbacks() <= 20
