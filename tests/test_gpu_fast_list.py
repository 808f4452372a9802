"""GPU parity of the 4-bit FastScan by inverted list (k_fast_list.hip), the
route of large batches: ids equal to the oracle's and float32 distances
bit-identical over the numbers of codebooks and widths it is compiled for
(whole and partial groups of four codebooks, one and two code words per lane),
ragged lists, an empty list and one below 16 entries (the exact float path), k
from 1 to 200 and beyond the candidates, reranked, rotated residuals, and more
equal distances than can be ranked or kept (the scan of flagged queries)."""

import numpy as np
import pytest

from test_gpu_list_scan import _index, _same

pytestmark = pytest.mark.gpu


def _print_case(msg):
    print(f"[case] {msg}", flush=True)


def _enough(q, P, n, L):
    """The queries repeated until the batch scans the entries the route asks for."""
    return np.tile(q.astype(np.float32), (int(31e6 // (len(q) * P * n / L)) + 1, 1))


@pytest.mark.parametrize("M,ds", [(3, 4), (16, 1), (16, 4), (17, 2), (25, 4), (32, 2), (33, 1), (50, 2), (53, 2),
                                  (64, 4)])
def test_shapes(oracle, M, ds):
    _print_case(f"4-bit scan by list M={M} ds={ds}")
    d, n, L = M * ds, 6200, 24
    rng = np.random.default_rng(100 * M + ds)
    ix, oix, x = _index(oracle, rng, n, d, L, M, 16)
    for nq, k, P in [(3001, 10, 9), (2999, 1, 12), (2500, 100, 24), (2500, 200, 7)]:
        q = x[rng.integers(0, n, nq)] + 0.2 * rng.standard_normal((nq, d)).astype(np.float32)
        _same(ix, oix, _enough(q, P, n, L), k, P)
    _same(ix, oix, _enough(q, 9, n, L), 10, 9, pool=60)


def test_few_entries_and_rotated_residuals(oracle):
    rng = np.random.default_rng(3)
    _print_case("4-bit scan by list: k beyond the probed entries")
    ix, oix, x = _index(oracle, rng, 3000, 100, 30, 50, 16)
    q = x[rng.integers(0, 3000, 80_000)] + 0.1 * rng.standard_normal((80_000, 100)).astype(np.float32)
    _same(ix, oix, _enough(q, 2, 3000, 30), 250, 2)
    _print_case("4-bit scan by list: OPQ")
    rot = np.ascontiguousarray(np.linalg.qr(rng.standard_normal((64, 64)))[0].astype(np.float32))
    ix, oix, x = _index(oracle, rng, 5000, 64, 16, 32, 16, rotation=rot)
    q = x[rng.integers(0, 5000, 3000)] + 0.2 * rng.standard_normal((3000, 64)).astype(np.float32)
    for k, P in [(10, 5), (100, 16)]:
        _same(ix, oix, _enough(q, P, 5000, 16), k, P)


@pytest.mark.parametrize("copies,k", [(1500, 100), (9000, 10)])
def test_equal_distances_beyond_the_buffers(oracle, copies, k):
    """Copies of one vector: more than are ranked (1500) or kept (9000)."""
    _print_case(f"4-bit scan by list: {copies} equal entries, k {k}")
    rng = np.random.default_rng(copies)
    x = rng.standard_normal((4000, 100)).astype(np.float32)
    x = np.concatenate([np.repeat(x[:1], copies, axis=0), x])
    perm = rng.permutation(len(x))
    ix, oix, _ = _index(oracle, rng, len(x), 100, 16, 50, 16, x=x[perm], together=perm < copies)
    q = np.concatenate([np.repeat(x[:1], 40, axis=0), x[rng.integers(0, len(x), 3000)]])
    q = (q + 1e-3 * rng.standard_normal(q.shape)).astype(np.float32)
    _same(ix, oix, _enough(q, 16, len(x), 16), k, 16)
    assert ix.last_stats()["fallback_queries"] >= 40
