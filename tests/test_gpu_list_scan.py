"""GPU parity of the scan by inverted list (k_scan_list.hip), the route of
large 8-bit batches: ids equal to the oracle's and float32 distances
bit-identical over every padding of the score product (subvector widths 1, 2,
3, 4, 5, 8, 12; dimensions that are not whole 32-dimension steps), lists of
ragged length, empty ones and lists shorter than a 16-entry tile, k from 1
to 200 and beyond the candidates, reranked, with OPQ, and with more equal
distances than the survivor buffers hold (the exhaustive rescue).  Also, on
the CPU, its error bound against float32 emulations of the kernel."""

import ctypes

import numpy as np
import pytest


def _print_case(msg):
    print(f"[case] {msg}", flush=True)


def _route(ix, nq, k, nprobe, pool=0):
    from vicinity_amd import _lib

    out = ctypes.c_int(-1)
    _lib.check(_lib.load().vgpu_test_scan_route(ix._h, nq, k, nprobe, pool, ctypes.byref(out)))
    return out.value


def _always(ix, on=1):
    """The scan by list for every batch whose shape has it: these small indexes
    are for its edges, not for where it is the faster scan (test_rule)."""
    from vicinity_amd import _lib

    _lib.check(_lib.load().vgpu_test_set_list_scan(ix._h, on))


def _index(oracle, rng, n, d, L, M, K, rotation=None, x=None, together=None):
    """(GPU index, oracle index) over mixture data; the lists are cut from a
    random assignment with ragged sizes, one empty and one of three entries
    (rows `together` share a list)."""
    import vicinity_amd as v

    if x is None:
        c = rng.standard_normal((40, d)).astype(np.float32)
        x = c[rng.integers(0, 40, n)] + 0.5 * rng.standard_normal((n, d)).astype(np.float32)
    x = oracle.normalize_rows(x.astype(np.float32))
    cent = oracle.normalize_rows(x[rng.choice(n, L, replace=False)].copy())
    sizes = rng.integers(1, 9, L).astype(np.float64)
    assign = rng.choice(L, n, p=sizes / sizes.sum())
    assign[assign == 1] = 2  # list 1 is empty
    assign[assign == 3] = 4
    assign[:3] = 3
    if together is not None:
        assign[together] = 5
    order = np.argsort(assign, kind="stable").astype(np.uint32)
    off = np.concatenate([[0], np.cumsum(np.bincount(assign, minlength=L))]).astype(np.uint64)
    res = x - cent[assign]
    if rotation is not None:
        res = res @ rotation.T
    ds = d // M
    books = np.stack([res[rng.choice(n, K, replace=False), m * ds:(m + 1) * ds] for m in range(M)])
    books = np.ascontiguousarray(books.astype(np.float32))
    codes = np.empty((n, M), np.uint8)
    for m in range(M):
        s = res[:, m * ds:(m + 1) * ds]
        codes[:, m] = ((s * s).sum(1)[:, None] - 2 * s @ books[m].T + (books[m] ** 2).sum(1)).argmin(1)
    ix = v.IVFPQIndex(d, num_clusters=L, num_codebooks=M, codebook_size=K, nprobe=4,
                      use_opq=rotation is not None)
    ix.load_artifacts(cent, books, off, order, codes, vectors=x, rotation=rotation)
    _always(ix)
    oix = oracle.Index(cent, books.reshape(-1), off, order, codes, np.arange(n, dtype=np.uint32), x, M, K,
                       rotation)
    return ix, oix, x


def _same(ix, oix, q, k, P, pool=0, route=1):
    assert _route(ix, len(q), k, P, pool) == route, (len(q), k, P, pool)
    ids, dists = ix.batch_search(q, k, nprobe=P, rerank_pool=pool or None)
    oids, odists = oix.search_batch(q, k, P, rerank_pool=pool)
    assert np.array_equal(ids, oids), (k, P, pool)
    assert dists.tobytes() == odists.tobytes(), (k, P, pool)


@pytest.mark.gpu
@pytest.mark.parametrize("d,M,K", [(25, 25, 256), (50, 25, 256), (36, 12, 256), (100, 25, 256),
                                   (60, 12, 64), (96, 12, 256), (72, 6, 256), (104, 13, 100)])
def test_padded_shapes(oracle, d, M, K):
    _print_case(f"list scan d={d} M={M} ksub={K}")
    rng = np.random.default_rng(7 * d + M)
    ix, oix, x = _index(oracle, rng, 6000, d, 24, M, K)
    for nq, k, P in [(3001, 10, 9), (2999, 1, 12), (2500, 100, 24), (2500, 200, 7)]:
        q = (x[rng.integers(0, len(x), nq)] + 0.2 * rng.standard_normal((nq, d))).astype(np.float32)
        q = np.tile(q, (int(0.085e9 // (nq * P * 250 * M)) + 1, 1))  # enough work for the route
        _same(ix, oix, q, k, P)
    _same(ix, oix, q, 10, 9, pool=60)


@pytest.mark.gpu
def test_more_results_than_entries_and_rotated_residuals(oracle):
    rng = np.random.default_rng(3)
    _print_case("list scan: k beyond the probed entries")
    ix, oix, x = _index(oracle, rng, 900, 100, 30, 25, 256)
    q = x[rng.integers(0, 900, 70_000)] + 0.1 * rng.standard_normal((70_000, 100)).astype(np.float32)
    _same(ix, oix, q[:60_000].astype(np.float32), 150, 2)
    _print_case("list scan: OPQ")
    rot = np.ascontiguousarray(np.linalg.qr(rng.standard_normal((64, 64)))[0].astype(np.float32))
    ix, oix, x = _index(oracle, rng, 5000, 64, 16, 16, 64, rotation=rot)
    q = x[rng.integers(0, 5000, 1500)] + 0.2 * rng.standard_normal((1500, 64)).astype(np.float32)
    for k, P in [(10, 5), (100, 16)]:
        _same(ix, oix, q.astype(np.float32), k, P)


@pytest.mark.gpu
@pytest.mark.parametrize("copies,k", [(300, 10), (1500, 100), (9000, 10)])
def test_equal_distances_beyond_the_buffers(oracle, copies, k):
    """Copies of one vector: more entries within the bound than are rescored
    (300, 1500) or kept (9000); ties come back in insertion order."""
    _print_case(f"list scan: {copies} equal entries, k {k}")
    rng = np.random.default_rng(copies)
    x = rng.standard_normal((4000, 100)).astype(np.float32)
    x = np.concatenate([np.repeat(x[:1], copies, axis=0), x])
    perm = rng.permutation(len(x))
    ix, oix, xn = _index(oracle, rng, len(x), 100, 16, 25, 256, x=x[perm], together=perm < copies)
    q = np.concatenate([np.repeat(x[:1], 40, axis=0), x[rng.integers(0, len(x), 2000)]])
    q = (q + 1e-3 * rng.standard_normal(q.shape)).astype(np.float32)
    _same(ix, oix, q, k, 16)
    assert ix.last_stats()["fallback_queries"] >= 40


def _rule(d, M, K, L, n, nq, P, k, opq=0, repeats=1.0):
    from vicinity_amd import _lib

    out = ctypes.c_int(-1)
    _lib.check(_lib.load().vgpu_test_list_rule(d, M, K, L, n, nq, P, k, opq, repeats, ctypes.byref(out)))
    return out.value


@pytest.mark.parametrize("d,M,K,L,n,nq,P,k,opq", [
    # the sample's bound leaves more survivors than a buffer holds: few long lists, a large k
    (128, 16, 256, 256, 1_000_000, 1000, 64, 100, 0), (128, 16, 256, 16, 300_000, 1000, 8, 100, 0),
    (128, 16, 256, 1, 300_000, 500, 1, 10, 0), (128, 16, 256, 2, 300_000, 500, 2, 10, 0),
    (128, 16, 256, 64, 300_000, 1000, 64, 100, 0), (128, 16, 256, 16, 300_000, 5000, 8, 100, 1),
    # few entries per query: the FAST scan has little to do
    (32, 8, 256, 1024, 50_000, 4000, 20, 10, 0), (128, 16, 256, 1024, 300_000, 16_000, 1, 100, 0),
    (100, 50, 16, 1, 300_000, 500, 1, 100, 0), (100, 50, 16, 8, 300_000, 500, 4, 100, 0),
    # rescoring by odd widths costs more than the lookups saved
    (96, 16, 256, 1024, 300_000, 10_000, 32, 100, 0), (96, 32, 256, 1024, 300_000, 10_000, 32, 200, 0),
    (96, 6, 256, 1024, 300_000, 10_000, 32, 100, 0), (128, 4, 256, 1024, 300_000, 10_000, 32, 100, 0),
    # small codebooks: cheap tables and lookups
    (96, 8, 32, 1024, 300_000, 1200, 32, 10, 0), (96, 4, 64, 1024, 300_000, 2500, 32, 10, 0),
    (96, 16, 64, 1024, 300_000, 600, 32, 10, 0),
])
def test_rule_keeps_the_other_scan_where_it_is_faster(d, M, K, L, n, nq, P, k, opq):
    assert _rule(d, M, K, L, n, nq, P, k, opq) == 0


@pytest.mark.parametrize("d,M,K,L,n,nq,P,k,opq,tiles", [
    (128, 16, 256, 4096, 1_000_000, 10_000, 32, 100, 0, 32), (25, 25, 256, 1024, 1_183_514, 10_000, 32, 10, 0, 32),
    (96, 48, 256, 16_384, 10_000_000, 10_000, 64, 10, 0, 32), (128, 16, 256, 2048, 500_000, 5000, 32, 100, 1, 32),
    (100, 50, 16, 2048, 1_000_000, 10_000, 64, 100, 0, 128), (100, 50, 16, 64, 300_000, 500, 64, 100, 0, 128),
    # longer lists: a larger sample
    (100, 25, 256, 64, 300_000, 500, 16, 10, 0, 64), (100, 25, 256, 64, 300_000, 500, 64, 10, 0, 256),
    (100, 25, 256, 128, 300_000, 3000, 4, 100, 0, 64), (128, 16, 256, 512, 1_000_000, 1000, 32, 100, 0, 256),
])
def test_rule_takes_the_scan_by_list(d, M, K, L, n, nq, P, k, opq, tiles):
    assert _rule(d, M, K, L, n, nq, P, k, opq) == tiles


@pytest.mark.gpu
@pytest.mark.parametrize("M", [16, 12])
def test_rotated_entries_that_share_codes(oracle, M):
    """An OPQ index whose lists hold many copies of few code rows: its batches
    keep the EXACT scan, which has no ties to fail on; copies of no row: they do
    not."""
    rng = np.random.default_rng(M)
    d = M * 8
    rot = np.ascontiguousarray(np.linalg.qr(rng.standard_normal((d, d)))[0].astype(np.float32))
    for distinct, route in [(12, 0), (6000, 1)]:
        _print_case(f"list scan: OPQ M={M}, {distinct} distinct rows of 30,000")
        x = rng.standard_normal((distinct, d)).astype(np.float32)[rng.integers(0, distinct, 30_000)]
        if route:  # near copies: codes of their own
            x += 0.3 * rng.standard_normal(x.shape).astype(np.float32)
        ix, oix, xn = _index(oracle, rng, len(x), d, 12, M, 256, rotation=rot, x=x)
        _always(ix, 0)
        q = (x[rng.integers(0, len(x), 2000)] + 1e-3 * rng.standard_normal((2000, d))).astype(np.float32)
        _same(ix, oix, q, 10, 12, route=route)


@pytest.mark.gpu
@pytest.mark.parametrize("n,tiles", [(9000, 64), (25_000, 128), (50_000, 256)])
def test_larger_samples(oracle, n, tiles):
    _print_case(f"list scan: samples of {tiles} tiles")
    rng = np.random.default_rng(n)
    x = rng.random((n, 25)).astype(np.float32)
    ix, oix, _ = _index(oracle, rng, n, 25, 6, 25, 256, x=x)
    q = rng.random((1501, 25)).astype(np.float32)
    assert _rule(25, 25, 256, 6, n, len(q), 6, 100) == tiles
    _same(ix, oix, q, 100, 6)
    assert ix.last_stats()["fallback_queries"] < 15


@pytest.mark.gpu
@pytest.mark.parametrize("opq", [False, True])
def test_unclustered_rows_in_few_long_lists(oracle, opq):
    """Uniform rows, six lists, k 250: with the scan by list nearly every query
    leaves more survivors than its buffer holds, whatever
    its sample.  The mode's own scan is taken,
    and the scan by list still agrees."""
    _print_case(f"list scan: uniform rows in six lists, opq {opq}")
    rng = np.random.default_rng(8)
    n, d = 80_000, 32
    x = rng.random((n, d)).astype(np.float32)
    rot = np.ascontiguousarray(np.linalg.qr(rng.standard_normal((d, d)))[0].astype(np.float32)) if opq else None
    ix, oix, _ = _index(oracle, rng, n, d, 6, 8, 256, rotation=rot, x=x)
    q = rng.random((200, d)).astype(np.float32)
    _same(ix, oix, q, 250, 6)
    assert ix.last_stats()["fallback_queries"] > 64  # more than list_rescue_kernel takes
    _same(ix, oix, q[:20], 250, 6)
    assert 0 < ix.last_stats()["fallback_queries"] <= 64
    _always(ix, 0)
    _same(ix, oix, q, 250, 6, route=0)


@pytest.mark.gpu
@pytest.mark.parametrize("opq,d,M,K", [(False, 100, 25, 256), (True, 128, 16, 256), (True, 64, 16, 64)])
def test_crowds_of_flagged_queries(oracle, opq, d, M, K):
    """300 flagged queries in the first chunk and 20 in the second (16,384 a
    chunk), of which list_rescue_kernel takes the 20 and the EXACT kernel the
    300: 1500 equal entries are kept but not rescored, 6000 are not kept."""
    rng = np.random.default_rng(d + M)
    rot = np.ascontiguousarray(np.linalg.qr(rng.standard_normal((d, d)))[0].astype(np.float32)) if opq else None
    for copies in (1500, 6000):
        _print_case(f"list scan: crowds of flagged queries, {copies} copies, d={d} M={M} ksub={K} opq={opq}")
        x = rng.standard_normal((2000, d)).astype(np.float32)
        x = np.concatenate([np.repeat(x[:1], copies, axis=0), x])
        perm = rng.permutation(len(x))
        ix, oix, _ = _index(oracle, rng, len(x), d, 16, M, K, rotation=rot, x=x[perm], together=perm < copies)
        q = x[rng.integers(copies + 10, len(x), 16_450)]
        q[np.concatenate([np.arange(0, 3000, 10), np.arange(16_400, 16_420)])] = x[0]
        q = (q + 1e-3 * rng.standard_normal(q.shape)).astype(np.float32)
        _same(ix, oix, q, 20, 16)
        assert ix.last_stats()["fallback_queries"] >= 320
        _same(ix, oix, q[:2000], 20, 16)
        assert ix.last_stats()["fallback_queries"] >= 200


@pytest.mark.gpu
@pytest.mark.parametrize("d,K", [(64, 256), (96, 100), (100, 256)])
def test_one_dimensional_codebooks_of_several_steps(oracle, d, K):
    """Two to four 32-dimension steps of one-dimensional codebooks (25, one
    step, is among test_padded_shapes)."""
    _print_case(f"list scan: d=M={d} ksub={K}")
    rng = np.random.default_rng(d)
    ix, oix, x = _index(oracle, rng, 3000, d, 12, d, K)
    q = (x[rng.integers(0, 3000, 700)] + 0.2 * rng.standard_normal((700, d))).astype(np.float32)
    for k, P in [(10, 9), (100, 12)]:
        _same(ix, oix, q, k, P)


@pytest.mark.parametrize("d,M,scale", [(32, 8, 1.0), (96, 48, 0.05), (128, 16, 30.0)])
def test_error_bound(oracle, d, M, scale):
    """|a - e| <= list_tau with a from bf16x3 products as the score kernel makes
    them (32-dimension steps, low times high, high times low, high times high,
    started from -|y|^2 / 2; each step's sum rounded once, after every product, or
    toward zero) and e the reference's float32 distance.  Random residuals, and
    rows whose low halves are largest and of one sign: there the products dropped
    from bf16x3 alone exceed the bound's other terms."""
    from test_flat_key_bound import _score
    from test_proof_bounds import seq_sum

    from vicinity_amd import _lib

    rng = np.random.default_rng(d)
    F32 = np.float32
    r = (scale * rng.standard_normal((200, d))).astype(F32)
    y = (r + scale * 10.0 ** rng.uniform(-3, 0, (200, 1)) * rng.standard_normal((200, d))).astype(F32)
    r[:20] = y[:20] = 2.0 ** np.round(np.log2(scale)) * (1.0 + 2.0 ** -8 * rng.uniform(0.97, 0.999, (20, d)))
    yn = np.sum(y.astype(np.float64) ** 2, 1)
    t0 = seq_sum((r * r).astype(F32))
    diff = (r - y).astype(F32)
    e = seq_sum(seq_sum((diff * diff).astype(F32).reshape(200, M, -1))).astype(np.float64)
    out = ctypes.c_float()
    tau, rest = np.empty(200), np.empty(200)
    u, ds = 2.0 ** -24, d // M
    for i in range(200):
        _lib.check(_lib.load().vgpu_test_bound_list(d, M, ds, float(t0[i]), float(np.sqrt(yn[i])),
                                                    ctypes.byref(out)))
        tau[i] = out.value
        # the terms that are not the products'
        rest[i] = 1.25 * ((d + 4) * u * t0[i] + (ds + M + 6) * u * (np.sqrt(t0[i]) + np.sqrt(yn[i])) ** 2)
    for order in ("exact", "seq", "trunc"):
        D = _score(y, r, (-0.5 * yn).astype(F32), order).astype(np.float64)
        a = (t0.astype(np.float64) - 2.0 * D).astype(F32)  # one rounding, as the kernel's fma
        err = np.abs(a.astype(np.float64) - e)
        assert (err <= tau).all(), (order, (err / tau).max())
        assert (err[:20] > rest[:20]).all(), (order, (err[:20] / rest[:20]).min())
        assert (err / tau).max() > 0.05, (order, (err / tau).max())
