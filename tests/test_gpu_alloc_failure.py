"""Device-allocation failures through the C ABI (the injection hook
vgpu_test_fail_device_allocations): a failed allocation in a search, an
upload, a build or a flat-index add returns VGPU_ERR_OUT_OF_MEMORY, leaves
the handle usable, and the same call succeeds once the hook is disarmed,
with results equal to the oracle's."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _print_case(msg):
    print(f"[case] {msg}", flush=True)


@pytest.fixture
def fail():
    from vicinity_amd import _lib

    def arm(after, count=1):
        _lib.check(_lib.load().vgpu_test_fail_device_allocations(after, count))

    yield arm
    arm(0, 0)


def _oom(excinfo):
    from vicinity_amd import _lib

    assert excinfo.value.code == _lib.ERR_OUT_OF_MEMORY
    assert "injected" in str(excinfo.value)


def _oracle_index(oracle, art):
    return oracle.Index(art["centroids"], art["codebooks"], art["list_offsets"], art["list_ids"],
                        art["codes"], art["doc_ids"], art["vectors"], art["M"], art["K"])


def test_search_upload_and_build_recover_from_allocation_failure(oracle, fail):
    import vicinity_amd as v
    from vicinity_amd import VicinityGpuError

    assert v.device_available(), "no gfx950 device visible"
    w = v.datagen.ivfpq_small(n=6000, nq=200)
    _print_case("alloc failure: build 6000 x 32, nlist 32 with the 4th allocation failing")
    ix = v.IVFPQIndex(32, num_clusters=32, num_codebooks=8, codebook_size=256, nprobe=4, seed=3)
    ix.add_items(w.base)
    fail(3)
    with pytest.raises(VicinityGpuError) as e:
        ix.build(kmeans_max_iter=5)
    _oom(e)
    fail(0, 0)
    assert not ix.is_built
    ix.build(kmeans_max_iter=5)
    art = ix.export()
    oix, _ = oracle.ivfpq_build(oracle.normalize_rows(w.base), 32, 8, 256, 3, 0, 5)
    assert art["codes"].tobytes() == oix.codes.tobytes()
    assert art["centroids"].tobytes() == oix.centroids.tobytes()

    _print_case("alloc failure: first search on the handle (workspace allocation)")
    fail(0)
    with pytest.raises(VicinityGpuError) as e:
        ix.batch_search(w.queries, 10)
    _oom(e)
    fail(0, 0)
    ids, dists = ix.batch_search(w.queries, 10)
    oids, odists = _oracle_index(oracle, art).search_batch(w.queries, 10, 4)
    assert np.array_equal(ids, oids) and dists.tobytes() == odists.tobytes()

    _print_case("alloc failure: load_artifacts with the 3rd upload failing")
    ix2 = v.IVFPQIndex(32, num_clusters=32, num_codebooks=8, codebook_size=256, nprobe=4)
    args = (art["centroids"], art["codebooks"], art["list_offsets"], art["list_ids"], art["codes"])
    fail(2)
    with pytest.raises(VicinityGpuError) as e:
        ix2.load_artifacts(*args, vectors=art["vectors"])
    _oom(e)
    fail(0, 0)
    ix2.load_artifacts(*args, vectors=art["vectors"])
    ids2, dists2 = ix2.batch_search(w.queries, 10, rerank_pool=30)
    oids2, odists2 = _oracle_index(oracle, art).search_batch(w.queries, 10, 4, 30)
    assert np.array_equal(ids2, oids2) and dists2.tobytes() == odists2.tobytes()


def test_flat_add_recovers_from_allocation_failure(oracle, fail):
    from vicinity_amd import FlatIndex, VicinityGpuError

    _print_case("alloc failure: flat add 3000 x 48")
    rng = np.random.default_rng(4)
    base = rng.standard_normal((3000, 48)).astype(np.float32)
    q = rng.standard_normal((40, 48)).astype(np.float32)
    fx = FlatIndex(48, "l2")
    fail(0)
    with pytest.raises(VicinityGpuError) as e:
        fx.add(base[:1000])
    _oom(e)
    fail(0, 0)
    fx.add(base[:1000])
    # the second add's norm buffer fails after its rows were uploaded: the
    # index goes back to its first 1000 rows
    fail(1)
    with pytest.raises(VicinityGpuError) as e:
        fx.add(base[1000:])
    _oom(e)
    fail(0, 0)
    ids, dists = fx.search(q, 10)
    oids, odists = oracle.flat_search(base[:1000], q, 10, metric=0)
    assert np.array_equal(ids, oids) and dists.tobytes() == odists.tobytes()
    fx.add(base[1000:])
    ids, dists = fx.search(q, 10)
    oids, odists = oracle.flat_search(base, q, 10, metric=0)
    assert np.array_equal(ids, oids) and dists.tobytes() == odists.tobytes()


@pytest.mark.parametrize("d,M,K", [(64, 16, 256), (50, 25, 256), (32, 16, 16)])
def test_upload_without_memory_for_the_scan_by_list(oracle, fail, d, M, K):
    """The list-scan arrays are optional: an upload that cannot hold them
    succeeds, and a large batch takes the scan it has without them."""
    from test_gpu_list_scan import _always, _index, _route

    import vicinity_amd as v
    from vicinity_amd import VicinityGpuError

    _print_case(f"alloc failure: list-scan arrays, d={d} M={M} ksub={K}")
    rng = np.random.default_rng(d)
    ix, oix, x = _index(oracle, rng, 3000, d, 16, M, K)
    art = ix.export()
    q = (x[rng.integers(0, 3000, 500)] + 0.1 * rng.standard_normal((500, d))).astype(np.float32)
    want = oix.search_batch(q, 10, 16)
    without = 0
    for after in range(40):
        one = v.IVFPQIndex(d, num_clusters=16, num_codebooks=M, codebook_size=K, nprobe=16)
        fail(after)
        try:
            one.load_artifacts(*(art[n] for n in ("centroids", "codebooks", "list_offsets", "list_ids", "codes")))
        except VicinityGpuError:
            continue
        finally:
            fail(0, 0)
        _always(one)
        route = _route(one, 500, 10, 16)
        ids, dists = one.batch_search(q, 10)
        assert np.array_equal(ids, want[0]) and dists.tobytes() == want[1].tobytes(), after
        if route == 1:
            break
        without += 1
    assert route == 1 and without >= 2


@pytest.mark.parametrize("d,M,K", [(64, 16, 256), (32, 16, 16)])
def test_search_without_memory_for_the_scan_by_list(oracle, fail, d, M, K):
    """A batch whose list-scan workspace cannot be had takes the scan it has
    without it; the next batch takes the scan by list again."""
    import torch

    from test_gpu_list_scan import _index, _route
    from vicinity_amd import VicinityGpuError

    _print_case(f"alloc failure: list-scan workspace, d={d} M={M} ksub={K}")
    rng = np.random.default_rng(d)
    ix, oix, x = _index(oracle, rng, 3000, d, 16, M, K)
    q = (x[rng.integers(0, 3000, 500)] + 0.1 * rng.standard_normal((500, d))).astype(np.float32)
    want = oix.search_batch(q, 10, 16)
    qd = torch.from_numpy(q).to("cuda:0")
    assert _route(ix, 500, 10, 16) == 1

    def search():
        ids, dists = ix.search_batch_device(qd, 10, nprobe=16)
        assert np.array_equal(ids.cpu().numpy(), want[0]) and dists.cpu().numpy().tobytes() == want[1].tobytes()
        return ix.last_stats()["fast_appends"]  # the list scan: its survivors

    fail(0, 4)  # both scans' workspaces, each twice
    with pytest.raises(VicinityGpuError) as e:
        ix.search_batch_device(qd, 10, nprobe=16)
    _oom(e)
    fail(0, 2)
    without = search()
    fail(0, 0)
    assert search() != without
    fail(0, 1)
    ids, dists = ix.search_batch_device(qd, 10, nprobe=16)  # the workspace is there: nothing is allocated
    assert np.array_equal(ids.cpu().numpy(), want[0])


def test_search_tries_its_workspace_twice(fail):
    """A failed workspace is tried again once the idle ones' memory is free."""
    import vicinity_amd as v

    w = v.datagen.ivfpq_small(n=6000, nq=1000)
    _print_case("alloc failure: a larger workspace, once")
    ix = v.IVFPQIndex(32, num_clusters=32, num_codebooks=8, codebook_size=256, nprobe=4, seed=3)
    ix.add_items(w.base)
    ix.build(kmeans_max_iter=3)
    want = ix.batch_search(w.queries, 10)
    fail(3)  # the queries, ids and distances are staged, then the workspace fails
    ids, dists = ix.batch_search(np.concatenate([w.queries] * 3), 10)
    assert np.array_equal(ids[:1000], want[0]) and dists[2000:].tobytes() == want[1].tobytes()


@pytest.mark.parametrize("d,k", [(48, 10), (48, 100), (160, 10)])
def test_flat_without_memory_for_the_ranking_path(oracle, fail, d, k):
    """The packed copy is optional, and a search whose buffer fails goes in
    smaller passes."""
    from vicinity_amd import FlatIndex

    _print_case(f"alloc failure: flat pack and search buffers, d={d} k={k}")
    rng = np.random.default_rng(d + k)
    base = rng.standard_normal((4000, d)).astype(np.float32)
    q = rng.standard_normal((5000, d)).astype(np.float32)
    oids, odists = oracle.flat_search(base, q, k, metric=0)
    fx = FlatIndex(d, "l2")
    fail(2)  # rows and norms are there, the packed copy is not
    fx.add(base)
    fail(0, 0)
    ids, dists = fx.search(q[:500], k)
    assert np.array_equal(ids, oids[:500]) and dists.tobytes() == odists[:500].tobytes()
    fx = FlatIndex(d, "l2")
    fx.add(base)
    # the staged queries, ids and distances, then the search buffer twice
    fail(3, 2)
    ids, dists = fx.search(q, k)
    fail(0, 0)
    assert np.array_equal(ids, oids) and dists.tobytes() == odists.tobytes()
