"""The work this framework is used for, as cases that can be timed.

A case is one call of a public entry point on an index that is already
resident: batched IVF-PQ search (8-bit codes, 4-bit FastScan with rerank, OPQ,
filtered), exact flat search, and an index build.  Shapes are the benchmark's
five workloads (vicinity_amd/datagen.py), the shapes the reference publishes
(d 25 with one-dimensional subvectors; 10k x 96 with a rerank pool) and generic
ones.  Data are Gaussian mixtures like the benchmark's.  Index arrays are made
here with torch and uploaded with load_artifacts, as a program does that loads
a saved index.

Results are the reference's float32 values bit for bit (that is the search
path's contract, which the tests check against the oracle), so every tolerance
is "exact".
"""

from __future__ import annotations

import math

import numpy as np
import torch

DEV = "cuda:0"


def listed():
    return [
        # one interactive query on a small collection, host arrays in and out
        dict(name="one_query", kind="search", n=10_000, d=96, nlist=100, M=16, K=256, nprobe=8,
             k=10, pool=100, nq=1, centres=50, std=0.1, host=True, opq=False),
        # the benchmark's small workload: a batch where launches count
        dict(name="small_batch", kind="search", n=20_000, d=32, nlist=64, M=8, K=256, nprobe=8,
             k=10, pool=0, nq=1000, centres=0, std=0.0, host=False, opq=False),
        # a serving batch: a few dozen queries against a mid-sized collection, ragged sizes
        dict(name="serving_batch", kind="search", n=300_007, d=100, nlist=1021, M=25, K=256,
             nprobe=16, k=10, pool=0, nq=61, centres=300, std=0.1, host=False, opq=False),
        # the benchmark's headline batch
        dict(name="headline_1m_d128", kind="search", n=1_000_000, d=128, nlist=4096, M=16, K=256,
             nprobe=32, k=100, pool=0, nq=10_000, centres=1000, std=0.0096, cube=True, host=False,
             opq=False),
        # the reference's published shape: one-dimensional subvectors
        dict(name="glove_d25", kind="search", n=1_183_514, d=25, nlist=1024, M=25, K=256,
             nprobe=32, k=10, pool=0, nq=10_000, centres=1000, std=0.12, host=False, opq=False),
        # the benchmark's large workload: many short subvectors, many lists
        dict(name="angular_10m_d96", kind="search", n=10_000_000, d=96, nlist=16_384, M=48, K=256,
             nprobe=64, k=10, pool=0, nq=10_000, centres=10_000, std=0.1, host=False, opq=False),
        # text-embedding vectors
        dict(name="embedding_d768", kind="search", n=100_003, d=768, nlist=317, M=96, K=256,
             nprobe=12, k=10, pool=0, nq=1000, centres=200, std=0.04, host=False, opq=False),
        # an index trained with the OPQ rotation
        dict(name="opq_d128", kind="search", n=500_000, d=128, nlist=2048, M=16, K=256, nprobe=32,
             k=100, pool=0, nq=5000, centres=500, std=0.0096, cube=True, host=False, opq=True),
        # the benchmark's 4-bit workload: FastScan, then the exact rerank of a pool
        dict(name="fastscan_rerank", kind="search", n=1_000_000, d=100, nlist=2048, M=50, K=16,
             nprobe=64, k=10, pool=100, nq=10_000, centres=500, std=0.1, host=False, opq=False),
        # the benchmark's exact search
        dict(name="flat_100k_d96", kind="flat", n=100_000, d=96, k=10, metric="l2", nq=10_000,
             centres=100, std=0.05),
        # recall ground truth of the headline (its k, cosine distances, a quarter of its rows)
        dict(name="ground_truth_k100", kind="flat", n=250_000, d=128, k=100, metric="cosine",
             nq=10_000, centres=1000, std=0.0096, cube=True),
        # an index made from raw vectors: k-means, PQ training, encoding, lists
        dict(name="build_d64", kind="build", n=50_000, d=64, nlist=256, M=16, K=256, iters=10,
             sample=20_000, centres=200, std=0.08),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: searches mostly (8-bit and 4-bit,
    with and without a rerank, OPQ), flat searches, now and then a build."""
    kind = rng.choice(["search"] * 6 + ["flat"] * 2 + ["build"])
    centres, std, cube = _log_int(rng, 50, 2000), round(rng.uniform(0.05, 0.12), 3), False
    if rng.random() < 0.4:  # tight clusters, like the headline's
        std, cube = round(rng.uniform(0.008, 0.03), 4), True
    if kind == "build":
        ds, M = rng.choice([2, 4, 8]), rng.choice([4, 8, 16])
        return dict(kind="build", n=_log_int(rng, 5000, 60_000), d=ds * M,
                    nlist=_log_int(rng, 16, 300), M=M, K=rng.choice([16, 256]),
                    iters=rng.randint(4, 10), sample=_log_int(rng, 4000, 20_000), centres=centres,
                    std=std, cube=cube)
    if kind == "flat":
        return dict(kind="flat", n=_log_int(rng, 2000, 200_000), d=rng.randint(16, 200),
                    k=_log_int(rng, 1, 100), metric=rng.choice(["l2", "cosine"]),
                    nq=_log_int(rng, 1, 10_000), centres=centres, std=std, cube=cube)
    K = rng.choice([256, 256, 256, 256, 64, 16])
    M, ds = rng.choice([(8, 4), (8, 16), (12, 8), (16, 4), (16, 6), (16, 8), (20, 5), (25, 1),
                        (25, 2), (25, 4), (32, 3), (32, 4), (48, 2), (50, 2), (96, 8)])
    if K == 16:
        M, ds = rng.choice([(16, 4), (25, 4), (32, 2), (50, 2), (64, 2)])
    n = _log_int(rng, 10_000, 1_000_000 if M * ds <= 128 else 150_000)
    nlist = max(16, min(4096, int(n / rng.uniform(60, 900))))
    nprobe = min(nlist, _log_int(rng, 1, 64))
    pool = rng.choice([0, 0, 100]) if K != 16 else rng.choice([0, 100])
    k = _log_int(rng, 1, 100)
    nq = _log_int(rng, 1, 10_000 if M * ds <= 128 else 2000)
    return dict(kind="search", n=n, d=M * ds, nlist=nlist, M=M, K=K, nprobe=nprobe, k=k, pool=pool,
                nq=nq, centres=centres, std=std, cube=cube, host=nq < 50 and rng.random() < 0.5,
                opq=K != 16 and M * ds <= 128 and rng.random() < 0.15)


# ---- data -------------------------------------------------------------------

def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed(1_000_003 * (seed + 1) + salt)


def _unit(x):
    return x / x.norm(dim=1, keepdim=True).clamp_min(1e-30)


def _mixture(centres, n, std, g):
    """n rows around random centres, chunked so that the temporaries stay small."""
    out = torch.empty((n, centres.shape[1]), device=DEV)
    for s in range(0, n, 1 << 20):
        e = min(n, s + (1 << 20))
        lab = torch.randint(0, centres.shape[0], (e - s,), generator=g, device=DEV)
        x = torch.randn((e - s, centres.shape[1]), generator=g, device=DEV)
        out[s:e] = x.mul_(std).add_(centres[lab])
    return out


def _data(case, seed):
    """(base, queries) on the GPU: rows around unit centres (with "cube", centres
    of one orthant, like the benchmark's centres in [0, 128)^d), or uniform in
    [0, 1) without centres."""
    d, nq = case["d"], case.get("nq", 1)
    if not case["centres"]:
        return (torch.rand((case["n"], d), generator=_gen(seed, 1), device=DEV),
                torch.rand((nq, d), generator=_gen(seed, 2), device=DEV))
    make = torch.rand if case.get("cube") else torch.randn
    c = _unit(make((case["centres"], d), generator=_gen(seed, 0), device=DEV))
    return (_mixture(c, case["n"], case["std"], _gen(seed, 1)),
            _mixture(c, nq, case["std"], _gen(seed, 2)))


def _nearest(x, cent, by_dot):
    """The nearest centroid of each row (by dot product, or by Euclidean distance)."""
    out = torch.empty(x.shape[0], dtype=torch.int64, device=DEV)
    half = 0.5 * (cent * cent).sum(1)
    step = max(1, (1 << 29) // cent.shape[0])
    for s in range(0, x.shape[0], step):
        sc = x[s:s + step] @ cent.T
        out[s:s + step] = (sc if by_dot else sc.sub_(half)).argmax(1)
    return out


def _means(x, lab, cent):
    """Means of the rows of each label; a label without rows keeps its centroid.
    The sums are of integers (value * 2^20), so any order of adding gives the same."""
    acc = torch.zeros(cent.shape, dtype=torch.int64, device=DEV)
    acc.index_add_(0, lab, (x.double() * 2.0 ** 20).round().long())
    cnt = torch.bincount(lab, minlength=cent.shape[0])
    mean = (acc.double() / (2.0 ** 20 * cnt.clamp_min(1).unsqueeze(1))).float()
    return torch.where(cnt.unsqueeze(1) > 0, mean, cent)


def _artifacts(case, seed):
    """A trained IVF-PQ index as torch arrays: two k-means passes over a sample
    for the coarse centroids and for each codebook, then every row assigned
    and its residual (rotated, with OPQ) encoded."""
    n, d, L, M, K = case["n"], case["d"], case["nlist"], case["M"], case["K"]
    ds = d // M
    base, queries = _data(case, seed)
    base = _unit(base)
    g = _gen(seed, 3)
    pick = torch.randperm(n, generator=g, device=DEV)[:max(20 * L, 20_000)]
    sample = base[pick]
    cent = sample[:L].clone()
    for _ in range(2):
        cent = _unit(_means(sample, _nearest(sample, cent, True), cent))
    assign = _nearest(base, cent, True)
    rot = None
    if case["opq"]:
        r = torch.randn((d, d), generator=g, device=DEV).cpu().double().numpy()
        rot = torch.from_numpy(np.linalg.qr(r)[0].astype(np.float32)).to(DEV)

    def residual(rows, lists):
        r = rows - cent[lists]
        return r if rot is None else r @ rot.T

    rs = residual(sample[:16_384], assign[pick[:16_384]])
    books = torch.empty((M, K, ds), device=DEV)
    for m in range(M):
        sub = rs[:, m * ds:(m + 1) * ds].contiguous()
        cw = sub[:K].clone()
        for _ in range(2):
            cw = _means(sub, _nearest(sub, cw, False), cw)
        books[m] = cw
    codes = torch.empty((n, M), dtype=torch.uint8, device=DEV)
    step = 1 << 20
    for s in range(0, n, step):
        r = residual(base[s:s + step], assign[s:s + step])
        for m in range(M):
            codes[s:s + step, m] = _nearest(r[:, m * ds:(m + 1) * ds].contiguous(), books[m],
                                            False).to(torch.uint8)
    order = torch.sort(assign, stable=True).indices
    off = torch.zeros(L + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.bincount(assign, minlength=L).cumsum(0)
    return dict(base=base, queries=queries.contiguous(), centroids=cent, codebooks=books,
                codes=codes, order=order, offsets=off, rotation=rot)


# ---- the cases --------------------------------------------------------------

def prepare(case, seed):
    import vicinity_amd as v

    kind, state = case["kind"], dict(case=case)
    if kind == "build":
        state["base"] = _data(case, seed)[0].cpu().numpy()
        return state
    nq, k = case["nq"], case["k"]
    if kind == "flat":
        base, q = _data(case, seed)
        if case["metric"] == "cosine":
            base, q = _unit(base), _unit(q)
        ix = v.FlatIndex(case["d"], case["metric"])
        ix.add(base.cpu().numpy())
    else:
        a = _artifacts(case, seed)
        q = a["queries"]
        ix = v.IVFPQIndex(case["d"], num_clusters=case["nlist"], num_codebooks=case["M"],
                          codebook_size=case["K"], nprobe=case["nprobe"], use_opq=case["opq"])
        ix.load_artifacts(a["centroids"].cpu().numpy(), a["codebooks"].cpu().numpy(),
                          a["offsets"].cpu().numpy(), a["order"].cpu().numpy(),
                          a["codes"].cpu().numpy(),
                          vectors=a["base"].cpu().numpy() if case["pool"] else None,
                          rotation=None if a["rotation"] is None else a["rotation"].cpu().numpy())
    state["index"] = ix
    if kind == "search" and case["host"]:
        state["queries"] = q.cpu().numpy()
        return state
    state["queries"] = q.contiguous()
    state["ids"] = torch.empty((nq, k), dtype=torch.int64, device=DEV)
    state["dists"] = torch.empty((nq, k), dtype=torch.float32, device=DEV)
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "build":
        import vicinity_amd as v

        ix = v.IVFPQIndex(case["d"], num_clusters=case["nlist"], num_codebooks=case["M"],
                          codebook_size=case["K"], seed=42)
        ix.add_items(state["base"])
        ix.build(training_sample_size=min(case["sample"], case["n"]),
                 kmeans_max_iter=case["iters"])
        art = ix.export()
        return {name: art[name] for name in ("centroids", "codebooks", "list_offsets", "list_ids",
                                             "codes", "doc_ids", "vectors")}
    ix, q, k = state["index"], state["queries"], case["k"]
    if case["kind"] == "flat":
        return ix.search_device(q, k, state["ids"], state["dists"])
    pool = case["pool"] or None
    if case["host"] and case["nq"] == 1:
        return ix.search(q[0], k, rerank_pool=pool)
    if case["host"]:
        return ix.batch_search(q, k, rerank_pool=pool)
    return ix.search_batch_device(q, k, rerank_pool=pool, out_ids=state["ids"],
                                  out_dists=state["dists"])


def work(case):
    """Bytes: the arrays a pass reads (each once) and the rows it returns.
    Operations: the coarse products, the distance tables, one add per looked-up
    code of the probed entries; for a flat search the products; for a build the
    assignments of every k-means pass and the encoding."""
    n, d = case["n"], case["d"]
    if case["kind"] == "build":
        s = min(case["sample"], n)
        flops = 2 * d * (case["iters"] * s * (case["nlist"] + case["K"]) + n * (case["nlist"] + case["K"]))
        return dict(bytes=2 * n * d * 4 + n * case["M"] + 8 * n, flops=flops)
    nq, k = case["nq"], case["k"]
    io = nq * d * 4 + nq * k * 12
    if case["kind"] == "flat":
        return dict(bytes=n * d * 4 + io, flops=2 * n * d * nq)
    L, M, K, P = case["nlist"], case["M"], case["K"], min(case["nprobe"], case["nlist"])
    touched = min(1.0, nq * P / L)  # share of the lists that some query probes
    entries = nq * P * n / L
    code = M / 2 if K == 16 else M
    tables = nq * (P if case["opq"] or K == 16 else 1) * K * d * 2
    flops = 2 * nq * L * d + tables + entries * M + (2 * nq * P * d * d if case["opq"] else 0)
    bytes_ = L * d * 4 + M * K * (d // M) * 4 + touched * n * (code + 4) + io
    if case["pool"]:
        bytes_ += min(nq * max(case["pool"], k), n) * d * 4
        flops += 2 * nq * max(case["pool"], k) * d
    return dict(bytes=int(bytes_), flops=int(flops))


def tolerance(case):
    return "exact"


# ---- the same in 64 bits ----------------------------------------------------

def _pad(rows, k):
    if rows.shape[1] < k:
        fill = torch.full((rows.shape[0], k - rows.shape[1]), math.inf, dtype=rows.dtype, device=DEV)
        rows = torch.cat([rows, fill], 1)
    return rows


def _exact_flat(case, seed):
    base, q = _data(case, seed)
    if case["metric"] == "cosine":
        base, q = _unit(base), _unit(q)
    base, q = base.double(), q.double()
    bn = (base * base).sum(1)
    out = []
    step = max(1, (1 << 27) // case["n"])
    for s in range(0, case["nq"], step):
        qq = q[s:s + step]
        dots = qq @ base.T
        dist = 1.0 - dots if case["metric"] == "cosine" else (bn + (qq * qq).sum(1, keepdim=True)
                                                              - 2.0 * dots).clamp_min(0)
        out.append(dist.topk(min(case["k"], case["n"]), 1, largest=False, sorted=True).values)
    return None, _pad(torch.cat(out), case["k"])


def exact(case, seed):
    """(None for the ids, the distances in 64 bits); None for a build, whose
    arrays are the end of a chain of k-means passes, and for 4-bit codes,
    whose distances are of tables rounded to 8 bits by definition."""
    if case["kind"] == "flat":
        return _exact_flat(case, seed)
    if case["kind"] == "build" or case["K"] == 16:
        return None
    a = _artifacts(case, seed)
    nq, k, L, M = case["nq"], case["k"], case["nlist"], case["M"]
    P, kout = min(case["nprobe"], L), max(case["pool"], k)
    q = _unit(a["queries"].double())
    cent, books = a["centroids"].double(), a["codebooks"].double()
    probe = torch.cat([(q[s:s + 1024] @ cent.T).topk(P, 1).indices for s in range(0, nq, 1024)])
    off = a["offsets"].tolist()
    by_list = torch.sort(probe.reshape(-1), stable=True)
    starts = torch.searchsorted(by_list.values, torch.arange(L + 1, device=DEV)).tolist()
    dist = torch.full((nq, P * kout), math.inf, dtype=torch.float64, device=DEV)
    rows = torch.zeros((nq, P * kout), dtype=torch.int64, device=DEV)
    cols = torch.arange(kout, device=DEV)
    for l in range(L):
        pairs = by_list.indices[starts[l]:starts[l + 1]]
        ids = a["order"][off[l]:off[l + 1]]
        if not len(pairs) or not len(ids):
            continue
        r = q[pairs // P] - cent[l]
        if a["rotation"] is not None:
            r = r @ a["rotation"].double().T
        y = books[torch.arange(M, device=DEV), a["codes"][ids].long()].reshape(len(ids), -1)
        dd = (r * r).sum(1, keepdim=True) + (y * y).sum(1) - 2.0 * (r @ y.T)
        top = dd.topk(min(kout, len(ids)), 1, largest=False)
        at = (pairs // P).unsqueeze(1), (pairs % P * kout).unsqueeze(1) + cols[:top.values.shape[1]]
        dist[at] = top.values
        rows[at] = ids[top.indices]
    top = dist.topk(kout if P * kout >= kout else P * kout, 1, largest=False, sorted=True)
    if not case["pool"]:
        res = top.values[:, :k].clamp_min(0)
    else:
        res = []
        base = a["base"].double()
        for s in range(0, nq, 1024):
            ids = rows[s:s + 1024].gather(1, top.indices[s:s + 1024])
            dots = (base[ids] * q[s:s + 1024].unsqueeze(1)).sum(2)
            dots = torch.where(top.values[s:s + 1024].isfinite(), 1.0 - dots, math.inf)
            res.append(dots.sort(1).values[:, :k])
        res = torch.cat(res)
    if case["host"] and nq == 1:
        res = res[0][res[0].isfinite()]
        return None, res.cpu().numpy()
    return None, res.cpu().numpy() if case["host"] else res
