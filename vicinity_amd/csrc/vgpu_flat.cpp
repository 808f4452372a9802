// Flat exact index: database resident in HBM, batched top-k.
// Reference: brute force over l2_distance_squared / cosine_distance_normalized
// (src/distance.rs:78-109), as the reference's ground truth
// (src/ivf_pq/search.rs:3376-3392, tests/common/mod.rs:49-57).
#include <algorithm>
#include <cmath>

#include "vgpu_bounds.h"
#include "vgpu_runtime.h"

namespace vgpu {

// Flagged queries the ranking path's fallback takes with the count read on the device
constexpr size_t kFlatFallbackCap = 256;
// The others of one launch (their keys: at most 112 MiB)
constexpr int kFlatFallbackPass = 4096;

FlatIndex::FlatIndex(size_t dim, int met) : d(dim), metric(met) {
    if (dim == 0) throw Error(VGPU_ERR_INVALID_CONFIG, "dimension must be greater than 0");
    if (met != 0 && met != 1) throw Error(VGPU_ERR_INVALID_CONFIG, "metric must be 0 (L2) or 1 (1 - dot)");
    rowsum.assign(d, 0.0);
    VGPU_HIP(hipStreamCreate(&stream));
    for (auto& e : ev) VGPU_HIP(hipEventCreate(&e));
}

FlatIndex::~FlatIndex() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (auto& e : ev)
        if (e) (void)hipEventDestroy(e);
    if (stream) (void)hipStreamDestroy(stream);
}

void FlatIndex::add(const float* x, size_t count) {
    if (n + count >= 0xffffffffull) throw Error(VGPU_ERR_INVALID_PARAMETER, "more than 2^32-1 vectors");
    const size_t n0 = n;
    const double xmax0 = xmax2;
    const bool finite0 = finite;
    const std::vector<double> rowsum0 = rowsum;
    const double sqsum0 = sqsum;
    const size_t sampled0 = sampled;
    host.insert(host.end(), x, x + count * d);
    double sum = 0.0;
    for (size_t i = 0; i < count; i++) {
        double p[4] = {0.0, 0.0, 0.0, 0.0};  // four chains: one waits for each add
        const float* r = x + i * d;
        size_t j = 0;
        for (; j + 4 <= d; j += 4)
            for (int c = 0; c < 4; c++) p[c] += (double)r[j + c] * r[j + c];
        for (; j < d; j++) p[0] += (double)r[j] * r[j];
        const double t = (p[0] + p[1]) + (p[2] + p[3]);
        xmax2 = std::max(xmax2, t);
        sum += t;
    }
    for (size_t i = (16 - n0 % 16) % 16; d > 96 && i < count; i += 16, sampled++) {  // rank_bound_lost
        const float* r = x + i * d;
        double t = 0.0;
        for (size_t j = 0; j < d; j++) {
            rowsum[j] += r[j];
            t += (double)r[j] * r[j];
        }
        sqsum += t;
    }
    finite = finite && std::isfinite(sum);  // squares of floats: no overflow in double
    n += count;
    try {
        sync_device();
    } catch (...) {
        // A failed allocation has released the buffer it was growing: go
        // back to the previous rows and rebuild their device copy.
        host.resize(n0 * d);
        n = n0;
        xmax2 = xmax0;
        finite = finite0;
        rowsum = rowsum0;
        sqsum = sqsum0;
        sampled = sampled0;
        try {
            sync_device();
        } catch (...) {
            stale = true;
        }
        throw;
    }
}

void FlatIndex::sync_device() {
    stale = true;
    if (n) {
        d_x.upload(host.data(), n * d, stream);
        d_xnorm.reserve(n);
        launch_flat_norms(d_x.p, (int)n, (int)d, d_xnorm.p, stream);
        // the ranking path's copy, as large as the rows: only where a search can
        // use it, and without it the fp32 path serves every search
        if (flat_rank_ok((int)d, 1, finite && xmax2 < 1e30)) {
            try {
                d_xb.reserve(flat_pack_chunks((int)n, (int)d));
                launch_flat_pack(d_x.p, (int)n, (int)d, d_xb.p, stream);
            } catch (const Error& e) {
                if (e.code != VGPU_ERR_OUT_OF_MEMORY) throw;
            }
        } else {
            d_xb.release();
        }
        VGPU_HIP(hipGetLastError());
        VGPU_HIP(hipStreamSynchronize(stream));
    }
    stale = false;
}

// Whether the ranking path's bf16x3 bound is lost in the rows' common offset
// while the fp32 path's is not.  Distances are spread over about the rows'
// variance (dot products over the norm times a dimension's deviation); where
// the bound reaches half of that, a good part of the vectors are within it of
// the k-th and every query ends in the exhaustive fallback, in either path.
// 100k x 200 around unit centres plus 2, 2.5 and 3 in every dimension, k 10, 1000
// queries: fp32 5.3 ms each, ranking path 0.6, 10.5 and 10.6; plus 10, where both
// bounds are lost: 16.3 and 10.6.  Up to 96 dimensions the fallback is the
// cheaper one (100k x 32, k 40: fp32 8.2 ms, ranking path 2.6, all in fallback).
bool FlatIndex::rank_bound_lost() const {
    if (sampled == 0) return false;
    const double m = (double)sampled;
    double mean2 = 0.0;
    for (double x : rowsum) mean2 += (x / m) * (x / m);
    const double var = std::max(sqsum / m - mean2, 0.0), norm = std::sqrt(xmax2);
    const double spread = metric == 0 ? var : norm * std::sqrt(var / d);
    const float xn = (float)norm;
    const double fp32 = 4.0 * (d + 8.0) * 5.9604645e-08 * (metric == 0 ? 4.0 * xmax2 : 1.0 + xmax2);
    return flat_bf16_tau((int)d, metric, xn, xn, 0) > 0.5 * spread && fp32 < 0.5 * spread;
}

void FlatIndex::search_device(const float* d_q, size_t nq, size_t k, int64_t* d_ids, float* d_dists,
                              hipStream_t s) {
    if (!s) s = stream;
    if (stale)
        throw Error(VGPU_ERR_DEVICE, "the device copy of the flat index was lost in a failed add; add again");
    if (nq == 0 || k == 0) return;
    if (k > 112) throw Error(VGPU_ERR_INVALID_PARAMETER, "flat search supports k <= 112");
    if (n == 0) {
        launch_finalize(nullptr, nullptr, nullptr, (int)nq, 0, (int)k, d_ids, d_dists, s);
        VGPU_HIP(hipStreamSynchronize(s));
        return;
    }
    const bool rank = d_xb.n && flat_rank_ok((int)d, (int)k, finite && xmax2 < 1e30) &&
                      ((d <= 128 && k <= 32) || !rank_bound_lost());
    size_t step = rank && k > 32 ? std::min(nq, (size_t)flat_rank_chunk()) : nq;
    for (;;) {  // the largest buffer; the ranking path needs more of it per query
        try {
            w_partial.reserve(flat_partial_count((int)step, (int)n, (int)k, rank));
            break;
        } catch (const Error& e) {
            if (e.code != VGPU_ERR_OUT_OF_MEMORY || !rank || step <= 1024) throw;
            step = (step + 1) / 2;
        }
    }
    float gemm = 0.f, total = 0.f;
    unsigned int fb = 0;
    for (size_t q0 = 0; q0 < nq; q0 += step) {
        search_pass(d_q + q0 * d, std::min(step, nq - q0), k, rank, d_ids + q0 * k, d_dists + q0 * k, s);
        gemm += ms_gemm;
        total += ms_total;
        fb += fallbacks;
    }
    ms_gemm = gemm;
    ms_total = total;
    fallbacks = fb;
}

void FlatIndex::search_pass(const float* d_q, size_t nq, size_t k, bool rank, int64_t* d_ids, float* d_dists,
                            hipStream_t s) {
    const float xmax = (float)(std::sqrt(xmax2) * 1.0001 + 1e-30);
    w_qnorm.reserve(nq);
    w_partial.reserve(flat_partial_count((int)nq, (int)n, (int)k, rank));
    w_idx.reserve(nq * k);
    w_dist.reserve(nq * k);
    w_overflow.reserve(1);
    w_flag.reserve(nq);
    w_fb.reserve(nq);
    VGPU_HIP(hipMemsetAsync(w_overflow.p, 0, sizeof(unsigned int), s));
    // the bf16x3 ranking path computes the query norms in its merge
    const int rsl = rank ? flat_rank_fallback_slices((int)nq, (int)n, (int)k) : 0;
    if (!rsl) launch_flat_norms(d_q, (int)nq, (int)d, w_qnorm.p, s);
    VGPU_HIP(hipEventRecord(ev[0], s));
    launch_flat_search(d_q, rsl ? nullptr : w_qnorm.p, (int)nq, d_x.p, rank ? d_xb.p : nullptr, d_xnorm.p,
                       (int)n, (int)d, (int)k, metric, xmax, w_partial.p, w_idx.p, w_dist.p, w_overflow.p, w_flag.p,
                       w_fb.p, s, ev[3]);
    // the unproved queries (rare): exact scans over many workgroups.  The
    // ranking path runs the first kFlatFallbackCap of them with the count
    // read on the device (no host round trip), the rest after the final
    // wait; the other path reads the count first.
    const int cap = rsl ? (int)std::min<size_t>(nq, kFlatFallbackCap) : 0;
    if (rsl) {
        w_fbkeys.reserve((size_t)cap * rsl * k);
        launch_flat_rank_fallback_dev(w_flag.p, w_overflow.p, cap, w_fb.p, w_partial.p, (int)nq, (int)n, (int)d,
                                      (int)k, metric, d_q, d_x.p, w_fbkeys.p, w_idx.p, w_dist.p, s);
    } else {
        VGPU_HIP(hipMemcpyAsync(&fallbacks, w_overflow.p, sizeof(unsigned int), hipMemcpyDeviceToHost, s));
        VGPU_HIP(hipStreamSynchronize(s));
        if (fallbacks) {
            w_fbkeys.reserve((size_t)fallbacks * flat_fallback_slices((int)n, (int)k) * k);
            launch_flat_fallback(w_flag.p, (int)fallbacks, d_q, d_x.p, (int)n, (int)d, (int)k, metric,
                                 w_fbkeys.p, w_idx.p, w_dist.p, s);
        }
    }
    VGPU_HIP(hipEventRecord(ev[1], s));
    launch_finalize(w_idx.p, w_dist.p, nullptr, (int)nq, (int)k, (int)k, d_ids, d_dists, s);
    VGPU_HIP(hipEventRecord(ev[2], s));
    if (rsl) VGPU_HIP(hipMemcpyAsync(&fallbacks, w_overflow.p, sizeof(unsigned int), hipMemcpyDeviceToHost, s));
    VGPU_HIP(hipGetLastError());
    VGPU_HIP(hipStreamSynchronize(s));
    if (rsl && fallbacks > (unsigned int)cap) {  // more than the device-driven pass took
        const int all = (int)fallbacks;
        w_fbkeys.reserve((size_t)std::min(all - cap, kFlatFallbackPass) * rsl * k);
        for (int f0 = cap; f0 < all; f0 += kFlatFallbackPass)
            launch_flat_rank_fallback(w_flag.p + f0, std::min(all - f0, kFlatFallbackPass), w_fb.p, w_partial.p, (int)nq,
                                      (int)n, (int)d, (int)k, metric, d_q, d_x.p, w_fbkeys.p, w_idx.p, w_dist.p, s);
        launch_finalize(w_idx.p, w_dist.p, nullptr, (int)nq, (int)k, (int)k, d_ids, d_dists, s);
        VGPU_HIP(hipEventRecord(ev[2], s));
        VGPU_HIP(hipGetLastError());
        VGPU_HIP(hipStreamSynchronize(s));
    }
    VGPU_HIP(hipEventElapsedTime(&ms_gemm, ev[0], ev[3]));
    VGPU_HIP(hipEventElapsedTime(&ms_total, ev[0], ev[2]));
}

}  // namespace vgpu
