// Batched 8-bit scan by inverted list.
//
// The scan kernels of k_scan8_fast.hip take one query per workgroup and look
// every code up in that query's table.  In a large batch each list is probed
// by many queries (78 at 1M x 128, nlist 4096, nprobe 32, 10k queries), and
// the scores of one list against its queries are a matrix product: with the
// residual r = q - c (or its rotation) and the decoded codeword vector y,
//
//     |r - y|^2 = |r|^2 - 2 (r.y - |y|^2 / 2).
//
// So the batch is scored list by list on the matrix cores and the tables
// disappear:
//
//   list_count / list_plan / list_scatter   the (query, probe slot) pairs of
//       every list, and the work items (a list's segment x up to 64 of its
//       pairs) the score kernel's waves take in turn.
//   list_score_kernel<.., SAMPLE>   the first 16 TCAP entries of each query's
//       nearest lists: an upper bound of every entry's distance.  TCAP is 32 to
//       256 by the rule in vgpu_index.cpp: the longer the lists and the larger
//       k, the more entries the bound of a small sample leaves.
//   list_bound_kernel     the k-th smallest of those bounds, which bounds the
//       query's k-th distance from above.
//   list_score_kernel<.., !SAMPLE>  every pair: entries whose distance may be
//       within the bound are appended to the query's survivors.
//   list_final_kernel     per query: survivors that cannot be among the k
//       nearest are dropped, the rest rescored with the reference's
//       arithmetic (pq.rs:232-251, pq_simd.rs:349-355), ranked by (distance,
//       insertion index) and written.
//
// Scores are bf16x3 (r = rh + rl, y = yh + yl; rh.yh + rh.yl + rl.yh in
// float32, v_mfma_f32_16x16x32_bf16) and every comparison allows for their
// error bound list_tau, so the rescored set contains the reference's top k.
// A query with more survivors than its buffer holds, or more within the bound
// than are rescored, is flagged, like a FAST query whose proof fails:
// list_rescue_kernel, or for many of them the EXACT kernel, scores its entries
// with the reference's arithmetic.
//
// Bounds, at 10k queries: the score kernel is held by latency, of the decode's
// LDS gathers and of the work items' prologues, at two waves per SIMD (the
// operands of 64 pairs fill the registers).  126 us for 76M entries of 128
// dimensions: matrix cores 22% busy, VALU 30%, LDS 20% (half of it bank
// conflicts), waves waiting 45% of their time; 390 us for 390M of 96, 166 us for
// 370M of 25.  The final kernel is held by its codeword loads (109 us for 102
// rescored entries per query, 16 codebooks of 8: L1 64% of its cycles, VALU 54%,
// waves waiting 65%).  The whole scan against the kernels it replaces, traced: 1M
// x 128 331 -> 317 us (FAST scan and its tables), 10M x 96 3400 -> 726, 1.2M x 25
// 2520 -> 292, OPQ 500k x 128 (5k queries) 833 -> 199.
//
// MFMA layout (wave64): lane l holds row / column l % 16 and the eight
// dimensions 8 (l / 16) .. + 7 of a 32-dimension step, for A (entries) and B
// (queries); result element i of lane l is entry 4 (l / 16) + i of query
// l % 16.  A lane's compare threshold is therefore one register per query
// tile, and the float32 start value -|y|^2 / 2 of an accumulator comes from
// four consecutive floats.
#include "vgpu_device.h"
#include "vgpu_bounds.h"
#include "vgpu_launch.h"

namespace vgpu {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

#define SL_NT 4                     // query tiles (16 pairs each) per work item
#define SL_PAIRS (16 * SL_NT)
#define SL_WAVES 8
#define SL_THREADS (64 * SL_WAVES)
#define SL_STAGE 320                // survivors a wave stages in LDS before it flushes
#define SL_MAXSEG 16                // segments per list, at most

// Padded shape of the score product: dsp dimensions per codebook in the MFMA
// operands (1, 2, 4 or 8; wider subvectors are cut into several virtual
// codebooks of 8 that share a code), zero beyond the real ones.
ListShape list_shape(int d, int M, int K, int ds) {
    ListShape s;
    s.dsp = ds <= 2 ? ds : ds <= 4 ? 4 : 8;
    s.parts = (ds + 7) / 8;
    s.Mv = M * s.parts;
    const int dp = s.Mv * s.dsp;
    s.KT = (dp + 31) / 32;
    s.LW = (s.KT * (8 / s.dsp) + 3) / 4;
    s.contig = s.parts * s.dsp == ds && (d & 3) == 0;
    s.table_bytes = (size_t)s.KT * 32 / s.dsp * K * s.dsp * 4;
    // the table and the staging buffers share the CU's 160 KiB of LDS, and
    // KT 4 already fills the registers with 64 pairs of operands
    s.ok = K != 16 && s.KT <= 4 && s.table_bytes <= (size_t)128 * 1024;
    return s;
}

// ---- index arrays ---------------------------------------------------------

// lcodes: tile T (16 entries of one list), lane l, LW words: the code bytes
// of the eight padded dimensions of entry l % 16, group l / 16, step by step.
// lbias: -|y|^2 / 2 per entry, -inf past the end of the list.
__global__ __launch_bounds__(256) void list_tiles_kernel(DevIndex ix, const double* __restrict__ cwn, ListShape sh,
                                                         uint32_t* __restrict__ lcodes, float* __restrict__ lbias) {
    const int l = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t o0 = ix.offsets[l], len = ix.offsets[l + 1] - o0;
    const uint32_t t0 = ix.ltoff[l], nt = ix.ltoff[l + 1] - t0;
    const int e = lane & 15, kg = lane >> 4, nb = 8 / sh.dsp;
    for (uint32_t t = wave; t < nt; t += 4) {
        const uint32_t j = t * 16 + e;
        const bool ok = j < len;
        const uint8_t* row = ix.codes + (size_t)(o0 + (ok ? j : 0u)) * ix.M;
        uint32_t* out = lcodes + ((size_t)(t0 + t) * 64 + lane) * sh.LW;
        for (int w = 0; w < sh.LW; w++) {
            uint32_t v = 0;
            for (int b = 0; b < 4; b++) {
                const int x = 4 * w + b;  // byte x: step x / nb, codeword x % nb of the group
                const int kt = x / nb, mv = (32 * kt + 8 * kg) / sh.dsp + x % nb;
                if (ok && kt < sh.KT && mv < sh.Mv) v |= (uint32_t)row[mv / sh.parts] << (8 * b);
            }
            out[w] = v;
        }
        if (kg == 0) {
            double s = 0.0;
            if (ok)
                for (int m = 0; m < ix.M; m++) s += cwn[(size_t)m * ix.K + row[m]];
            lbias[(size_t)(t0 + t) * 16 + e] = ok ? (float)(-0.5 * s) : -__int_as_float(0x7f800000);
        }
    }
}

void launch_list_tiles(const DevIndex& ix, const double* cwn, const ListShape& sh, uint32_t* lcodes, float* lbias,
                       hipStream_t s) {
    if (ix.L <= 0) return;
    hipLaunchKernelGGL(list_tiles_kernel, dim3(ix.L), dim3(256), 0, s, ix, cwn, sh, lcodes, lbias);
}

// ---- pairs and work items -------------------------------------------------

// A workgroup counts the pairs of qw queries (one wave per query in turn):
// the LDS count before a pair is its place among the workgroup's pairs of its
// list (low half: every pair; high half: the sample pairs, those with fewer
// than tcap tiles of nearer lists before them).  Counting in LDS first leaves
// no atomic on global memory: with one per pair on the lists' counters the
// kernel took 33 us (4096 lists) to 81 us (1024 lists) for 320,000 pairs.
__global__ __launch_bounds__(1024) void list_count_kernel(DevIndex ix, ScanArgs a, ListWs w) {
    extern __shared__ __align__(16) char smem[];
    uint32_t* hist = reinterpret_cast<uint32_t*>(smem);  // [L]
    const int tid = threadIdx.x, lane = tid & 63;
    if (blockIdx.x == 0)  // heads, then rescued: first used by the kernels that follow
        for (int i = tid; i < 4 + SL_RESCUE_MAX; i += 1024) w.heads[i] = 0u;
    for (int l = tid; l < ix.L; l += 1024) hist[l] = 0u;
    __syncthreads();
    const int q0 = blockIdx.x * w.qw, q1 = min(q0 + w.qw, a.nq);
    for (int q = q0 + (tid >> 6); q < q1; q += 16) {
        const uint32_t* pr = a.probe + (size_t)q * a.P;
        uint32_t tiles0 = 0, entries = 0;
        for (int s0 = 0; s0 < a.P; s0 += 64) {
            const int s = s0 + lane;
            const uint32_t l = s < a.P ? pr[s] : 0u;
            // no such list: scanned as empty
            const uint32_t len = s < a.P && l < (uint32_t)ix.L ? ix.offsets[l + 1] - ix.offsets[l] : 0u;
            const uint32_t nt = (len + 15) >> 4;
            uint32_t inc = nt;
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t x = __shfl_up(inc, o, 64);
                if (lane >= o) inc += x;
            }
            const uint32_t tb = tiles0 + inc - nt;
            if (nt) {
                const size_t p = (size_t)q * a.P + s;
                w.pos[p] = atomicAdd(&hist[l], tb < (uint32_t)w.tcap ? 0x10001u : 1u);
                w.tbase[p] = tb;
            }
            entries += len;
            tiles0 += __shfl(inc, 63, 64);
        }
        for (int o = 32; o > 0; o >>= 1) entries += __shfl_xor(entries, o, 64);
        if (w.padded)
            for (int j = lane; j < w.ld; j += 64) {
                const int x = w.dimmap[j];
                w.padded[(size_t)q * w.ld + j] = x < 0 ? 0.0f : a.qn[(size_t)q * ix.d + x];
            }
        if (lane == 0) {
            a.qstat[(size_t)q * QSTAT_WORDS] = entries;
            w.ntiles[q] = min(tiles0, (uint32_t)w.tcap);
            w.scount[q] = 0u;
        }
    }
    __syncthreads();
    uint32_t* out = w.cnt + (size_t)blockIdx.x * ix.L;
    for (int l = tid; l < ix.L; l += 1024) out[l] = hist[l];
}

// Segments of a list of nt tiles: seg tiles each, at most SL_MAXSEG.
__device__ __forceinline__ uint32_t sl_segs(uint32_t nt, uint32_t seg) {
    return min((nt + seg - 1) / seg, (uint32_t)SL_MAXSEG);
}

// 256 lists per workgroup, four threads each (a quarter of the counting
// workgroups' rows): room for every list's pairs and work items, and the
// first pair of every counting workgroup.  One reservation per workgroup (the
// order of lists does not matter): atomics on one address take about 13 ns
// each here.  An item is (list, first pair, pairs, segment | segments << 8).
__global__ __launch_bounds__(1024) void list_plan_kernel(DevIndex ix, ListWs w) {
    __shared__ uint32_t part[2][4][256];
    __shared__ uint32_t wsum[4][4], base[4];
    const int tid = threadIdx.x, li = tid & 255, quarter = tid >> 8, lane = tid & 63, wave = (tid >> 6) & 3;
    const int l = blockIdx.x * 256 + li;
    const bool in = l < ix.L;
    const uint32_t nt = in ? ix.ltoff[l + 1] - ix.ltoff[l] : 0u;
    const int b0 = quarter * w.nwg / 4, b1 = (quarter + 1) * w.nwg / 4;
    uint32_t p[2] = {0u, 0u};  // 0: sample, 1: every pair
    if (in) {
#pragma unroll 8
        for (int b = b0; b < b1; b++) {
            const uint32_t x = w.cnt[(size_t)b * ix.L + l];
            p[0] += x >> 16;
            p[1] += x & 0xffffu;
        }
    }
    part[0][quarter][li] = p[0];
    part[1][quarter][li] = p[1];
    __syncthreads();
    uint32_t before[2], c[2], nb[2], ns[2], v[4], inc[4];
#pragma unroll
    for (int ph = 0; ph < 2; ph++) {
        before[ph] = c[ph] = 0u;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            if (g == quarter) before[ph] = c[ph];
            c[ph] += part[ph][g][li];
        }
        nb[ph] = (c[ph] + (uint32_t)w.ipairs - 1u) / (uint32_t)w.ipairs;
        ns[ph] = sl_segs(ph ? nt : min(nt, (uint32_t)w.tcap), (uint32_t)w.seg);
        v[2 * ph] = c[ph];
        v[2 * ph + 1] = nb[ph] * ns[ph];
    }
    // prefix sums over the workgroup's lists (every quarter computes the same)
#pragma unroll
    for (int i = 0; i < 4; i++) {
        inc[i] = v[i];
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t x = __shfl_up(inc[i], o, 64);
            if (lane >= o) inc[i] += x;
        }
        if (quarter == 0 && lane == 63) wsum[i][wave] = inc[i];
    }
    __syncthreads();
    if (tid < 4) base[tid] = atomicAdd(&w.heads[tid], wsum[tid][0] + wsum[tid][1] + wsum[tid][2] + wsum[tid][3]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t o = base[i];
        for (int g = 0; g < wave; g++) o += wsum[i][g];
        inc[i] = o + inc[i] - v[i];  // now the list's first pair / item
    }
    if (!in) return;
#pragma unroll
    for (int ph = 0; ph < 2; ph++) {
        uint4* items = ph ? w.items : w.items1;
        // pairs spread evenly over the blocks, in whole tiles
        const uint32_t per = nb[ph] ? ((c[ph] + nb[ph] - 1) / nb[ph] + 15) / 16 * 16 : 0u;
        for (uint32_t b = quarter; b < nb[ph]; b += 4) {
            const uint32_t p0 = min(b * per, c[ph]), np = min(per, c[ph] - p0);
            for (uint32_t sg = 0; sg < ns[ph]; sg++)
                items[inc[2 * ph + 1] + b * ns[ph] + sg] =
                    make_uint4((uint32_t)l, inc[2 * ph] + p0, np, sg | ns[ph] << 8);
        }
    }
    uint32_t f0 = inc[0] + before[0], f1 = inc[2] + before[1];
#pragma unroll 8
    for (int b = b0; b < b1; b++) {
        const size_t o = (size_t)b * ix.L + l;
        const uint32_t x = w.cnt[o];
        w.first1[o] = f0;
        w.first[o] = f1;
        f0 += x >> 16;
        f1 += x & 0xffffu;
    }
}

// Pair word: query << SL_SLOT_BITS | probe slot.
__global__ __launch_bounds__(256) void list_scatter_kernel(DevIndex ix, ScanArgs a, ListWs w) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= (uint32_t)a.nq * (uint32_t)a.P) return;
    const uint32_t q = i / (uint32_t)a.P, s = i % (uint32_t)a.P;
    const uint32_t l = a.probe[i];
    if (l >= (uint32_t)ix.L || ix.offsets[l + 1] == ix.offsets[l]) return;
    const uint32_t word = q << SL_SLOT_BITS | s, pos = w.pos[i];
    const size_t o = (size_t)(q / (uint32_t)w.qw) * ix.L + l;
    w.pairs[w.first[o] + (pos & 0xffffu)] = word;
    if (w.tbase[i] < (uint32_t)w.tcap) w.pairs1[w.first1[o] + (pos >> 16)] = word;
}

// ---- scores ---------------------------------------------------------------

__device__ __forceinline__ uint32_t sl_pack(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 v = {(__bf16)a, (__bf16)b};  // round to nearest even
    return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ void sl_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A raw buffer over n bytes: loads past them give 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sl_rsrc(const void* p, uint32_t n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)n, 0x00020000);
}
#define SL_PAST 0xfffffff0u  // an offset past every buffer

// A wave's LDS: staged survivors, their per-pair counts and reservations, and
// the item's pairs.
struct SlWave {
    uint2 stage[SL_STAGE];      // (score bits, entry | pair << 26)
    uint32_t cnt[SL_PAIRS];
    uint32_t base[SL_PAIRS];
    uint32_t pair[SL_PAIRS];    // pair words
    float t0[SL_PAIRS];         // |r|^2
};

// Decode one tile's A operands: lane (e, kg) gathers the eight padded
// dimensions of entry e, group kg from the codeword table in LDS: per
// codeword the bf16 high halves, then the low halves; for 8 dimensions two
// tables (16-byte halves 32 bytes apart would leave half the LDS banks idle).
template <int KT, int DSP, int LW>
__device__ __forceinline__ void sl_decode(const char* tab, uint32_t lbase, uint32_t kbytes, uint32_t lotab,
                                          const uint32_t (&cw)[LW], u32x4 (&ah)[KT], u32x4 (&al)[KT]) {
    constexpr int NB = 8 / DSP, CB = DSP == 8 ? 16 : DSP * 4;  // codewords per lane and step, bytes per codeword
#pragma unroll
    for (int kt = 0; kt < KT; kt++) {
        uint32_t h[4], l[4];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int x = kt * NB + b;
            const uint32_t code = (cw[x >> 2] >> (8 * (x & 3))) & 0xffu;
            // kbytes: bytes of one codebook; lbase holds the group's first
            const char* p = tab + lbase + (uint32_t)((32 * kt) / DSP + b) * kbytes + code * CB;
            if constexpr (DSP == 8) {
                const u32x4 H = *reinterpret_cast<const u32x4*>(p), Lw = *reinterpret_cast<const u32x4*>(p + lotab);
                h[0] = H.x; h[1] = H.y; h[2] = H.z; h[3] = H.w;
                l[0] = Lw.x; l[1] = Lw.y; l[2] = Lw.z; l[3] = Lw.w;
            } else if constexpr (DSP == 4) {
                const u32x4 W = *reinterpret_cast<const u32x4*>(p);
                h[2 * b] = W.x; h[2 * b + 1] = W.y;
                l[2 * b] = W.z; l[2 * b + 1] = W.w;
            } else if constexpr (DSP == 2) {
                const u32x2 W = *reinterpret_cast<const u32x2*>(p);
                h[b] = W.x;
                l[b] = W.y;
            } else {
                const uint32_t W = *reinterpret_cast<const uint32_t*>(p);  // high half | low half << 16
                if (b & 1) {
                    const uint32_t W0 = h[b >> 1];
                    h[b >> 1] = __builtin_amdgcn_perm(W, W0, 0x05040100u);
                    l[b >> 1] = __builtin_amdgcn_perm(W, W0, 0x07060302u);
                } else {
                    h[b >> 1] = W;
                }
            }
        }
        ah[kt] = u32x4{h[0], h[1], h[2], h[3]};
        al[kt] = u32x4{l[0], l[1], l[2], l[3]};
    }
}

// One survivor at place `to` of its query's buffer.
__device__ __forceinline__ void sl_write(const SlWave& sw, const ListWs& w, uint2 st, uint32_t to) {
    const uint32_t p = st.y >> 26, word = sw.pair[p];
    const float d = fmaf(-2.0f, __uint_as_float(st.x), sw.t0[p]);
    if (to < (uint32_t)w.cap)
        w.surv[(size_t)(word >> SL_SLOT_BITS) * w.cap + to] = make_uint2(
            (word & ((1u << SL_SLOT_BITS) - 1u)) << w.tbits | (st.y & 0x3ffffffu), __float_as_uint(d));
}

// Write the staged survivors to their queries' buffers: one reservation per
// pair with any (lane p reserves for pair p), then every entry at its place.
__device__ __forceinline__ void sl_flush(SlWave& sw, const ListWs& w, uint32_t& ns) {
    const int lane = threadIdx.x & 63;
    sl_wave_sync();
    sw.cnt[lane] = 0u;
    sl_wave_sync();
    uint32_t at[SL_STAGE / 64];
    uint2 st[SL_STAGE / 64];
#pragma unroll
    for (int i = 0; i < SL_STAGE / 64; i++) {
        const uint32_t x = i * 64 + lane;
        if (x < ns) {
            st[i] = sw.stage[x];
            at[i] = atomicAdd(&sw.cnt[st[i].y >> 26], 1u);
        }
    }
    sl_wave_sync();
    const uint32_t c = sw.cnt[lane];
    if (c) sw.base[lane] = atomicAdd(&w.scount[sw.pair[lane] >> SL_SLOT_BITS], c);
    sl_wave_sync();
#pragma unroll
    for (int i = 0; i < SL_STAGE / 64; i++) {
        const uint32_t x = i * 64 + lane;
        if (x < ns) sl_write(sw, w, st[i], sw.base[st[i].y >> 26] + at[i]);
    }
    ns = 0;
    sl_wave_sync();
}

// A work item: list, pairs, entry tiles, and its pair words (lane i: pair i).
struct SlItem {
    uint32_t l, p0, np, tile0, tile1, word;
};

// One work item with NT query tiles.
template <int KT, int DSP, int LW, int NT, bool SAMPLE>
__device__ __forceinline__ void sl_item(const DevIndex& ix, const ScanArgs& a, const ListWs& w, const char* tab,
                                        SlWave& sw, const SlItem& im) {
    const int lane = threadIdx.x & 63, col = lane & 15, kg = lane >> 4;
    const uint32_t tb0 = ix.ltoff[im.l];
    const __amdgpu_buffer_rsrc_t rlc = sl_rsrc(ix.lcodes, ix.ltiles * (256u * LW));
    const __amdgpu_buffer_rsrc_t rlb = sl_rsrc(ix.lbias, ix.ltiles * 64u);
    // codes and start values two tiles ahead (set S: tile tile0 + S, + 2, ..)
    uint32_t cw[2][LW];
    floatx4 bias[2];
    auto fetch = [&](const int S, uint32_t t) {
        t = min(t, im.tile1 - 1);  // past the item: any of its tiles, never used
        const uint32_t so = (tb0 + t) * (256u * LW), vo = (uint32_t)lane * (4u * LW);
        if constexpr (LW % 4 == 0) {
#pragma unroll
            for (int i = 0; i < LW / 4; i++) {
                const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(rlc, vo + 16 * i, so, 0);
                cw[S][4 * i] = x.x;
                cw[S][4 * i + 1] = x.y;
                cw[S][4 * i + 2] = x.z;
                cw[S][4 * i + 3] = x.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < LW; i++) cw[S][i] = __builtin_amdgcn_raw_buffer_load_b32(rlc, vo + 4 * i, so, 0);
        }
        bias[S] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rlb, 16u * kg, (tb0 + t) * 64u, 0));
    };
    fetch(0, im.tile0);
    fetch(1, im.tile0 + 1);
    // nearest lists first: entries within the bound gather in the first tiles
    uint32_t kw[1] = {(uint32_t)lane < im.np ? im.word << (32 - SL_SLOT_BITS) | im.word >> SL_SLOT_BITS : 0xffffffffu};
    if (!SAMPLE) wave_sort_u32<1>(kw);
    const uint32_t myword = kw[0] >> (32 - SL_SLOT_BITS) | kw[0] << SL_SLOT_BITS;
    // B operands: r of pair col of every tile, |r|^2 and the compare threshold.
    // The rows come through buffer resources (dimensions past a row read as
    // 0), two tiles' loads in flight.
    u32x4 bh[NT][KT], bl[NT][KT];
    float T[NT], t0v[NT];
    uint32_t gq[NT], tlim[NT];  // SAMPLE: the pair's bound row, and its tiles to write
    const uint32_t ld = (uint32_t)w.ld;
    const __amdgpu_buffer_rsrc_t rc = sl_rsrc(w.cent + (size_t)im.l * ld, a.rres ? 0u : ld * 4u);
    const __amdgpu_buffer_rsrc_t rq =
        a.rres ? sl_rsrc(a.rres, (uint32_t)a.nq * a.P * ld * 4u) : sl_rsrc(w.rows, (uint32_t)a.nq * ld * 4u);
    u32x4 craw[KT][2], qraw[2][KT][2];
    float Bv[2];
    uint32_t tbv[2];
#pragma unroll
    for (int kt = 0; kt < KT; kt++)
#pragma unroll
        for (int h = 0; h < 2; h++)
            craw[kt][h] = __builtin_amdgcn_raw_buffer_load_b128(rc, 4u * (32 * kt + 8 * kg + 4 * h), 0, 0);
    auto pair_word = [&](const int t) {
        const uint32_t pi = t * 16 + col;
        return (uint32_t)__shfl((int)myword, (int)(pi < im.np ? pi : 0u), 64);
    };
    auto load_rows = [&](const int S, const int t) {
        const uint32_t word = pair_word(t), q = word >> SL_SLOT_BITS;
        const uint32_t pair = q * (uint32_t)a.P + (word & ((1u << SL_SLOT_BITS) - 1u));
        if (SAMPLE) tbv[S] = w.tbase[pair];
        else Bv[S] = w.bound[q];
        const uint32_t row = (a.rres ? pair : q) * ld * 4u;
#pragma unroll
        for (int kt = 0; kt < KT; kt++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t j = (uint32_t)(32 * kt + 8 * kg + 4 * h);
                qraw[S][kt][h] = __builtin_amdgcn_raw_buffer_load_b128(rq, j < ld ? row + 4 * j : SL_PAST, 0, 0);
            }
    };
    load_rows(0, 0);
    if (NT > 1) load_rows(1, 1);
#pragma unroll
    for (int t = 0; t < NT; t++) {
        __builtin_amdgcn_sched_barrier(0);
        const int S = t & 1;
        const uint32_t pi = t * 16 + col;
        const bool ok = pi < im.np;
        const uint32_t word = pair_word(t);
        const uint32_t q = word >> SL_SLOT_BITS, slot = word & ((1u << SL_SLOT_BITS) - 1u);
        float s = 0.0f;
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            uint32_t h[4], lo[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const u32x4 x = qraw[S][kt][e >> 1], c = craw[kt][e >> 1];
                const float r0 = __uint_as_float(x[2 * (e & 1)]) - __uint_as_float(c[2 * (e & 1)]);
                const float r1 = __uint_as_float(x[2 * (e & 1) + 1]) - __uint_as_float(c[2 * (e & 1) + 1]);
                h[e] = sl_pack(r0, r1);
                lo[e] = sl_pack(r0 - __uint_as_float(h[e] << 16), r1 - __uint_as_float(h[e] & 0xffff0000u));
                s = fmaf(r0, r0, s);
                s = fmaf(r1, r1, s);
            }
            bh[t][kt] = u32x4{h[0], h[1], h[2], h[3]};
            bl[t][kt] = u32x4{lo[0], lo[1], lo[2], lo[3]};
        }
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        const float tau = list_tau(32 * KT, ix.M, ix.ds, s, ix.rmax);
        t0v[t] = s + (SAMPLE ? tau : 0.0f);
        if (SAMPLE) {
            gq[t] = q * (uint32_t)(16 * w.tcap) + 16u * tbv[S];
            tlim[t] = ok ? (uint32_t)w.tcap - tbv[S] : 0u;
        } else {
            // a = t0 - 2 D may be within the bound: a - tau <= B, with room
            // for the rounding of this line
            const float B = Bv[S];
            T[t] = ok ? fmaxf(0.5f * (s - tau - B) - 1e-6f * (s + fabsf(B)), -3.0e38f) : 3.0e38f;
            if (kg == 0) {
                sw.pair[pi] = word;
                sw.t0[pi] = s;
                if (ok) w.t0[q * (uint32_t)a.P + slot] = s;
            }
        }
        if (t + 2 < NT) load_rows(S, t + 2);
    }
    sl_wave_sync();
    const uint32_t kbytes = (uint32_t)ix.K * (DSP == 8 ? 16 : DSP * 4), lbase = (uint32_t)kg * (8 / DSP) * kbytes;
    uint32_t ns = 0;
    // the next tile's operands are decoded before this tile's products where
    // the registers hold both
    constexpr bool DB = KT * NT <= 12;
    u32x4 ah[DB ? 2 : 1][KT], al[DB ? 2 : 1][KT];
    floatx4 b0[DB ? 2 : 1];
    auto load = [&](const int S, const int O, uint32_t t) {  // operands O of tile t from set S
        sl_decode<KT, DSP, LW>(tab, lbase, kbytes, w.sh.table_bytes / 2, cw[S], ah[O], al[O]);
        b0[O] = bias[S];
        fetch(S, t + 2);
    };
    if (DB) load(0, 0, im.tile0);
    auto step = [&](const int C, uint32_t t) {  // C: tile's code set
        if (DB) load(C ^ 1, C ^ 1, t + 1);
        else load(C, 0, t);
        const int S = DB ? C : 0;
        floatx4 acc[NT];
#pragma unroll
        for (int i = 0; i < NT; i++) acc[i] = b0[S];
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            const bf16x8 xh = __builtin_bit_cast(bf16x8, ah[S][kt]), xl = __builtin_bit_cast(bf16x8, al[S][kt]);
#pragma unroll
            for (int i = 0; i < NT; i++)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, __builtin_bit_cast(bf16x8, bl[i][kt]), acc[i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < NT; i++)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xl, __builtin_bit_cast(bf16x8, bh[i][kt]), acc[i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < NT; i++)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, __builtin_bit_cast(bf16x8, bh[i][kt]), acc[i], 0, 0, 0);
        }
        if constexpr (SAMPLE) {
#pragma unroll
            for (int i = 0; i < NT; i++)
                if (t < tlim[i]) {
                    floatx4 v;
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = fmaf(-2.0f, acc[i][e], t0v[i]);
                    *reinterpret_cast<floatx4*>(w.gbound + gq[i] + 16 * t + 4 * kg) = v;
                }
        } else {
            uint64_t m[NT][4], any = 0;  // entries that may be within the bound
#pragma unroll
            for (int i = 0; i < NT; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    m[i][e] = __ballot(acc[i][e] >= T[i]);
                    any |= m[i][e];
                }
            if (any) {
#pragma unroll
                for (int i = 0; i < NT; i++) {
                    if (!(m[i][0] | m[i][1] | m[i][2] | m[i][3])) continue;
                    if (ns > SL_STAGE - 256) sl_flush(sw, w, ns);
                    const uint32_t lb0 = (t * 16 + 4 * kg) | (uint32_t)(i * 16 + col) << 26;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint64_t b = m[i][e];
                        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32),
                                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
                        if (acc[i][e] >= T[i]) sw.stage[ns + below] = make_uint2(__float_as_uint(acc[i][e]), lb0 + e);
                        ns += (uint32_t)__popcll(b);
                    }
                }
            }
        }
    };
    for (uint32_t t = im.tile0; t < im.tile1; t += 2) {
        step(0, t);
        if (t + 1 < im.tile1) step(1, t + 1);
    }
    if (!SAMPLE && ns) sl_flush(sw, w, ns);
}

// Persistent: workgroup b takes the work items b, b + gridDim.x, ..; its
// waves share them through a counter in LDS (one counter in global memory
// for every wave of the chip cost more than the scores: 16,000 atomics on one
// address are 210 us).  The next item's descriptor and pair words are fetched
// while an item runs.  LDS: the codeword table, then one SlWave per wave.
template <int KT, int DSP, bool SAMPLE>
__global__ __launch_bounds__(SL_THREADS, KT == 1 ? 4 : 2) void list_score_kernel(DevIndex ix, ScanArgs a, ListWs w) {
    extern __shared__ __align__(16) char smem[];
    __shared__ uint32_t head;
    constexpr int LW = (KT * (8 / DSP) + 3) / 4;
    const uint32_t tbytes = (uint32_t)w.sh.table_bytes;
    const uint32_t nitems = w.heads[SAMPLE ? 1 : 3];
    const uint4* items = SAMPLE ? w.items1 : w.items;
    const uint32_t* pairs = SAMPLE ? w.pairs1 : w.pairs;
    const int lane = threadIdx.x & 63;
    if (blockIdx.x >= nitems) return;
    if (threadIdx.x == 0) head = SL_WAVES;
    uint32_t it = blockIdx.x + gridDim.x * (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint4 dn = make_uint4(0u, 0u, 1u, 0u);
    uint32_t wn = 0;
    if (it < nitems) {
        dn = items[it];
        wn = pairs[dn.y + min((uint32_t)lane, dn.z - 1u)];
    }
    for (uint32_t o = threadIdx.x * 16; o < tbytes; o += SL_THREADS * 16)
        *reinterpret_cast<u32x4*>(smem + o) = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(ix.ltable) + o);
    __syncthreads();
    SlWave& sw = reinterpret_cast<SlWave*>(smem + tbytes)[threadIdx.x >> 6];
    while (it < nitems) {
        SlItem im;
        im.l = __builtin_amdgcn_readfirstlane(dn.x);
        im.p0 = __builtin_amdgcn_readfirstlane(dn.y);
        im.np = __builtin_amdgcn_readfirstlane(dn.z);
        const uint32_t sg = __builtin_amdgcn_readfirstlane(dn.w);
        im.word = wn;
        uint32_t nx = 0;
        if (lane == 0) nx = atomicAdd(&head, 1u);
        it = blockIdx.x + gridDim.x * (uint32_t)__builtin_amdgcn_readfirstlane(nx);
        if (it < nitems) {
            dn = items[it];
            wn = pairs[dn.y + min((uint32_t)lane, dn.z - 1u)];
        }
        uint32_t nt = ix.ltoff[im.l + 1] - ix.ltoff[im.l];
        if (SAMPLE) nt = min(nt, (uint32_t)w.tcap);
        const uint32_t s0 = sg & 255u, nseg = sg >> 8;
        const uint32_t per = (nt + nseg - 1) / nseg;
        im.tile0 = min(s0 * per, nt);
        im.tile1 = min(im.tile0 + per, nt);
        if (im.tile0 < im.tile1) {
            switch ((im.np + 15) >> 4) {
                case 1: sl_item<KT, DSP, LW, 1, SAMPLE>(ix, a, w, smem, sw, im); break;
                case 2: sl_item<KT, DSP, LW, 2, SAMPLE>(ix, a, w, smem, sw, im); break;
                case 3: sl_item<KT, DSP, LW, 3, SAMPLE>(ix, a, w, smem, sw, im); break;
                default: sl_item<KT, DSP, LW, 4, SAMPLE>(ix, a, w, smem, sw, im); break;
            }
        }
    }
}

// ---- bound ----------------------------------------------------------------

// One wave per query: an upper bound of the k-th smallest of its sample
// bounds (+inf when there are fewer than k): the smallest value of the
// leading 20 bits (11 of the mantissa) that k keys are not above, found bit by
// bit over ballot counts below the keys' common leading bits.
template <int E>
__global__ __launch_bounds__(256) void list_bound_kernel(ScanArgs a, ListWs w) {
    const int q = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (q >= a.nq) return;
    const uint32_t n4 = 4 * w.ntiles[q];  // groups of four
    const float4* g = reinterpret_cast<const float4*>(w.gbound + (size_t)q * (16 * w.tcap));
    uint32_t key[E][4], lo = 0xffffffffu, hi = 0u;
#pragma unroll
    for (int e = 0; e < E; e++) {
        const uint32_t i = e * 64 + lane;
        const float inf = __int_as_float(0x7f800000);
        const float4 v = i < n4 ? g[i] : make_float4(inf, inf, inf, inf);
        key[e][0] = fkey(v.x);
        key[e][1] = fkey(v.y);
        key[e][2] = fkey(v.z);
        key[e][3] = fkey(v.w);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            lo = min(lo, key[e][j]);
            if (key[e][j] < fkey(3.0e38f)) hi = max(hi, key[e][j]);  // padding entries are +inf
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 64));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, o, 64));
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    auto below = [&](uint32_t c) {
        uint32_t b = 0;
#pragma unroll
        for (int e = 0; e < E; e++) {
#pragma unroll
            for (int j = 0; j < 4; j++) b += (uint32_t)__popcll(__ballot(key[e][j] < c));
        }
        return b;
    };
    float B = __int_as_float(0x7f800000);
    if (hi >= lo && hi != 0u && below(hi) + 1u >= (uint32_t)a.kout) {
        int b = lo == hi ? 11 : 31 - __clz((int)(lo ^ hi));
        uint32_t ans = b >= 31 ? 0u : hi >> (b + 1) << (b + 1);
        for (; b >= 12; b--) {
            const uint32_t c = ans | 1u << b;
            if (below(c) < (uint32_t)a.kout) ans = c;
        }
        B = fkey_to_float(min(ans | 0xfffu, hi));
    }
    if (lane == 0) w.bound[q] = B;
}

// ---- final ----------------------------------------------------------------

// One codebook's part of the reference's distance: sum of (r_j - cw_j)^2 in
// index order, every step rounded (pq.rs:232-251).
template <int DS>
__device__ __forceinline__ float sl_sub(const float* q, const float* __restrict__ c, const float* __restrict__ cw,
                                        int ds, bool resid) {
    float e = 0.0f;
    if constexpr (DS == 8 || DS == 4) {
        float4 x[DS / 4], y[DS / 4], z[DS / 4];
#pragma unroll
        for (int i = 0; i < DS / 4; i++) {
            y[i] = reinterpret_cast<const float4*>(c)[i];
            z[i] = reinterpret_cast<const float4*>(cw)[i];
        }
#pragma unroll
        for (int i = 0; i < DS / 4; i++) {
            if (resid) {
                x[i] = y[i];
            } else {
                const float4 qq = reinterpret_cast<const float4*>(q)[i];
                x[i] = make_float4(__fsub_rn(qq.x, y[i].x), __fsub_rn(qq.y, y[i].y), __fsub_rn(qq.z, y[i].z),
                                   __fsub_rn(qq.w, y[i].w));
            }
            const float d0 = __fsub_rn(x[i].x, z[i].x), d1 = __fsub_rn(x[i].y, z[i].y);
            const float d2 = __fsub_rn(x[i].z, z[i].z), d3 = __fsub_rn(x[i].w, z[i].w);
            e = __fadd_rn(e, __fmul_rn(d0, d0));
            e = __fadd_rn(e, __fmul_rn(d1, d1));
            e = __fadd_rn(e, __fmul_rn(d2, d2));
            e = __fadd_rn(e, __fmul_rn(d3, d3));
        }
    } else {
        const int n = DS > 0 ? DS : ds;
        for (int j = 0; j < n; j++) {
            const float r = resid ? c[j] : __fsub_rn(q[j], c[j]);
            const float t = __fsub_rn(r, cw[j]);
            e = __fadd_rn(e, __fmul_rn(t, t));
        }
    }
    return e;
}

// The reference's distance of one entry, by two adjacent lanes (h = lane & 1;
// M a multiple of 4, ds 8).  Lane h scores codebooks 2 t + h.  The lanes of a
// pair load the two 16-byte halves of a codeword, one cache line for both (a
// lane that loads whole codewords asks for a line per load, and the cache's
// line rate is what bounds the rescoring), and swap the halves they lack;
// both add the scores in codebook order.
__device__ __forceinline__ float sl_pair_distance(const float* q, const float* __restrict__ c, bool resid,
                                                  const float* __restrict__ cb, const uint8_t* __restrict__ row, int M,
                                                  int K, uint32_t h) {
    float total = 0.0f;
    const uint32_t* words = reinterpret_cast<const uint32_t*>(row);
    for (int w = 0; w < M / 4; w++) {
        const uint32_t code4 = words[w];
        float4 A[2], B[2], c0[2], c1[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int m = 4 * w + 2 * t;
            const uint32_t k0 = (code4 >> (16 * t)) & 0xffu, k1 = (code4 >> (16 * t + 8)) & 0xffu;
            A[t] = reinterpret_cast<const float4*>(cb + ((size_t)m * K + k0) * 8)[h];
            B[t] = reinterpret_cast<const float4*>(cb + ((size_t)(m + 1) * K + k1) * 8)[h];
            c0[t] = reinterpret_cast<const float4*>(c + (m + h) * 8)[0];
            c1[t] = reinterpret_cast<const float4*>(c + (m + h) * 8)[1];
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int m = 4 * w + 2 * t + (int)h;
            auto swap1 = [](float x) {
                return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, true));
            };
            const float4 snd = h ? A[t] : B[t];
            const float4 rcv = make_float4(swap1(snd.x), swap1(snd.y), swap1(snd.z), swap1(snd.w));
            const float4 lo = h ? rcv : A[t], hi = h ? B[t] : rcv;
            const float cw[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            const float cc[8] = {c0[t].x, c0[t].y, c0[t].z, c0[t].w, c1[t].x, c1[t].y, c1[t].z, c1[t].w};
            float e = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float r = resid ? cc[j] : __fsub_rn(q[m * 8 + j], cc[j]);
                const float x = __fsub_rn(r, cw[j]);
                e = __fadd_rn(e, __fmul_rn(x, x));
            }
            const float o = swap1(e);
            total = __fadd_rn(__fadd_rn(total, h ? o : e), h ? e : o);
        }
    }
    return total;
}

// LDS of list_final_kernel, bytes from its start.
struct SlFinalLds {
    int q, slot, lab, key, sub, subn, bytes;
};
__host__ __device__ inline SlFinalLds sl_final_lds(int d, int M, int P, int rcap, int nth) {
    SlFinalLds s;
    int o = 0;
    s.key = o;
    o += rcap * 8;
    s.lab = o;
    o += rcap * 4;
    s.q = o;
    o += (d + 3) / 4 * 16;
    s.slot = o;  // list offset, list, tau per slot
    o += P * 12;
    o = (o + 15) / 16 * 16;
    s.sub = o;
    s.subn = nth <= 64 ? 32 : 64;  // entries rescored per pass
    while (s.subn > 16 && s.subn * (M | 1) * 4 > 8 * 1024) s.subn >>= 1;
    o += s.subn * (M | 1) * 4;
    s.bytes = o;
    return s;
}

template <int NTH, int DS>
__global__ __launch_bounds__(NTH) void list_final_kernel(DevIndex ix, ScanArgs a, ListWs w) {
    extern __shared__ __align__(16) char smem[];
    __shared__ uint32_t hist[256];
    __shared__ uint32_t misc[8];
    __shared__ float red[2 * (NTH / 64)];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = blockIdx.x;
    const int P = a.P, M = ix.M, d = ix.d, kout = a.kout;
    const uint32_t total = w.scount[q];
    uint32_t* st = a.qstat + (size_t)q * QSTAT_WORDS;
    auto give_up = [&]() {  // left to list_rescue_kernel
        if (tid == 0) {
            a.flag_list[atomicAdd(a.flag_count, 1u)] = (uint32_t)q;
            st[3] = 1u;
        }
    };
    if (tid == 0) {
        st[1] = 0u;
        st[2] = total;
        st[3] = 0u;
        misc[0] = 0u;
    }
    if (total > (uint32_t)w.cap) {
        give_up();
        return;
    }
    const SlFinalLds lay = sl_final_lds(d, M, P, w.rcap, NTH);
    uint64_t* keys = reinterpret_cast<uint64_t*>(smem + lay.key);
    uint32_t* lab = reinterpret_cast<uint32_t*>(smem + lay.lab);
    float* sq = reinterpret_cast<float*>(smem + lay.q);
    uint32_t* soff = reinterpret_cast<uint32_t*>(smem + lay.slot);
    uint32_t* slist = soff + P;
    float* stau = reinterpret_cast<float*>(slist + P);
    float* sub = reinterpret_cast<float*>(smem + lay.sub);
    const uint2* sv = w.surv + (size_t)q * w.cap;
    const uint32_t tmask = (1u << w.tbits) - 1u;
    // a thread's first C survivors stay in registers, later ones are read again
    constexpr uint32_t C = NTH <= 64 ? 4 : 2;
    uint2 mine[C];
#pragma unroll
    for (uint32_t j = 0; j < C; j++) mine[j] = tid + j * NTH < total ? sv[tid + j * NTH] : make_uint2(0u, 0u);
    for (int i = tid; i < 256; i += NTH) hist[i] = 0u;
    for (int j = tid; j < d; j += NTH) sq[j] = a.qn[(size_t)q * d + j];
    for (int s = tid; s < P; s += NTH) {
        const uint32_t l = min(a.probe[(size_t)q * P + s], (uint32_t)ix.L - 1u);
        slist[s] = l;
        soff[s] = ix.offsets[l];
        stau[s] = list_tau(32 * w.sh.KT, M, ix.ds, w.t0[(size_t)q * P + s], ix.rmax);
    }
    __syncthreads();
    auto each = [&](auto f) {  // f(survivor, valid); every lane of a wave calls it alike
#pragma unroll
        for (uint32_t j = 0; j < C; j++)
            if (j * NTH < total) f(mine[j], tid + j * NTH < total);
        for (uint32_t i0 = C * NTH; i0 < total; i0 += NTH) {
            const bool v = i0 + tid < total;
            f(v ? sv[i0 + tid] : make_uint2(0u, 0u), v);
        }
    };
    uint32_t n = total;
    if (total > (uint32_t)kout) {
        // Upper bounds a + tau in 256 bins; the first bin that reaches k
        // entries bounds the k-th distance, and an entry whose lower bound
        // a - tau falls in a later bin is beyond it (the binning is monotone).
        float mn = 3.0e38f, mxv = -3.0e38f;
        each([&](uint2 s, bool v) {
            const float hi = __uint_as_float(s.y) + stau[s.x >> w.tbits];
            mn = v ? fminf(mn, hi) : mn;
            mxv = v ? fmaxf(mxv, hi) : mxv;
        });
        for (int o = 32; o > 0; o >>= 1) {
            mn = fminf(mn, __shfl_xor(mn, o, 64));
            mxv = fmaxf(mxv, __shfl_xor(mxv, o, 64));
        }
        if (lane == 0) {
            red[wave] = mn;
            red[NTH / 64 + wave] = mxv;
        }
        __syncthreads();
        mn = red[0];
        mxv = red[NTH / 64];
#pragma unroll
        for (int i = 1; i < NTH / 64; i++) {
            mn = fminf(mn, red[i]);
            mxv = fmaxf(mxv, red[NTH / 64 + i]);
        }
        const float sc = mxv > mn ? 255.0f / (mxv - mn) : 0.0f;
        auto bin = [&](float x) { return (uint32_t)fminf(fmaxf((x - mn) * sc, 0.0f), 255.0f); };
        each([&](uint2 s, bool v) {
            if (v) atomicAdd(&hist[bin(__uint_as_float(s.y) + stau[s.x >> w.tbits])], 1u);
        });
        __syncthreads();
        if (tid < 64) {
            const uint32_t h0 = hist[4 * lane], h1 = hist[4 * lane + 1], h2 = hist[4 * lane + 2], h3 = hist[4 * lane + 3];
            uint32_t s = h0 + h1 + h2 + h3;
            const uint32_t own = s;
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t x = __shfl_up(s, o, 64);
                if (lane >= o) s += x;
            }
            const uint32_t ex = s - own, kk = (uint32_t)kout;
            if (ex < kk && s >= kk)
                misc[1] = 4 * lane + (ex + h0 >= kk ? 0 : ex + h0 + h1 >= kk ? 1 : ex + h0 + h1 + h2 >= kk ? 2 : 3);
        }
        __syncthreads();
        const uint32_t bk = misc[1];
        each([&](uint2 s, bool v) {
            const bool take = v && bin(__uint_as_float(s.y) - stau[s.x >> w.tbits]) <= bk;
            const int at = wave_append_slot(take, &misc[0]);
            if (take && at < w.rcap) lab[at] = s.x;
        });
        __syncthreads();
        n = misc[0];
        if (n > (uint32_t)w.rcap) {
            give_up();
            return;
        }
    } else {
        for (uint32_t i = tid; i < total; i += NTH) lab[i] = sv[i].x;
        __syncthreads();
    }
    if (DS == 8 && (M & 3) == 0) {
        for (uint32_t i0 = 0; i0 < n; i0 += NTH / 2) {
            const uint32_t i = i0 + (uint32_t)(tid >> 1), x = lab[min(i, n - 1u)], slot = x >> w.tbits;
            const size_t pos = (size_t)soff[slot] + (x & tmask);
            const uint32_t vid = ix.list_ids[pos];
            const float* c = a.rres ? a.rres + ((size_t)q * P + slot) * d : ix.centroids + (size_t)slist[slot] * d;
            const float s = sl_pair_distance(sq, c, a.rres != nullptr, ix.codebooks, ix.codes + pos * M, M, ix.K,
                                             (uint32_t)tid & 1u);
            if (i < n && (tid & 1) == 0) keys[i] = cand_key(s, vid);
        }
        __syncthreads();
    } else {
    // Exact distances: G lanes per entry, lane m takes codebooks m, m + G, ..;
    // then one thread per entry adds the parts in codebook order.  U entries'
    // codes, then their codewords, are in flight together: one at a time the
    // kernel is a chain of memory round trips.
    constexpr int U = DS == 8 ? 4 : 8;
    int G = 1;
    while (G < M && G < 64) G <<= 1;
    const int g = tid / G, m0 = tid & (G - 1), ng = NTH / G, ms = M | 1;
    for (uint32_t b0 = 0; b0 < n; b0 += lay.subn) {
        const uint32_t nb = min((uint32_t)lay.subn, n - b0);
        const uint32_t xt = lab[b0 + min((uint32_t)tid, nb - 1u)];  // this thread's entry (subn <= NTH)
        const uint32_t vid = ix.list_ids[(size_t)soff[xt >> w.tbits] + (xt & tmask)];
        for (int m = m0; m < M; m += G)
            for (uint32_t i0 = g; i0 < nb; i0 += ng * U) {
                uint32_t code[U], at[U];
                const float* c[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    at[u] = min(i0 + u * ng, nb - 1u);  // past the end: the last entry again
                    const uint32_t x = lab[b0 + at[u]], slot = x >> w.tbits, t = x & tmask;
                    code[u] = ix.codes[((size_t)soff[slot] + t) * M + m];
                    c[u] = (a.rres ? a.rres + ((size_t)q * P + slot) * d : ix.centroids + (size_t)slist[slot] * d) + m * ix.ds;
                }
                float e[U];
#pragma unroll
                for (int u = 0; u < U; u++)
                    e[u] = sl_sub<DS>(sq + m * ix.ds, c[u], ix.codebooks + ((size_t)m * ix.K + code[u]) * ix.ds, ix.ds,
                                      a.rres != nullptr);
#pragma unroll
                for (int u = 0; u < U; u++) sub[at[u] * ms + m] = e[u];
            }
        __syncthreads();
        if ((uint32_t)tid < nb) {
            float s = 0.0f;
            int m = 0;
            for (; m + 8 <= M; m += 8) {
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; j++) x[j] = sub[tid * ms + m + j];
#pragma unroll
                for (int j = 0; j < 8; j++) s = __fadd_rn(s, x[j]);
            }
            for (; m < M; m++) s = __fadd_rn(s, sub[tid * ms + m]);
            keys[b0 + tid] = cand_key(s, vid);
        }
        __syncthreads();
    }
    }
    // Each key to its rank, the number of smaller keys (all distinct).
    for (uint32_t i = tid; i < n; i += NTH) {
        const uint64_t ki = keys[i];
        const uint32_t vi = (uint32_t)ki;
        const uint32_t doc = a.out_ids && a.doc_ids ? a.doc_ids[vi] : vi;  // flies during the count
        uint32_t r = 0;
        uint32_t j = 0;
        for (; j + 4 <= n; j += 4) {
            const ulonglong2 x = *reinterpret_cast<const ulonglong2*>(keys + j);
            const ulonglong2 y = *reinterpret_cast<const ulonglong2*>(keys + j + 2);
            r += (x.x < ki ? 1u : 0u) + (x.y < ki ? 1u : 0u) + (y.x < ki ? 1u : 0u) + (y.y < ki ? 1u : 0u);
        }
        for (; j < n; j++) r += keys[j] < ki ? 1u : 0u;
        if (r < (uint32_t)kout) {
            const size_t o = (size_t)q * kout + r;
            if (a.out_ids) {
                a.out_ids[o] = (int64_t)doc;
                a.out_dists[o] = key_dist(ki);
            } else {
                a.out_vidx[o] = vi;
                a.out_dist[o] = key_dist(ki);
            }
        }
    }
    for (int j = (int)n + tid; j < kout; j += NTH) scan_emit(a, q, j, ~0ull, false);
}

// ---- flagged queries ------------------------------------------------------

// Keys kept in an LDS buffer: append, and when the buffer is nearly full sort
// and cut it to the k smallest.  All 256 threads call it alike.
struct SlTop {
    uint64_t* keys;  // [SL_TOP]
    uint32_t* cnt;
    uint64_t thr;    // keys from here on are out
};
#define SL_TOP 2048
__device__ __forceinline__ void sl_top_cut(SlTop& t, int k) {
    __syncthreads();
    const uint32_t c = *t.cnt;
    __syncthreads();
    if (c <= SL_TOP - VGPU_BLOCK) return;
    for (uint32_t i = c + threadIdx.x; i < SL_TOP; i += VGPU_BLOCK) t.keys[i] = ~0ull;
    block_bitonic_sort_keys(t.keys, SL_TOP);
    t.thr = t.keys[k - 1];
    if (threadIdx.x == 0) *t.cnt = (uint32_t)k;
    __syncthreads();
}
__device__ __forceinline__ void sl_top_add(SlTop& t, uint64_t key, bool valid, int k) {
    const bool take = valid && key < t.thr;
    const int at = wave_append_slot(take, t.cnt);
    if (take) t.keys[at] = key;
    sl_top_cut(t, k);
}
// Sorts what is kept; returns how many keys (at most k).
__device__ __forceinline__ uint32_t sl_top_end(SlTop& t, int k) {
    __syncthreads();
    const uint32_t c = *t.cnt;
    const int n2 = next_pow2(c > 0 ? (int)c : 1);
    for (uint32_t i = c + threadIdx.x; i < (uint32_t)n2; i += VGPU_BLOCK) t.keys[i] = ~0ull;
    block_bitonic_sort_keys(t.keys, n2);
    return min(c, (uint32_t)k);
}

// Up to SL_RESCUE_MAX flagged queries with the reference's arithmetic: each
// one's survivors, when its buffer holds them all, or else every entry of its
// lists, spread over up to 64 workgroups whose k smallest keys the last of them
// to finish merges.  One workgroup per query, as the EXACT kernel has it, took
// 380 us for a single query at 10M x 96; but the entries here cost an L1 gather
// per codeword (6 per ns), where the EXACT kernel looks them up in LDS (50 per
// ns over a full chip), so more flagged queries than that are left to it.
template <int DS>
__global__ __launch_bounds__(256) void list_rescue_kernel(DevIndex ix, ScanArgs a, ListWs w) {
    extern __shared__ __align__(16) char smem[];
    __shared__ uint32_t cnt, last;
    __shared__ uint64_t bound;
    const uint32_t nf = *a.flag_count;
    if (nf == 0 || nf > SL_RESCUE_MAX) return;
    uint64_t* keys = reinterpret_cast<uint64_t*>(smem);
    const int tid = threadIdx.x, d = ix.d, M = ix.M, k = a.kout;
    float* r = reinterpret_cast<float*>(smem + SL_TOP * 8);  // [d]
    uint32_t* sl_l = reinterpret_cast<uint32_t*>(r + (d + 3) / 4 * 4);  // [P] lists, first positions, lengths
    uint32_t *sl_o = sl_l + a.P, *sl_n = sl_o + a.P;
    const uint32_t S = min(64u, SL_RESCUE / nf);  // workgroups per query: 8 to 64
    for (uint32_t job = blockIdx.x; job < nf * S; job += gridDim.x) {
        const uint32_t f = job / S, sl = job % S, q = a.flag_list[f];
        const uint32_t* pr = a.probe + (size_t)q * a.P;
        const uint32_t kept = w.scount[q];
        const bool all_kept = kept <= (uint32_t)w.cap;
        const uint64_t E = all_kept ? kept : a.qstat[(size_t)q * QSTAT_WORDS];
        const uint64_t e0 = E * sl / S, e1 = E * (sl + 1) / S;
        __syncthreads();
        if (tid == 0) cnt = 0u;
        for (int p = tid; p < a.P; p += VGPU_BLOCK) {
            const bool in = pr[p] < (uint32_t)ix.L;
            const uint32_t l = in ? pr[p] : 0u, o = ix.offsets[l];
            sl_l[p] = l;
            sl_o[p] = o;
            sl_n[p] = in ? ix.offsets[l + 1] - o : 0u;
        }
        __syncthreads();
        SlTop top{keys, &cnt, ~0ull};
        if (all_kept) {
            const uint2* sv = w.surv + (size_t)q * w.cap;
            for (uint64_t b = e0; b < e1; b += VGPU_BLOCK) {
                const bool ok = b + tid < e1;
                const uint32_t x = sv[ok ? b + tid : e0].x, slot = x >> w.tbits;
                const size_t pos = (size_t)sl_o[slot] + (x & ((1u << w.tbits) - 1u));
                const float* c = a.rres ? a.rres + ((size_t)q * a.P + slot) * d : ix.centroids + (size_t)sl_l[slot] * d;
                float s = 0.0f;
#pragma unroll 4
                for (int m = 0; m < M; m++) {
                    const float* cw = ix.codebooks + ((size_t)m * ix.K + ix.codes[pos * M + m]) * ix.ds;
                    s = __fadd_rn(s, sl_sub<DS>(a.qn + (size_t)q * d + m * ix.ds, c + m * ix.ds, cw, ix.ds,
                                                a.rres != nullptr));
                }
                sl_top_add(top, cand_key(s, ix.list_ids[pos]), ok, k);
            }
        }
        uint64_t at = 0;  // entries of the lists before
        for (int p = 0; !all_kept && p < a.P && at < e1; p++) {
            const uint32_t l = sl_l[p], o0 = sl_o[p], len = sl_n[p];
            const uint64_t lo = at > e0 ? at : e0, hi = at + len < e1 ? at + len : e1;
            if (lo < hi) {
                __syncthreads();
                for (int j = tid; j < d; j += VGPU_BLOCK)
                    r[j] = a.rres ? a.rres[((size_t)q * a.P + p) * d + j]
                                  : __fsub_rn(a.qn[(size_t)q * d + j], ix.centroids[(size_t)l * d + j]);
                __syncthreads();
                for (uint64_t b = lo; b < hi; b += VGPU_BLOCK) {
                    const bool ok = b + tid < hi;
                    const size_t pos = o0 + (size_t)((ok ? b + tid : lo) - at);
                    float s = 0.0f;
#pragma unroll 8
                    for (int m = 0; m < M; m++) {
                        const float* cw = ix.codebooks + ((size_t)m * ix.K + ix.codes[pos * M + m]) * ix.ds;
                        s = __fadd_rn(s, sl_sub<DS>(nullptr, r + m * ix.ds, cw, ix.ds, true));
                    }
                    sl_top_add(top, cand_key(s, ix.list_ids[pos]), ok, k);
                }
            }
            at += len;
        }
        uint32_t n = sl_top_end(top, k);
        uint64_t* part = w.rescue + (size_t)f * S * k;
        for (int i = tid; i < k; i += VGPU_BLOCK) part[sl * k + i] = (uint32_t)i < n ? keys[i] : ~0ull;
        __threadfence();
        __syncthreads();
        if (tid == 0) last = atomicAdd(&w.rescued[f], 1u) == S - 1u;
        __syncthreads();
        if (!last) continue;
        __threadfence();
        // Every workgroup has (k - 1) / S + 1 keys up to the largest of their keys of
        // that rank, together at least k: keys above it are out (6400 keys of 64
        // workgroups at k 100 were four sorts of the buffer, 80 us).
        if (tid < 64) {
            uint64_t t = tid < S ? __hip_atomic_load(part + (size_t)tid * k + (k - 1) / S, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)
                                 : 0ull;
            for (int o = 32; o > 0; o >>= 1) {
                const uint64_t x = (uint64_t)__shfl_xor((long long)t, o, 64);
                t = x > t ? x : t;
            }
            if (tid == 0) {
                cnt = 0u;
                bound = t;
            }
        }
        __syncthreads();
        top.thr = bound == ~0ull ? ~0ull : bound + 1ull;
        for (uint32_t b = 0; b < S * (uint32_t)k; b += VGPU_BLOCK) {
            const bool ok = b + tid < S * (uint32_t)k;
            const uint64_t key =
                ok ? __hip_atomic_load(part + b + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : ~0ull;
            sl_top_add(top, key, ok && key != ~0ull, k);
        }
        n = sl_top_end(top, k);
        for (int j = tid; j < k; j += VGPU_BLOCK)
            scan_emit(a, (int)q, j, (uint32_t)j < n ? keys[j] : ~0ull, (uint32_t)j < n);
        __syncthreads();
    }
}

// ---- launch ---------------------------------------------------------------

static size_t sl_score_lds(const ListShape& sh) { return sh.table_bytes + SL_WAVES * sizeof(SlWave); }

template <int KT, int DSP>
static void launch_score(const DevIndex& ix, const ScanArgs& a, const ListWs& w, bool sample, hipStream_t s) {
    const size_t lds = sl_score_lds(w.sh);
    const int per_cu = lds * 2 <= 160 * 1024 ? 2 : 1;
    auto k = sample ? list_score_kernel<KT, DSP, true> : list_score_kernel<KT, DSP, false>;
    ensure_dyn_lds((const void*)k, lds);
    hipLaunchKernelGGL(k, dim3(256 * per_cu), dim3(SL_THREADS), lds, s, ix, a, w);
}

template <int KT>
static void launch_score_d(const DevIndex& ix, const ScanArgs& a, const ListWs& w, bool sample, hipStream_t s) {
    switch (w.sh.dsp) {
        case 1: launch_score<KT, 1>(ix, a, w, sample, s); break;
        case 2: launch_score<KT, 2>(ix, a, w, sample, s); break;
        case 4: launch_score<KT, 4>(ix, a, w, sample, s); break;
        default: launch_score<KT, 8>(ix, a, w, sample, s); break;
    }
}

static void launch_score_any(const DevIndex& ix, const ScanArgs& a, const ListWs& w, bool sample, hipStream_t s) {
    switch (w.sh.KT) {
        case 1: launch_score_d<1>(ix, a, w, sample, s); break;
        case 2: launch_score_d<2>(ix, a, w, sample, s); break;
        case 3: launch_score_d<3>(ix, a, w, sample, s); break;
        default: launch_score_d<4>(ix, a, w, sample, s); break;
    }
}

template <int NTH>
static void launch_final(const DevIndex& ix, const ScanArgs& a, const ListWs& w, hipStream_t s) {
    const size_t lds = (size_t)sl_final_lds(ix.d, ix.M, a.P, w.rcap, NTH).bytes;
    auto k = ix.ds == 8 ? list_final_kernel<NTH, 8> : ix.ds == 4 ? list_final_kernel<NTH, 4>
             : ix.ds == 2 ? list_final_kernel<NTH, 2> : ix.ds == 1 ? list_final_kernel<NTH, 1>
                                                                 : list_final_kernel<NTH, 0>;
    ensure_dyn_lds((const void*)k, lds);
    hipLaunchKernelGGL(k, dim3(a.nq), dim3(NTH), lds, s, ix, a, w);
}

static void launch_rescue(const DevIndex& ix, const ScanArgs& a, const ListWs& w, hipStream_t s) {
    const size_t lds = SL_TOP * 8 + (size_t)(ix.d + 3) / 4 * 16 + (size_t)a.P * 12;
    auto k = ix.ds == 8 ? list_rescue_kernel<8> : ix.ds == 4 ? list_rescue_kernel<4>
             : ix.ds == 2 ? list_rescue_kernel<2> : list_rescue_kernel<0>;
    ensure_dyn_lds((const void*)k, lds);
    hipLaunchKernelGGL(k, dim3(SL_RESCUE), dim3(VGPU_BLOCK), lds, s, ix, a, w);
}

// The pairs and work items of a chunk.
void launch_list_pairs(const DevIndex& ix, const ScanArgs& a, ListWs& w, hipStream_t s) {
    w.qw = list_count_queries(a.nq);
    w.nwg = (a.nq + w.qw - 1) / w.qw;
    const size_t lds = (size_t)ix.L * 4;
    ensure_dyn_lds((const void*)list_count_kernel, lds);
    hipLaunchKernelGGL(list_count_kernel, dim3((a.nq + w.qw - 1) / w.qw), dim3(1024), lds, s, ix, a, w);
    hipLaunchKernelGGL(list_plan_kernel, dim3((ix.L + 255) / 256), dim3(1024), 0, s, ix, w);
    const size_t np = (size_t)a.nq * a.P;
    hipLaunchKernelGGL(list_scatter_kernel, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, s, ix, a, w);
}

void launch_list_bound(const ScanArgs& a, const ListWs& w, hipStream_t s) {
    const dim3 bg((a.nq + 3) / 4);
    switch (w.tcap) {
        case 32: hipLaunchKernelGGL(list_bound_kernel<2>, bg, dim3(256), 0, s, a, w); break;
        case 64: hipLaunchKernelGGL(list_bound_kernel<4>, bg, dim3(256), 0, s, a, w); break;
        case 256: hipLaunchKernelGGL(list_bound_kernel<16>, bg, dim3(256), 0, s, a, w); break;
        default: hipLaunchKernelGGL(list_bound_kernel<8>, bg, dim3(256), 0, s, a, w); break;
    }
}

void launch_scan_list(const DevIndex& ix, const ScanArgs& a, const ListWs& ws, hipStream_t s) {
    if (a.nq <= 0) return;
    ListWs w = ws;
    w.rows = w.padded ? w.padded : a.qn;
    launch_list_pairs(ix, a, w, s);
    launch_score_any(ix, a, w, true, s);
    launch_list_bound(a, w, s);
    launch_score_any(ix, a, w, false, s);
    if (a.kout <= 16) launch_final<64>(ix, a, w, s);
    else launch_final<256>(ix, a, w, s);
    launch_rescue(ix, a, w, s);
    ScanArgs e = a;  // more flagged queries than that: the EXACT kernel
    e.exact = 1;
    e.only_flagged = 1;
    e.flag_over = SL_RESCUE_MAX;
    launch_scan8_exact(ix, e, s);
}

}  // namespace vgpu
