// Batched 4-bit FastScan by inverted list.
//
// fastscan_kernel (k_fastscan.hip) takes one query per workgroup and looks
// every nibble up with byte selects: 2.5 ms for 312M entries of 50 codebooks
// (10,000 queries of 64 lists), bound by those vector instructions (16 per
// dword of 8 nibbles).  A quantised distance is the sum of one byte of the
// pair's table per codebook, i.e. a product of the entry's one-hot vector (16
// positions per codebook, one of them 1) with the table; the one-hot vectors
// of a list are shared by every query that probes it, so the sums of a list
// against its pairs are an int8 matrix product:
//
//   pairs and work items   k_scan_list.hip's
//   fs_list_kernel<.., SAMPLE>    distances of the first 16 tcap entries of
//       each query's nearest lists; list_bound_kernel takes the k-th smallest
//   fs_list_kernel<.., !SAMPLE>   every pair: entries within the bound are
//       appended to the query's survivors with their distances
//   fs_final_kernel               the k nearest survivors, ranked
//   fastscan_flagged              queries whose survivors did not fit
//
// The tables are the reference's (quantize_lut_flat, pq_simd.rs:576-611) and
// the sums are integers, so every distance is the reference's bit for bit
// (pq_simd.rs:721-769) and nothing is rescored.  Table bytes go in less 128
// (signed operands); the accumulators start from 128 M.
//
// Layout: a wave takes 32 pairs (two tiles of 16) of one list and builds their
// tables straight in the B operand registers: lane (pair col, group kg) holds
// the 16 bytes of codebook 4 x + kg of its pair for step x (64 one-hot
// positions, four codebooks) of v_mfma_i32_16x16x64_i8.  An A operand is one
// 16-byte read of the nibble's one-hot row from LDS.  Each codeword that is
// read from LDS serves both tiles.
//
// Bounds, at 10k queries x 64 lists of 488 entries, M 50: the vector
// instructions, most of them the table build's (two passes over 800 values per
// pair, as in fastscan_kernel).  VALU 62% busy, matrix cores 16% (115 us), LDS
// 14%, waves waiting 43% of their time, in the 738 us of the scan; the sample
// takes 144.  Whole search 2718 -> 1117 us.  The rows' parts of the next step
// are loaded under the present one (1313 -> 1253), and items hold 32 pairs, one
// pass of a wave: with 64 the few popular lists' waves ran twice as long at the
// end of the sample and of the scan (1253 -> 1117).
#include "vgpu_device.h"
#include "vgpu_launch.h"

namespace vgpu {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

#define FL_NT 2                   // pair tiles per pass over a list's entries
#define FL_PAIRS (16 * FL_NT)
#define FL_WAVES 8
#define FL_THREADS (64 * FL_WAVES)
#define FL_STAGE 320              // survivors a wave stages in LDS before it flushes
#define FL_RCAP 1024              // survivors that can be ranked

bool fast_list_shape(int M, int ds) { return M <= 64 && (ds == 1 || ds == 2 || ds == 4); }
int fast_list_words(int M) { return M <= 32 ? 1 : 2; }

// Tile T (16 entries of one list), lane l: nibble x is the code of codebook
// 4 x + l / 16 of entry l % 16 (0 past the list or the codebooks).
__global__ __launch_bounds__(256) void fs_list_tiles_kernel(DevIndex ix, int LW, uint32_t* __restrict__ out) {
    const int l = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t o0 = ix.offsets[l], len = ix.offsets[l + 1] - o0;
    const uint32_t t0 = ix.ltoff[l], nt = ix.ltoff[l + 1] - t0;
    const int e = lane & 15, kg = lane >> 4;
    for (uint32_t t = wave; t < nt; t += 4) {
        const uint32_t j = t * 16 + e;
        const bool ok = j < len;
        const uint8_t* row = ix.codes + (size_t)(o0 + (ok ? j : 0u)) * ix.M;
        for (int w = 0; w < LW; w++) {
            uint32_t v = 0;
            for (int x = 0; x < 8; x++) {
                const int m = 4 * (8 * w + x) + kg;
                if (ok && m < ix.M) v |= (uint32_t)(row[m] & 15) << (4 * x);
            }
            out[((size_t)(t0 + t) * 64 + lane) * LW + w] = v;
        }
    }
}

void launch_fast_list_tiles(const DevIndex& ix, uint32_t* lcodes, hipStream_t s) {
    if (ix.L <= 0) return;
    hipLaunchKernelGGL(fs_list_tiles_kernel, dim3(ix.L), dim3(256), 0, s, ix, fast_list_words(ix.M), lcodes);
}

__device__ __forceinline__ void fl_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A wave's LDS: staged survivors, and per pair their count and reservation and
// the pair word.
struct FlWave {
    uint2 stage[FL_STAGE];  // (distance bits, entry | pair << 26)
    uint32_t cnt[FL_PAIRS];
    uint32_t base[FL_PAIRS];
    uint32_t pair[FL_PAIRS];
};

// Write the staged survivors to their queries' buffers: one reservation per
// pair with any, then every entry at its place.
__device__ __forceinline__ void fl_flush(FlWave& sw, const ListWs& w, uint32_t& ns) {
    const int lane = threadIdx.x & 63;
    fl_wave_sync();
    if (lane < FL_PAIRS) sw.cnt[lane] = 0u;
    fl_wave_sync();
    uint32_t at[FL_STAGE / 64];
    uint2 st[FL_STAGE / 64];
#pragma unroll
    for (int i = 0; i < FL_STAGE / 64; i++) {
        const uint32_t x = i * 64 + lane;
        if (x < ns) {
            st[i] = sw.stage[x];
            at[i] = atomicAdd(&sw.cnt[st[i].y >> 26], 1u);
        }
    }
    fl_wave_sync();
    if (lane < FL_PAIRS) {
        const uint32_t c = sw.cnt[lane];
        if (c) sw.base[lane] = atomicAdd(&w.scount[sw.pair[lane] >> SL_SLOT_BITS], c);
    }
    fl_wave_sync();
#pragma unroll
    for (int i = 0; i < FL_STAGE / 64; i++) {
        const uint32_t x = i * 64 + lane;
        if (x >= ns) continue;
        const uint32_t p = st[i].y >> 26, word = sw.pair[p], to = sw.base[p] + at[i];
        if (to < (uint32_t)w.cap)
            w.surv[(size_t)(word >> SL_SLOT_BITS) * w.cap + to] =
                make_uint2((word & ((1u << SL_SLOT_BITS) - 1u)) << w.tbits | (st[i].y & 0x3ffffffu), st[i].x);
    }
    ns = 0;
    fl_wave_sync();
}

// Stage the lanes' survivors (take may differ by lane; at most 64 a call).
__device__ __forceinline__ void fl_stage(FlWave& sw, const ListWs& w, uint32_t& ns, bool take, float dist,
                                         uint32_t label) {
    const uint64_t b = __ballot(take);
    if (!b) return;
    if (ns > FL_STAGE - 64) fl_flush(sw, w, ns);
    const uint32_t below =
        __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
    if (take) sw.stage[ns + below] = make_uint2(__float_as_uint(dist), label);
    ns += (uint32_t)__popcll(b);
}

// Dimensions DS m .. of a row.
template <int DS>
__device__ __forceinline__ void fl_load(const float* __restrict__ row, int m, float (&x)[DS]) {
    if constexpr (DS == 4) {
        const float4 v = *reinterpret_cast<const float4*>(row + m * 4);
        x[0] = v.x, x[1] = v.y, x[2] = v.z, x[3] = v.w;
    } else if constexpr (DS == 2) {
        const float2 v = *reinterpret_cast<const float2*>(row + m * 2);
        x[0] = v.x, x[1] = v.y;
    } else {
        x[0] = row[m];
    }
}

// The residual part of codebook m of a pair: row - c, or the rotated residual
// (its row less 0, which changes nothing: no branch splits the steps).
template <int DS>
__device__ __forceinline__ void fl_resid(const float (&x)[DS], const float (&c)[DS], bool resid, float (&r)[DS]) {
#pragma unroll
    for (int j = 0; j < DS; j++) r[j] = __fsub_rn(x[j], resid ? 0.0f : c[j]);
}

// sum_j (r_j - cw_j)^2 in j order, every step rounded (pq.rs:232-251).
template <int DS>
__device__ __forceinline__ float fl_value(const float (&r)[DS], const float* cw) {
    float e = 0.0f;
#pragma unroll
    for (int j = 0; j < DS; j++) {
        const float t = __fsub_rn(r[j], cw[j]);
        e = j ? __fadd_rn(e, __fmul_rn(t, t)) : __fmul_rn(t, t);  // 0 + x is x
    }
    return e;
}

// Floats of one codebook in LDS: 16 codewords and four of padding, so that
// the four groups' codebooks start in different banks.
template <int DS>
constexpr int fl_cb_stride() {
    return 16 * DS + 4;
}

// 32 pairs (word: lane i's pair word, i < np) against tiles [tile0, tile1) of
// list l.
template <int KS, int DS, int LW, bool SAMPLE>
__device__ __forceinline__ void fl_item(const DevIndex& ix, const ScanArgs& a, const ListWs& w, const float* cbs,
                                        const u32x4* onehot, FlWave& sw, uint32_t l, uint32_t np, uint32_t lword,
                                        uint32_t tile0, uint32_t tile1) {
    constexpr int CS = fl_cb_stride<DS>();
    const int lane = threadIdx.x & 63, col = lane & 15, kg = lane >> 4;
    const int M = ix.M, d = ix.d;
    const bool resid = a.rres != nullptr;
    const uint32_t o0 = ix.offsets[l], len = ix.offsets[l + 1] - o0, tb0 = ix.ltoff[l];
    const float* cent = ix.centroids + (size_t)l * d;
    uint32_t word[FL_NT];
    const float* row[FL_NT];
    bool ok[FL_NT];
    float B[FL_NT];
    uint32_t gq[FL_NT], tlim[FL_NT];  // SAMPLE: the pair's bound row, and its tiles to write
#pragma unroll
    for (int i = 0; i < FL_NT; i++) {
        const uint32_t pi = i * 16 + col;
        ok[i] = pi < np;
        word[i] = (uint32_t)__shfl((int)lword, (int)(ok[i] ? pi : 0u), 64);
        const uint32_t q = word[i] >> SL_SLOT_BITS, slot = word[i] & ((1u << SL_SLOT_BITS) - 1u);
        const uint32_t pair = q * (uint32_t)a.P + slot;
        row[i] = resid ? a.rres + (size_t)pair * d : a.qn + (size_t)q * d;
        if (SAMPLE) {
            const uint32_t tb = w.tbase[pair];
            gq[i] = q * (uint32_t)(16 * w.tcap) + 16u * tb;
            tlim[i] = ok[i] ? (uint32_t)w.tcap - tb : 0u;
        } else {
            B[i] = w.bound[q];
            if (kg == 0) sw.pair[pi] = word[i];
        }
    }
    fl_wave_sync();
    uint32_t ns = 0;
    if (len < 16) {
        // the exact float path (search.rs:1355-1375), lane (entry col, pairs
        // kg, kg + 4, ..): m-ordered sum of the float table (pq.rs:272-279)
        for (uint32_t p0 = 0; p0 < np; p0 += 4) {
            const uint32_t p = p0 + kg;
            const uint32_t pw = (uint32_t)__shfl((int)lword, (int)min(p, np - 1u), 64);
            const uint32_t q = pw >> SL_SLOT_BITS, pair = q * (uint32_t)a.P + (pw & ((1u << SL_SLOT_BITS) - 1u));
            const bool take = p < np && (uint32_t)col < len;
            float dist = __int_as_float(0x7f800000);
            if (take) {
                const float* rw = resid ? a.rres + (size_t)pair * d : a.qn + (size_t)q * d;
                const uint8_t* cr = ix.codes + (size_t)(o0 + col) * M;
                dist = 0.0f;
                for (int m = 0; m < M; m++) {
                    float x[DS], c[DS], r[DS];
                    fl_load<DS>(rw, m, x);
                    fl_load<DS>(cent, m, c);
                    fl_resid<DS>(x, c, resid, r);
                    dist = __fadd_rn(dist, fl_value<DS>(r, cbs + m * CS + cr[m] * DS));
                }
            }
            if (SAMPLE) {
                // one tile, and the pair is a sample pair: it has room
                if (p < np) w.gbound[q * (uint32_t)(16 * w.tcap) + 16u * w.tbase[pair] + col] = dist;
            } else {
                fl_stage(sw, w, ns, take && dist <= w.bound[q], dist, (uint32_t)col | p << 26);
            }
        }
        if (!SAMPLE && ns) fl_flush(sw, w, ns);
        return;
    }
    // codes two tiles ahead
    uint32_t cw[2][LW];
    const uint32_t* codes = ix.lcodes + ((size_t)tb0 * 64 + lane) * LW;
    auto fetch = [&](const int S, uint32_t t) {
        t = min(t, tile1 - 1);  // past the item: any of its tiles, never used
#pragma unroll
        for (int i = 0; i < LW; i++) cw[S][i] = codes[(size_t)t * 64 * LW + i];
    };
    fetch(0, tile0);
    fetch(1, tile0 + 1);
    // the tables: smallest and largest value, then every value again as its
    // byte, (v - min) * 255 / range rounded half away from zero
    float mn[FL_NT], mx[FL_NT];
#pragma unroll
    for (int i = 0; i < FL_NT; i++) {
        mn[i] = __int_as_float(0x7f800000);
        mx[i] = __int_as_float(0xff800000);
    }
    auto values = [&](int m, const float (&r)[FL_NT][DS], auto f) {  // f(codeword, pair tile, value)
        const float4* p = reinterpret_cast<const float4*>(cbs + m * CS);
#pragma unroll
        for (int g = 0; g < 4 * DS; g++) {
            const float4 v = p[g];
            const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int c = 0; c < 4 / DS; c++)
#pragma unroll
                for (int i = 0; i < FL_NT; i++) f(g * (4 / DS) + c, i, fl_value<DS>(r[i], x + c * DS));
        }
    };
    // the rows' and the centroid's part of the next step fly while a step runs
    float rx[2][FL_NT][DS], rc[2][DS];
    auto load_step = [&](const int S, int x) {
        int m = min(4 * x + kg, M - 1);  // past the codebooks: the last again
        // both passes' loads are one where the registers hold all of them
        if constexpr (KS * DS > 26) asm volatile("" : "+v"(m));
        fl_load<DS>(cent, m, rc[S]);
#pragma unroll
        for (int i = 0; i < FL_NT; i++) fl_load<DS>(row[i], m, rx[S][i]);
    };
    load_step(0, 0);
#pragma unroll
    for (int x = 0; x < KS; x++) {
        int m = min(4 * x + kg, M - 1);
        asm volatile("" : "+v"(m));
        __builtin_amdgcn_sched_barrier(0);
        load_step((x + 1) & 1, x + 1 < KS ? x + 1 : 0);
        float r[FL_NT][DS];
#pragma unroll
        for (int i = 0; i < FL_NT; i++) fl_resid<DS>(rx[x & 1][i], rc[x & 1], resid, r[i]);
        values(m, r, [&](int, int i, float v) {
            mn[i] = fminf(mn[i], v);
            mx[i] = fmaxf(mx[i], v);
        });
#pragma unroll
        for (int i = 0; i < FL_NT; i++) asm volatile("" : "+v"(mn[i]), "+v"(mx[i]));  // computed by here
    }
    float sc[FL_NT], off[FL_NT], inv[FL_NT];
    int T[FL_NT];
#pragma unroll
    for (int i = 0; i < FL_NT; i++) {
        mn[i] = fminf(mn[i], __shfl_xor(mn[i], 16, 64));
        mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], 16, 64));
        mn[i] = fminf(mn[i], __shfl_xor(mn[i], 32, 64));
        mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], 32, 64));
        const float range = mx[i] - mn[i];
        sc[i] = range < 1.1920929e-07f ? 1.0f : range / 255.0f;
        inv[i] = range < 1.1920929e-07f ? 0.0f : 255.0f / range;
        off[i] = __fmul_rn(mn[i], (float)M);
        if (!SAMPLE) {
            // sums whose distance may be within the bound, with room for the
            // roundings of a distance and of this line
            const float lim = (B[i] - off[i]) / sc[i] + 2.0f + 4.8e-7f * ((fabsf(B[i]) + fabsf(off[i])) / sc[i]);
            T[i] = !ok[i] ? -1 : lim < 65536.0f ? (int)fmaxf(lim, -1.0f) : 65536;
        }
    }
    u32x4 tab[FL_NT][KS];
#pragma unroll
    for (int x = 0; x < KS; x++) {
        // one step's codewords at a time, none kept from one item to the next:
        // the tables fill the registers
        int m = min(4 * x + kg, M - 1);
        asm volatile("" : "+v"(m));
        __builtin_amdgcn_sched_barrier(0);
        const bool in = 4 * x + kg < M;
        constexpr int S0 = KS & 1;  // where the first pass left step 0
        if (x + 1 < KS) load_step((x + 1 + S0) & 1, x + 1);
        float r[FL_NT][DS];
#pragma unroll
        for (int i = 0; i < FL_NT; i++) fl_resid<DS>(rx[(x + S0) & 1][i], rc[(x + S0) & 1], resid, r[i]);
        uint32_t b[FL_NT][4];
        values(m, r, [&](int c, int i, float v) {
            const float y = __fmul_rn(__fsub_rn(v, mn[i]), inv[i]);
            // y + 0.5 is exact or rounds to the right side but just below 0.5
            const uint32_t u = y < 0.5f ? 0u : (uint32_t)__fadd_rn(y, 0.5f);
            b[i][c >> 2] = (c & 3) ? b[i][c >> 2] | u << (8 * (c & 3)) : u;
        });
#pragma unroll
        for (int i = 0; i < FL_NT; i++)
#pragma unroll
            for (int h = 0; h < 4; h++) {
                b[i][h] = in ? b[i][h] ^ 0x80808080u : 0u;
                asm volatile("" : "+v"(b[i][h]));  // computed by here
                tab[i][x][h] = b[i][h];
            }
    }
    auto step = [&](const int S, uint32_t t) {
        i32x4 acc[FL_NT];
#pragma unroll
        for (int i = 0; i < FL_NT; i++) acc[i] = i32x4{128 * M, 128 * M, 128 * M, 128 * M};
#pragma unroll
        for (int x = 0; x < KS; x++) {
            const u32x4 oh = onehot[(cw[S][x >> 3] >> (4 * (x & 7))) & 15u];
#pragma unroll
            for (int i = 0; i < FL_NT; i++)
                acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, oh),
                                                               __builtin_bit_cast(i32x4, tab[i][x]), acc[i], 0, 0, 0);
        }
        fetch(S, t + 2);
        const uint32_t e0 = t * 16 + 4 * kg;  // the lane's entries e0 .. + 3 of pair col
        if constexpr (SAMPLE) {
#pragma unroll
            for (int i = 0; i < FL_NT; i++)
                if (t < tlim[i]) {
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        v[e] = e0 + e < len ? __fadd_rn(__fmul_rn((float)acc[i][e], sc[i]), off[i])
                                            : __int_as_float(0x7f800000);
                    *reinterpret_cast<float4*>(w.gbound + gq[i] + 16 * t + 4 * kg) = make_float4(v[0], v[1], v[2], v[3]);
                }
        } else {
            bool any = false;
#pragma unroll
            for (int i = 0; i < FL_NT; i++) {
                const int lo = min(min(acc[i][0], acc[i][1]), min(acc[i][2], acc[i][3]));
                any |= lo <= T[i];
            }
            if (__any(any)) {
#pragma unroll
                for (int i = 0; i < FL_NT; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float dist = __fadd_rn(__fmul_rn((float)acc[i][e], sc[i]), off[i]);
                        fl_stage(sw, w, ns, acc[i][e] <= T[i] && dist <= B[i] && e0 + e < len, dist,
                                 (e0 + e) | (uint32_t)(i * 16 + col) << 26);
                    }
            }
        }
    };
    for (uint32_t t = tile0; t < tile1; t += 2) {
        step(0, t);
        if (t + 1 < tile1) step(1, t + 1);
    }
    if (!SAMPLE && ns) fl_flush(sw, w, ns);
}

// Persistent, like list_score_kernel: workgroup b takes the work items b, b +
// gridDim.x, ..; its waves share them through a counter in LDS.  LDS: the
// codebooks, the one-hot rows, then one FlWave per wave.
template <int KS, int DS, bool SAMPLE>
__global__ __launch_bounds__(FL_THREADS, 2) void fs_list_kernel(DevIndex ix, ScanArgs a, ListWs w) {
    extern __shared__ __align__(16) char smem[];
    __shared__ uint32_t head;
    constexpr int LW = KS <= 8 ? 1 : 2, CS = fl_cb_stride<DS>();
    const uint32_t nitems = w.heads[SAMPLE ? 1 : 3];
    const uint4* items = SAMPLE ? w.items1 : w.items;
    const uint32_t* pairs = SAMPLE ? w.pairs1 : w.pairs;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (blockIdx.x >= nitems) return;
    if (threadIdx.x == 0) head = FL_WAVES;
    float* cbs = reinterpret_cast<float*>(smem);
    u32x4* onehot = reinterpret_cast<u32x4*>(smem + (size_t)ix.M * CS * 4);
    for (int i = threadIdx.x; i < ix.M * 16 * DS; i += FL_THREADS) cbs[i / (16 * DS) * CS + i % (16 * DS)] = ix.codebooks[i];
    if (threadIdx.x < 16) {
        const uint32_t c = threadIdx.x, b = 1u << (8 * (c & 3));
        onehot[c] = u32x4{c >> 2 == 0 ? b : 0u, c >> 2 == 1 ? b : 0u, c >> 2 == 2 ? b : 0u, c >> 2 == 3 ? b : 0u};
    }
    __syncthreads();
    FlWave& sw = reinterpret_cast<FlWave*>(smem + (size_t)ix.M * CS * 4 + 256)[wave];
    uint32_t it = blockIdx.x + gridDim.x * (uint32_t)__builtin_amdgcn_readfirstlane(wave);
    while (it < nitems) {
        const uint4 dn = items[it];
        const uint32_t l = __builtin_amdgcn_readfirstlane(dn.x), p0 = __builtin_amdgcn_readfirstlane(dn.y);
        const uint32_t np = __builtin_amdgcn_readfirstlane(dn.z), sg = __builtin_amdgcn_readfirstlane(dn.w);
        uint32_t nx = 0;
        if (lane == 0) nx = atomicAdd(&head, 1u);
        it = blockIdx.x + gridDim.x * (uint32_t)__builtin_amdgcn_readfirstlane(nx);
        uint32_t nt = ix.ltoff[l + 1] - ix.ltoff[l];
        if (SAMPLE) nt = min(nt, (uint32_t)w.tcap);
        const uint32_t s0 = sg & 255u, nseg = sg >> 8, per = (nt + nseg - 1) / nseg;
        const uint32_t tile0 = min(s0 * per, nt), tile1 = min(tile0 + per, nt);
        if (tile0 < tile1)  // np <= FL_PAIRS
            fl_item<KS, DS, LW, SAMPLE>(ix, a, w, cbs, onehot, sw, l, np, pairs[p0 + min((uint32_t)lane, np - 1u)], tile0,
                                        tile1);
    }
}

// Per query: the survivors in 256 bins by distance, those up to the bin that
// reaches k ranked by (distance, insertion index) and written.
__global__ __launch_bounds__(256) void fs_final_kernel(DevIndex ix, ScanArgs a, ListWs w) {
    __shared__ __align__(16) uint64_t keys[FL_RCAP];
    __shared__ uint32_t hist[256], misc[2];
    __shared__ float red[8];
    __shared__ uint32_t soff[1 << SL_SLOT_BITS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = blockIdx.x, P = a.P, kout = a.kout;
    const uint32_t total = w.scount[q];
    uint32_t* st = a.qstat + (size_t)q * QSTAT_WORDS;
    auto give_up = [&]() {  // left to the flagged scan
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
        misc[1] = 255u;
    }
    if (total > (uint32_t)w.cap) {
        give_up();
        return;
    }
    const uint2* sv = w.surv + (size_t)q * w.cap;
    const uint32_t tmask = (1u << w.tbits) - 1u;
    hist[tid] = 0u;
    for (int s = tid; s < P; s += 256) soff[s] = ix.offsets[min(a.probe[(size_t)q * P + s], (uint32_t)ix.L - 1u)];
    float mn = 3.0e38f, mx = -3.0e38f;
    for (uint32_t i = tid; i < total; i += 256) {
        const float x = __uint_as_float(sv[i].y);
        mn = fminf(mn, x);
        mx = fmaxf(mx, x);
    }
    for (int o = 32; o > 0; o >>= 1) {
        mn = fminf(mn, __shfl_xor(mn, o, 64));
        mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    }
    if (lane == 0) {
        red[wave] = mn;
        red[4 + wave] = mx;
    }
    __syncthreads();
    mn = fminf(fminf(red[0], red[1]), fminf(red[2], red[3]));
    mx = fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7]));
    const float sc = mx > mn ? 255.0f / (mx - mn) : 0.0f;
    auto bin = [&](float x) { return (uint32_t)fminf(fmaxf((x - mn) * sc, 0.0f), 255.0f); };
    for (uint32_t i = tid; i < total; i += 256) atomicAdd(&hist[bin(__uint_as_float(sv[i].y))], 1u);
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
    for (uint32_t i0 = 0; i0 < total; i0 += 256) {
        const uint32_t i = i0 + tid;
        const uint2 s = i < total ? sv[i] : make_uint2(0u, 0u);
        const bool take = i < total && bin(__uint_as_float(s.y)) <= bk;
        const int at = wave_append_slot(take, &misc[0]);
        if (take && at < FL_RCAP)
            keys[at] = cand_key(__uint_as_float(s.y), ix.list_ids[(size_t)soff[s.x >> w.tbits] + (s.x & tmask)]);
    }
    __syncthreads();
    const uint32_t n = misc[0];
    if (n > FL_RCAP) {
        give_up();
        return;
    }
    // each key to its rank, the number of smaller keys (all distinct)
    for (uint32_t i = tid; i < n; i += 256) {
        const uint64_t ki = keys[i];
        uint32_t r = 0, j = 0;
        for (; j + 4 <= n; j += 4) {
            const ulonglong2 x = *reinterpret_cast<const ulonglong2*>(keys + j);
            const ulonglong2 y = *reinterpret_cast<const ulonglong2*>(keys + j + 2);
            r += (x.x < ki ? 1u : 0u) + (x.y < ki ? 1u : 0u) + (y.x < ki ? 1u : 0u) + (y.y < ki ? 1u : 0u);
        }
        for (; j < n; j++) r += keys[j] < ki ? 1u : 0u;
        if (r < (uint32_t)kout) scan_emit(a, q, (int)r, ki, true);
    }
    for (int j = (int)n + tid; j < kout; j += 256) scan_emit(a, q, j, ~0ull, false);
}

template <int KS, int DS>
static void launch_fs(const DevIndex& ix, const ScanArgs& a, const ListWs& w, bool sample, hipStream_t s) {
    const size_t lds = (size_t)ix.M * fl_cb_stride<DS>() * 4 + 256 + FL_WAVES * sizeof(FlWave);
    auto k = sample ? fs_list_kernel<KS, DS, true> : fs_list_kernel<KS, DS, false>;
    ensure_dyn_lds((const void*)k, lds);
    hipLaunchKernelGGL(k, dim3(256), dim3(FL_THREADS), lds, s, ix, a, w);
}

template <int DS>
static void launch_fs_d(const DevIndex& ix, const ScanArgs& a, const ListWs& w, bool sample, hipStream_t s) {
    if (ix.M <= 16) launch_fs<4, DS>(ix, a, w, sample, s);
    else if (ix.M <= 32) launch_fs<8, DS>(ix, a, w, sample, s);
    else if (ix.M <= 52) launch_fs<13, DS>(ix, a, w, sample, s);
    else launch_fs<16, DS>(ix, a, w, sample, s);
}

void launch_fast_list(const DevIndex& ix, const ScanArgs& a, const ListWs& ws, hipStream_t s) {
    if (a.nq <= 0) return;
    ListWs w = ws;
    auto scores = [&](bool sample) {
        if (ix.ds == 4) launch_fs_d<4>(ix, a, w, sample, s);
        else if (ix.ds == 2) launch_fs_d<2>(ix, a, w, sample, s);
        else launch_fs_d<1>(ix, a, w, sample, s);
    };
    launch_list_pairs(ix, a, w, s);
    scores(true);
    launch_list_bound(a, w, s);
    scores(false);
    hipLaunchKernelGGL(fs_final_kernel, dim3(a.nq), dim3(256), 0, s, ix, a, w);
    launch_fastscan_flagged(ix, a, s);
}

}  // namespace vgpu
