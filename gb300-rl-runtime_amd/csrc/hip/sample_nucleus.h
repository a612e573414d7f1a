// sample_nucleus.h - sampling without top-k over rows too long for one
// workgroup's registers (specification: sample.h), spread over the slices of
// the split kernel. Used by sample.hip.
//
// Why: the exact whole-row path streams such a row twice from one compute
// unit. A 128,256-logit row took it 97 us whatever the batch, while 37 rows
// are 19 MB, 4 us of HBM. Here every pass over the row is a launch over
// (slice, row) workgroups, and only the last, which touches about a thousand
// elements, is one workgroup per row. Passes after the first read the logits
// from the Infinity Cache. Every sum is of integers, so the token does not
// depend on the split.
//
//  nucleus_split_kernel    slice maxima and exp sums (split_slice of
//                          sample_core.h); the row's histograms cleared
//  nucleus_weigh_kernel    the row maximum m, then w = rl_sample_weight(x - m):
//                          added up per bin of d = m - x (kNucBins over
//                          nuc_scale's span, a monotone map, so a bin is a run
//                          of the (x desc, index asc) order) when the row has
//                          a nucleus, per round of 256 elements when it has
//                          none
//  nucleus_edge_kernel     the bin where the cumulative weight reaches
//                          thr = ceil(p W); per round, the weight in the bins
//                          above it; that bin's members, listed per slice and
//                          added up per sub-bin (1/kNucBins of the bin)
//  nucleus_pick_kernel     the sub-bin where thr is reached and the boundary
//                          member in it, the round where the cumulative weight
//                          first exceeds the draw, and the element in it
// A slice whose members exceed its list is read again in the last kernel. A
// row whose boundary sub-bin holds more than one member per thread (ties), or
// whose maximum is not finite, takes the exact whole-row path there.
// Measured, calls back to back, against split + exact path (us): 37 x 128,256
// ~N(0, 1) at top-p 0.95 33.6 against 104.4 (the four kernels 5.2, 9.9, 11.9
// and 8.3), ~N(0, 0.3^2) at 0.9 33.0 against 107.9; 256 rows of those 112
// against 130; 64 x 262,144 ~N(0, 1) at 0.9 65.6 against 206, 64 x 524,288 118
// against 400; 512 x 131,072 203 against 250; 1 x 50,257 20.3 against 47.1; 64 x
// 128,256 at top-p 1 (no edge pass) 22.4 against 97.2; 37 x 128,256 ~N(0,
// 0.05^2) under five logits of 8 (every slice read again in the pick) 82
// against 685 (there the radix search).
// Bound: vector-ALU issue in the edge pass, 56 instructions a logit: 6.9 of its
// 11.9 us over the whole device, 9 on a compute unit with three of the 592
// workgroups; 5.0 of 9.9 us in the weigh pass (41 a logit), whose rest is the
// histogram's LDS atomics (0.13 conflict cycles a logit) and the device-wide
// ones. Launch and dependent-load latency in the pick, whose waves wait 70% of
// their cycles. So the weights are not computed before the histograms arrive
// (13.2 -> 14.1 us: more registers, no less issue).
#pragma once

#include "sample_core.h"

namespace {

constexpr int kNucBins = kMergeThreads;                // 512: one bin per thread
constexpr int kNucRounds = kSplitLen / 256;            // 32 rounds of 256 elements per slice
constexpr int kNucWaveRounds = kNucRounds / kMergeWaves;
constexpr int kNucMembers = 480;                       // boundary-bin members a slice lists
constexpr uint32_t kNucXcds = 8;
constexpr uint32_t kNucLast = 32;

// A slice's part of the workspace, in place of its candidate list. A row's
// weights are added up in two of its slices' records, by one device-wide
// atomic per bin and slice: per bin in slice 0's hist, per sub-bin of the
// boundary bin in slice 1's (these rows have five slices and more). So the
// later passes read 4 KiB a workgroup whatever the number of slices; each
// slice with its own histogram, and the edge pass adding them up, took 35.5
// us against 33.1 at 37 x 128,256 and reads slices^2 of them a row.
struct NucSlice {
    unsigned long long hist[kNucBins];
    unsigned long long rounds[kNucRounds];
    uint32_t members;           // in the boundary bin (> kNucMembers: not all listed)
    uint32_t bstar;             // slice 0: the row's boundary bin, ...
    unsigned long long above;   // ... the weight in the bins above it
    unsigned long long thr;     // ... the nucleus threshold
    float scale;                // ... and its bins per unit of d (nuc_scale)
    uint32_t pad;
    uint2 list[kNucMembers];    // (bits of x, index)
};
static_assert(sizeof(NucSlice) <= kCandStride * sizeof(uint2), "a slice's record fits its candidate list");
static_assert(kCandStride * sizeof(uint2) % 16 == 0, "records stay 16-byte aligned");
static_assert(RL_ROW_SAMPLER_VOCAB >= kSplitLen, "longer rows have a slice 1");

__device__ __forceinline__ NucSlice *nuc_slice(const SampleParams &p, uint32_t row, uint32_t split)
{
    return reinterpret_cast<NucSlice *>(p.cand + ((size_t)row * p.splits + split) * kCandStride);
}

// The (slice, row) of a workgroup. Workgroup b runs on XCD b % 8: a row's
// slices all go to XCD row % 8, in every pass and in the pick. (Each pass
// still fetches its 19 MB of logits at 37 rows from beyond the L2s.) False for
// a workgroup past the last row.
__device__ __forceinline__ bool nuc_place(const SampleParams &p, uint32_t &split, uint32_t &row)
{
    const uint32_t local = blockIdx.x / kNucXcds;
    split = local % p.splits;
    row = local / p.splits * kNucXcds + blockIdx.x % kNucXcds;
    return row < p.rows;
}

__device__ __forceinline__ bool nuc_trunc(float topp) { return topp > 0.f && topp < 1.f; }

// The row maximum and the sum of exp(x - max) from the slices' records
// (splits <= 64: one per lane).
__device__ __forceinline__ void nuc_row(const SampleParams &p, uint32_t row, int lane, float &m, float &z)
{
    float mx = -INFINITY, zs = 0.f;
    if ((uint32_t)lane < p.splits) {
        mx = p.stats[(size_t)row * p.splits + lane].max_x;
        zs = p.stats[(size_t)row * p.splits + lane].sum_exp;
    }
    m = wave_max(mx);
    z = wave_sum(mx == -INFINITY ? 0.f : zs * exp2f((mx - m) * 1.4426950408889634f));
}

// Bins per unit of d. The elements past d = D weigh at most V e^-D together,
// which is below the (1 - p) z outside the nucleus from D = ln(V / ((1 - p) z))
// on: the bins span that much (an eighth more, for the roundings) and the last
// one takes the rest, so that they are as narrow as the row's spread allows
// (128,256 logits ~N(0, 0.3^2) at p 0.9 span 3.7: 800 members in the boundary
// bin, 3,600 with a span of 17 for every row).
__device__ __forceinline__ float nuc_scale(float z, uint32_t vocab, float topp)
{
    const float span = fminf(logf((float)vocab / (z * (1.0f - topp))) + 0.125f, kBinSpan);
    return (float)(kNucBins - 1) / fmaxf(span, 0.125f);
}

// Bin coordinate of x, the bin of a coordinate and the sub-bin of a coordinate
// in bin b: all monotone in x (t - b is exact or monotone, and the factor a
// power of two).
__device__ __forceinline__ float nuc_t(float m, float x, float scale) { return (m - x) * scale; }

__device__ __forceinline__ uint32_t nuc_bin(float t)
{
    return t < (float)(kNucBins - 1) ? (uint32_t)t : (uint32_t)(kNucBins - 1);
}

__device__ __forceinline__ uint32_t nuc_sub(float t, uint32_t b) { return nuc_bin((t - (float)b) * (float)kNucBins); }

// Bin b is the coordinates from b to below nuc_end(b); the last one is open.
__device__ __forceinline__ float nuc_end(uint32_t b)
{
    return b < (uint32_t)(kNucBins - 1) ? (float)(b + 1u) : INFINITY;
}

__device__ __forceinline__ void nuc_add(unsigned long long *to, unsigned long long v)
{
    if (v)
        (void)__hip_atomic_fetch_add(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// This wave's rounds of the slice: round j of the wave is elements
// [i0 + 256 j, + 256) with i0 = slice start + 256 kNucWaveRounds wave, lane l
// the quad at 4 l, so every load instruction reads 1 KiB of consecutive
// logits; all of them in flight together. Past the vocabulary: -inf.
__device__ __forceinline__ void nuc_load(const SampleParams &p, uint32_t row, uint32_t first, float inv_t,
                                         float (&x)[kNucWaveRounds][4])
{
    const float *l = p.logits + (size_t)row * p.row_stride;
    rl_f32x4 raw[kNucWaveRounds];
#pragma unroll
    for (int j = 0; j < kNucWaveRounds; j++)
        raw[j] = load_quad(l, first + 256u * j, p.vocab);
#pragma unroll
    for (int j = 0; j < kNucWaveRounds; j++)
#pragma unroll
        for (int e = 0; e < 4; e++)
            x[j][e] = quad_at(raw[j], e) * inv_t;
}

__device__ __forceinline__ uint32_t nuc_weight(float d)
{
    float f;
    return rl_sample_weight_f(d, &f);
}

// Sum over the wave of a value of at most 2^26 per lane.
__device__ __forceinline__ uint64_t nuc_wave_sum(uint32_t s)
{
    return ((uint64_t)rl_wave_sum_u32(s >> 8) << 8) + rl_wave_sum_u32(s & 0xFFu);
}

__global__ __launch_bounds__(kThreads) void nucleus_split_kernel(SampleParams p)
{
    __shared__ SplitLds L;
    uint32_t split, row;
    if (!nuc_place(p, split, row))
        return;
    if (split < 2 && nuc_trunc(row_topp(p, row))) {
        unsigned long long *h = nuc_slice(p, row, split)->hist;
#pragma unroll
        for (int k = 0; k < kNucBins / kThreads; k++)
            h[threadIdx.x + k * kThreads] = 0;
    }
    split_slice(p, split, row, L);
}

__global__ __launch_bounds__(kMergeThreads) void nucleus_weigh_kernel(SampleParams p)
{
    // (the last bin, which may hold a quarter of a peaked row's elements, is
    // kept kNucLast times, lane l's elements in copy l % kNucLast)
    __shared__ unsigned long long hist[kNucBins - 1 + kNucLast];
    uint32_t split, row;
    if (!nuc_place(p, split, row))
        return;
    const uint32_t tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const float temp = row_temperature(p, row);
    if (!(temp > 0.f))
        return;  // a greedy row: its slices' argmaxima are enough
    const uint32_t first = split * kSplitLen + (uint32_t)wave * (256u * kNucWaveRounds) + (uint32_t)lane * 4u;
    float x[kNucWaveRounds][4];
    nuc_load(p, row, first, 1.0f / temp, x);
    hist[tid] = 0;
    if (tid < kNucLast - 1)
        hist[kNucBins + tid] = 0;
    float m, z;
    nuc_row(p, row, lane, m, z);
    const float topp = row_topp(p, row);
    NucSlice *out = nuc_slice(p, row, split);
    if (!nuc_trunc(topp)) {
#pragma unroll
        for (int j = 0; j < kNucWaveRounds; j++) {
            uint32_t s = 0;  // at most 4 x 2^24
#pragma unroll
            for (int e = 0; e < 4; e++)
                s += nuc_weight(x[j][e] - m);
            const uint64_t sum = nuc_wave_sum(s);
            if (lane == 0)
                out->rounds[wave * kNucWaveRounds + j] = sum;
        }
        return;
    }
    const float scale = nuc_scale(z, p.vocab, topp);
    if (tid == 0 && split == 0)
        out->scale = scale;
    __syncthreads();
    const float lane_last = (float)(kNucBins - 1 + (lane & (kNucLast - 1)));
#pragma unroll
    for (int j = 0; j < kNucWaveRounds; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t w = nuc_weight(x[j][e] - m);
            if (w)
                atomicAdd(&hist[(uint32_t)fminf(nuc_t(m, x[j][e], scale), lane_last)], (unsigned long long)w);
        }
    __syncthreads();
    uint64_t own = hist[tid];
    if (wave == kMergeWaves - 1) {  // thread kNucBins - 1: the sum of the last bin's copies
        const uint64_t sum = wave_inclusive_scan_u64(lane < (int)kNucLast ? hist[kNucBins - 1 + lane] : 0ull);
        own = lane == 63 ? sum : own;
    }
    nuc_add(&nuc_slice(p, row, 0)->hist[tid], own);
}

__global__ __launch_bounds__(kMergeThreads) void nucleus_edge_kernel(SampleParams p)
{
    __shared__ BlockShared bs;
    __shared__ unsigned long long sub[kNucBins];
    uint32_t split, row;
    if (!nuc_place(p, split, row))
        return;
    const uint32_t tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const float temp = row_temperature(p, row);
    const float topp = row_topp(p, row);
    if (!(temp > 0.f) || !nuc_trunc(topp))
        return;
    const uint32_t first = split * kSplitLen + (uint32_t)wave * (256u * kNucWaveRounds) + (uint32_t)lane * 4u;
    float x[kNucWaveRounds][4];
    nuc_load(p, row, first, 1.0f / temp, x);
    float m, z;
    nuc_row(p, row, lane, m, z);
    const float scale = nuc_slice(p, row, 0)->scale;
    const uint64_t own = nuc_slice(p, row, 0)->hist[tid];
    sub[tid] = 0;
    uint64_t wk;
    if (tid == 0) {
        bs.cnt[0] = 0;
        bs.n = kNucBins;  // no weight at all (no finite maximum): no bin
        bs.sel64 = 0;
    }
    const uint64_t excl = block_excl_scan_u64_inl(own, wk, bs);
    const uint64_t thr = rl_topp_threshold(topp, wk);
    if (excl < thr && excl + own >= thr) {  // exactly one thread, when wk > 0
        bs.n = tid;
        bs.sel64 = excl;
    }
    __syncthreads();
    const uint32_t bstar = bs.n;

    NucSlice *out = nuc_slice(p, row, split);
    const float lo = (float)bstar, hi = nuc_end(bstar);  // t < lo: a bin above; lo <= t < hi: bin bstar
#pragma unroll
    for (int j = 0; j < kNucWaveRounds; j++) {
        uint32_t s = 0, tot = 0;
        uint64_t bal[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t w = nuc_weight(x[j][e] - m);
            const float t = nuc_t(m, x[j][e], scale);
            s += t < lo ? w : 0u;
            bal[e] = __ballot(t < hi) & ~__ballot(t < lo);
            tot += (uint32_t)__popcll(bal[e]);
            if (bal[e] >> lane & 1)
                atomicAdd(&sub[nuc_sub(t, bstar)], (unsigned long long)w);
        }
        if (tot) {  // one LDS atomic per wave and round
            uint32_t at = 0;
            if (lane == 0)
                at = atomicAdd(&bs.cnt[0], tot);
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (bal[e] == 0)
                    continue;
                const uint32_t pos = at + __builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(bal[e] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal[e], 0u));
                if ((bal[e] >> lane & 1) && pos < (uint32_t)kNucMembers)
                    out->list[pos] = make_uint2(__float_as_uint(x[j][e]), first + 256u * j + e);
                at += (uint32_t)__popcll(bal[e]);
            }
        }
        const uint64_t sum = nuc_wave_sum(s);
        if (lane == 0)
            out->rounds[wave * kNucWaveRounds + j] = sum;
    }
    __syncthreads();
    nuc_add(&nuc_slice(p, row, 1)->hist[tid], sub[tid]);
    if (tid == 0) {
        out->members = bs.cnt[0];
        out->bstar = bstar;
        out->above = bs.sel64;
        out->thr = thr;
    }
}

struct NucLds {
    unsigned long long rounds[64 * kNucRounds];
    unsigned long long key[kMergeThreads];  // the boundary sub-bin: composite keys and weights
    uint32_t w[kMergeThreads];
};

// Grid (row).
__global__ __launch_bounds__(kMergeThreads) void nucleus_pick_kernel(SampleParams p)
{
    __shared__ union {
        NucLds n;
        RowScratch x;  // the exact whole-row path
    } lds;
    __shared__ uint32_t s_hist[256];
    __shared__ unsigned long long s_whist[256];
    __shared__ BlockShared bs;
    NucLds &L = lds.n;
    const uint32_t row = blockIdx.x, tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const SplitStat *st = p.stats + (size_t)row * p.splits;
    const float temp = row_temperature(p, row);
    if (!(temp > 0.f)) {
        greedy_merge_row(p, row, lane, tid == 0);
        return;
    }
    const float inv_t = 1.0f / temp;
    const float topp = row_topp(p, row);
    const bool trunc = nuc_trunc(topp);
    const uint64_t draw = st[0].draw;
    const NucSlice *head = nuc_slice(p, row, 0);
    const uint32_t R = p.splits * kNucRounds;
    for (uint32_t r = tid; r < R; r += kMergeThreads)
        L.rounds[r] = nuc_slice(p, row, r / kNucRounds)->rounds[r % kNucRounds];
    // the first 128 members of the lists this wave reads first, before their
    // counts are known (in bounds; past a list's count, not used)
    uint2 pv[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        pv[k] = nuc_slice(p, row, min((uint32_t)(wave + k / 2 * kMergeWaves), p.splits - 1))->list[k % 2 * 64 + lane];
    float mx = -INFINITY, zs = 0.f;
    uint32_t cnt = 0;
    if ((uint32_t)lane < p.splits) {
        mx = st[lane].max_x;
        zs = st[lane].sum_exp;
        if (trunc)
            cnt = nuc_slice(p, row, lane)->members;
    }
    const float m = wave_max(mx);
    const float *l = p.logits + (size_t)row * p.row_stride;

    bool ok = m > -INFINITY && m < INFINITY;
    float scale = 0.f;
    uint32_t bstar = kNucBins;  // every bin is in the nucleus
    uint64_t tau = 0, wp = 0;
    if (trunc && ok) {
        scale = head->scale;
        bstar = head->bstar;
        const float lo = (float)bstar, hi = nuc_end(bstar);
        const uint64_t above = head->above, thr = head->thr;
        // ---- the sub-bin of the boundary bin where thr is reached -----------
        if (tid == 0)
            bs.cnt[1] = 0;
        const uint64_t own = nuc_slice(p, row, 1)->hist[tid];
        uint64_t total;
        const uint64_t excl = above + block_excl_scan_u64_inl(own, total, bs);
        if (excl < thr && excl + own >= thr) {  // exactly one thread
            bs.res64[0] = excl;
            bs.n = tid;
        }
        __syncthreads();
        const uint64_t sub_above = bs.res64[0];
        const uint32_t sb = bs.n;
        // ---- the bin's members: those in the sub-bins above join their
        // rounds, those in the sub-bin are gathered ---------------------------
        auto member = [&](float x, uint32_t idx) {
            const uint32_t sub = nuc_sub(nuc_t(m, x, scale), bstar);
            const uint32_t w = nuc_weight(x - m);
            if (sub < sb)
                atomicAdd(&L.rounds[idx / 256u], (unsigned long long)w);
            const bool edge = sub == sb && w != 0;
            const uint32_t pos = wave_append(edge, &bs.cnt[1]);
            if (edge && pos < (uint32_t)kMergeThreads) {
                L.key[pos] = composite_key(rl_float_key(x), idx);
                L.w[pos] = w;
            }
        };
        for (uint32_t s = wave; s < p.splits; s += kMergeWaves) {  // wave w: slices w, w + 8, ...
            const uint32_t c = rl_readlane(cnt, (int)s);
            if (c <= (uint32_t)kNucMembers) {
                const uint2 *src = nuc_slice(p, row, s)->list;
                for (uint32_t i = lane; i < c; i += 64) {
                    const uint2 v = s == (uint32_t)wave && i < 128u       ? (i < 64u ? pv[0] : pv[1])
                                    : s == (uint32_t)wave + kMergeWaves && i < 128u ? (i < 64u ? pv[2] : pv[3])
                                                                          : src[i];
                    member(__uint_as_float(v.x), v.y);
                }
            } else {
                const uint32_t i0 = s * (uint32_t)kSplitLen + (uint32_t)lane * 4u;
                for (uint32_t r = 0; r < (uint32_t)kNucRounds; r += kNucWaveRounds) {
                    float x[kNucWaveRounds][4];
                    nuc_load(p, row, i0 + 256u * r, inv_t, x);
#pragma unroll
                    for (int j = 0; j < kNucWaveRounds; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const float t = nuc_t(m, x[j][e], scale);
                            if (t < hi && !(t < lo))
                                member(x[j][e], i0 + 256u * (r + j) + e);
                        }
                }
            }
        }
        __syncthreads();
        const uint32_t ns = bs.cnt[1];
        ok = ns <= (uint32_t)kMergeThreads;
        if (ok) {
            // ---- the boundary element: compared pairwise --------------------
            if (tid < ns) {
                const uint64_t ck = L.key[tid];
                uint64_t s = sub_above;
                for (uint32_t j = 0; j < ns; j++)
                    s += L.key[j] > ck ? (uint64_t)L.w[j] : 0ull;
                if (s < thr && s + L.w[tid] >= thr) {  // exactly one element
                    bs.sel64 = ck;
                    bs.res64[1] = s + L.w[tid];
                }
            }
            __syncthreads();
            tau = bs.sel64;
            wp = bs.res64[1];
            if (tid < ns && L.key[tid] >= tau)
                atomicAdd(&L.rounds[(0xFFFFFFFFu - (uint32_t)L.key[tid]) / 256u], (unsigned long long)L.w[tid]);
        }
    }
    __syncthreads();

    uint32_t tok = 0;
    if (ok) {
        // ---- the round where the cumulative weight first exceeds the draw ----
        const uint32_t per = (R + kMergeThreads - 1) / kMergeThreads;
        const uint32_t r0 = min(R, tid * per), r1 = min(R, r0 + per);
        uint64_t own = 0, total;
        for (uint32_t r = r0; r < r1; r++)
            own += L.rounds[r];
        const uint64_t excl = block_excl_scan_u64_inl(own, total, bs);
        const uint64_t u = rl_mulhi_u64(draw, trunc ? wp : total);  // (total is W_P either way)
        if (excl <= u && u < excl + own) {  // exactly one thread: u < W_P
            uint64_t c = excl;
            uint32_t r = r0;
            while (c + L.rounds[r] <= u) {
                c += L.rounds[r];
                r++;
            }
            bs.n = r;
            bs.sel64 = c;
        }
        __syncthreads();
        // ---- the element in it -----------------------------------------------
        const uint32_t i0 = bs.n * 256u + (uint32_t)lane * 4u;
        if (wave == 0) {
            const rl_f32x4 v = load_quad(l, i0, p.vocab);
            uint32_t w4[4], mine = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x = quad_at(v, e) * inv_t;
                const uint32_t b = trunc ? nuc_bin(nuc_t(m, x, scale)) : 0u;
                const uint64_t ck = composite_key(rl_float_key(x), i0 + e);
                const uint32_t in = (uint32_t)(b < bstar) | ((uint32_t)(b == bstar) & (uint32_t)(ck >= tau));
                w4[e] = nuc_weight(x - m) & (0u - in);
                mine += w4[e];
            }
            uint64_t c = bs.sel64 + wave_inclusive_scan_u64(mine) - mine;
            uint32_t cand = 0xFFFFFFFFu;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                c += w4[e];
                if (cand == 0xFFFFFFFFu && c > u)
                    cand = i0 + e;
            }
            tok = rl_wave_min_u32(cand);
        }
    } else {
        tok = exact_row_sample(p, row, inv_t, 0u, topp, m, lds.x, s_hist, s_whist, bs);
    }
    if (tid < 64) {
        const float zterm = (mx == -INFINITY) ? 0.f : zs * exp2f((mx - m) * 1.4426950408889634f);
        const float lse = m + logf(wave_sum(zterm));
        if (tid == 0) {
            p.token_out[row] = tok;
            p.logprob_out[row] = l[tok] * inv_t - lse;
        }
    }
}

}  // namespace
