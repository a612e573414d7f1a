// sample_nucleus.h - sampling without top-k over rows too long for one
// workgroup's registers (specification: sample.h), spread over the slices of
// the split kernel. Used by sample.hip.
//
// Why: the exact whole-row path streams such a row twice from one compute
// unit. A 128,256-logit row took it 97 us whatever the batch, while 37 rows
// are 19 MB, 4 us of HBM. Here every pass over the row is a launch over
// (slice, row) workgroups, and only the last, which touches about a thousand
// elements, is one workgroup per row. Passes after the first read the logits
// from L2 / Infinity Cache. Every sum is of integers, so the token does not
// depend on the split.
//
//  sample_split_kernel     slice maxima and exp sums (sample_core.h)
//  nucleus_weigh_kernel    the row maximum m, then w = rl_sample_weight(x - m):
//                          per bin of d = m - x (kNucBins over kBinSpan, a
//                          monotone map, so a bin is a run of the (x desc,
//                          index asc) order) when the row has a nucleus, per
//                          round of 256 elements when it has none
//  nucleus_edge_kernel     the bin where the cumulative weight reaches
//                          thr = ceil(p W) (every slice's workgroup adds the
//                          row's histograms up itself: 4 KiB a slice, less
//                          than another launch costs); per round, the weight
//                          in the bins above it; that bin's members
//  nucleus_pick_kernel     the boundary member among them, the round where the
//                          cumulative weight first exceeds the draw, and the
//                          element in it
// A row whose boundary bin holds more members than the lists take (massive
// ties), or whose maximum is not finite, takes the exact whole-row path in
// the last kernel.
// Measured, calls back to back, against split + exact path (us): 37 x 128,256
// at top-p 0.95 34.8 against 104.3 (the four kernels 4.5, 7.9, 13.2 and 9.2);
// 256 rows 118 against 127; 512 x 131,072 217 against 250; 1 x 50,257 19.4
// against 46.4; 64 x 128,256 at top-p 1 (no edge pass) 22.5 against 97.1.
// Bound: vector-ALU issue in the weigh and edge passes (18 instructions of
// weight per element, 4 cycles each), launch and dependent-load latency in
// the pick. So the weights are not computed before the histograms arrive
// (13.2 -> 14.1 us: more registers, no less issue).
#pragma once

#include "sample_core.h"

namespace {

constexpr int kNucBins = kMergeThreads;                // 512: one bin per thread
constexpr int kNucRounds = kSplitLen / 256;            // 32 rounds of 256 elements per slice
constexpr int kNucWaveRounds = kNucRounds / kMergeWaves;
constexpr int kNucMembers = 480;                       // boundary-bin members per slice
constexpr int kNucRowMembers = 2048;                   // ... and per row, in LDS
constexpr int kNucSubBins = kMergeThreads;
constexpr uint32_t kNucXcds = 8;

// A slice's part of the workspace, in place of its candidate list.
struct NucSlice {
    unsigned long long hist[kNucBins];
    unsigned long long rounds[kNucRounds];
    uint32_t members;           // in the boundary bin (> kNucMembers: not all listed)
    uint32_t bstar;             // slice 0: the row's boundary bin, ...
    unsigned long long above;   // ... the weight in the bins above it
    unsigned long long thr;     // ... and the nucleus threshold
    uint2 list[kNucMembers];    // (bits of x, index)
};
static_assert(sizeof(NucSlice) <= kCandStride * sizeof(uint2), "a slice's record fits its candidate list");
static_assert(kCandStride * sizeof(uint2) % 16 == 0, "records stay 16-byte aligned");

__device__ __forceinline__ NucSlice *nuc_slice(const SampleParams &p, uint32_t row, uint32_t split)
{
    return reinterpret_cast<NucSlice *>(p.cand + ((size_t)row * p.splits + split) * kCandStride);
}

// The (slice, row) of a workgroup. Workgroup b runs on XCD b % 8, each XCD
// with its own L2: a row's slices all go to XCD row % 8, in every pass and in
// the pick, so that the histograms and lists one pass leaves for the next,
// and (up to about 64 rows of 128,256) the logits, are read from the L2 that
// wrote them. False for a workgroup past the last row.
__device__ __forceinline__ bool nuc_place(const SampleParams &p, uint32_t &split, uint32_t &row)
{
    const uint32_t local = blockIdx.x / kNucXcds;
    split = local % p.splits;
    row = local / p.splits * kNucXcds + blockIdx.x % kNucXcds;
    return row < p.rows;
}

__device__ __forceinline__ bool nuc_trunc(float topp) { return topp > 0.f && topp < 1.f; }

// The row maximum from the slices' records (splits <= 64: one per lane).
__device__ __forceinline__ float nuc_row_max(const SampleParams &p, uint32_t row, int lane)
{
    float mx = -INFINITY;
    if ((uint32_t)lane < p.splits)
        mx = p.stats[(size_t)row * p.splits + lane].max_x;
    return wave_max(mx);
}

// Bin coordinate of x and the bin of a coordinate: monotone in x.
__device__ __forceinline__ float nuc_t(float m, float x) { return (m - x) * ((float)kNucBins / kBinSpan); }

__device__ __forceinline__ uint32_t nuc_bin(float t)
{
    return t < (float)(kNucBins - 1) ? (uint32_t)t : (uint32_t)(kNucBins - 1);
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
    if (nuc_place(p, split, row))
        split_slice(p, split, row, L);
}

__global__ __launch_bounds__(kMergeThreads) void nucleus_weigh_kernel(SampleParams p)
{
    __shared__ unsigned long long hist[kNucBins];
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
    const float m = nuc_row_max(p, row, lane);
    NucSlice *out = nuc_slice(p, row, split);
    if (!nuc_trunc(row_topp(p, row))) {
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
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kNucWaveRounds; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t w = nuc_weight(x[j][e] - m);
            if (w)
                atomicAdd(&hist[nuc_bin(nuc_t(m, x[j][e]))], (unsigned long long)w);
        }
    __syncthreads();
    out->hist[tid] = hist[tid];
}

__global__ __launch_bounds__(kMergeThreads) void nucleus_edge_kernel(SampleParams p)
{
    __shared__ BlockShared bs;
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
    const float m = nuc_row_max(p, row, lane);

    // the row's weight in bin tid, eight slices' loads in flight
    uint64_t own = 0;
    for (uint32_t s0 = 0; s0 < p.splits; s0 += 8) {
        uint64_t h[8];
#pragma unroll
        for (uint32_t k = 0; k < 8; k++)
            h[k] = nuc_slice(p, row, min(s0 + k, p.splits - 1))->hist[tid];
#pragma unroll
        for (uint32_t k = 0; k < 8; k++)
            own += s0 + k < p.splits ? h[k] : 0ull;
    }
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
    // t < lo: a bin above bstar's; lo <= t < hi: bin bstar. (bstar is never the
    // last bin, which holds no weight, so hi bounds it.)
    const float lo = (float)bstar, hi = (float)(bstar + 1u);
#pragma unroll
    for (int j = 0; j < kNucWaveRounds; j++) {
        uint32_t s = 0, tot = 0;
        uint64_t bal[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t w = nuc_weight(x[j][e] - m);
            const float t = nuc_t(m, x[j][e]);
            s += t < lo ? w : 0u;
            bal[e] = __ballot(t < hi) & ~__ballot(t < lo);
            tot += (uint32_t)__popcll(bal[e]);
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
    if (tid == 0) {
        out->members = bs.cnt[0];
        out->bstar = bstar;
        out->above = bs.sel64;
        out->thr = thr;
    }
}

struct NucLds {
    unsigned long long rounds[64 * kNucRounds];
    unsigned long long sub[kNucSubBins];
    unsigned long long key[kNucRowMembers];  // the boundary bin: composite keys and weights
    uint32_t w[kNucRowMembers];
    unsigned long long skey[kSubCap];        // the boundary sub-bin
    uint32_t sw[kSubCap];
};

// Finds, among the boundary bin's members (n of them in L.key / L.w), the one
// at which the weight ranked (x desc, index asc) reaches thr, given `above`
// in the bins above: tau its composite key, wp the weight up to and with it.
// The bin is cut into kNucSubBins sub-bins (monotone again); the members of
// the one where thr is reached are compared pairwise. False when that
// sub-bin holds more than kSubCap (ties).
__device__ __forceinline__ bool nuc_boundary(uint32_t n, uint32_t bstar, uint64_t above, uint64_t thr, float m,
                                             NucLds &L, BlockShared &bs, uint64_t &tau, uint64_t &wp)
{
    const uint32_t tid = threadIdx.x;
    auto sub_of = [&](uint64_t key) {
        const float f = (nuc_t(m, rl_key_float((uint32_t)(key >> 32))) - (float)bstar) * (float)kNucSubBins;
        return f < (float)(kNucSubBins - 1) ? (uint32_t)f : (uint32_t)(kNucSubBins - 1);
    };
    for (uint32_t e = tid; e < n; e += kMergeThreads)
        atomicAdd(&L.sub[sub_of(L.key[e])], (unsigned long long)L.w[e]);
    __syncthreads();
    const uint64_t own = L.sub[tid];  // one sub-bin per thread
    uint64_t total;
    const uint64_t excl = above + block_excl_scan_u64_inl(own, total, bs);
    if (excl < thr && excl + own >= thr) {  // exactly one thread
        bs.res64[0] = excl;
        bs.n = tid;
    }
    __syncthreads();
    const uint64_t sub_above = bs.res64[0];
    const uint32_t sb = bs.n;
    for (uint32_t e0 = 0; e0 < n; e0 += kMergeThreads) {
        const uint32_t e = e0 + tid;
        const bool take = e < n && sub_of(L.key[e]) == sb;
        const uint32_t pos = wave_append(take, &bs.cnt[1]);
        if (take && pos < (uint32_t)kSubCap) {
            L.skey[pos] = L.key[e];
            L.sw[pos] = L.w[e];
        }
    }
    __syncthreads();
    const uint32_t ns = bs.cnt[1];
    if (ns > (uint32_t)kSubCap)
        return false;
    if (tid < ns) {
        const uint64_t ck = L.skey[tid];
        uint64_t s = sub_above;
        for (uint32_t j = 0; j < ns; j++)
            s += L.skey[j] > ck ? (uint64_t)L.sw[j] : 0ull;
        if (s < thr && s + L.sw[tid] >= thr) {  // exactly one element
            bs.sel64 = ck;
            bs.res64[1] = s + L.sw[tid];
        }
    }
    __syncthreads();
    tau = bs.sel64;
    wp = bs.res64[1];
    return true;
}

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
    // the first 128 members of the lists this wave copies, before their
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
    uint32_t bstar = kNucBins;  // every bin is in the nucleus
    uint64_t tau = 0, wp = 0;
    uint32_t n = 0;
    if (trunc && ok) {
        bstar = head->bstar;
        const uint64_t above = head->above, thr = head->thr;
        const bool over = __ballot(cnt > (uint32_t)kNucMembers) != 0;
        const uint32_t incl = rl_wave_incl_scan_u32(over ? 0u : cnt);
        n = rl_readlane(incl, 63);
        ok = !over && n <= (uint32_t)kNucRowMembers;
        if (ok) {
            L.sub[tid] = 0;
            if (tid == 0)
                bs.cnt[1] = 0;
            // wave w copies the members of slices w, w + 8, ...
            for (uint32_t s = wave; s < p.splits; s += kMergeWaves) {
                const uint32_t c = rl_readlane(cnt, (int)s), at = rl_readlane(incl, (int)s) - c;
                const uint2 *src = nuc_slice(p, row, s)->list;
                for (uint32_t i = lane; i < c; i += 64) {
                    const uint2 v = s == (uint32_t)wave && i < 128u       ? (i < 64u ? pv[0] : pv[1])
                                    : s == (uint32_t)wave + kMergeWaves && i < 128u ? (i < 64u ? pv[2] : pv[3])
                                                                          : src[i];
                    const float xv = __uint_as_float(v.x);
                    L.key[at + i] = composite_key(rl_float_key(xv), v.y);
                    L.w[at + i] = nuc_weight(xv - m);
                }
            }
            __syncthreads();
            ok = nuc_boundary(n, bstar, above, thr, m, L, bs, tau, wp);
        }
        // the members in the nucleus join their rounds
        if (ok)
            for (uint32_t e = tid; e < n; e += kMergeThreads) {
                const uint64_t ck = L.key[e];
                if (ck >= tau)
                    atomicAdd(&L.rounds[(0xFFFFFFFFu - (uint32_t)ck) / 256u], (unsigned long long)L.w[e]);
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
                const uint32_t b = nuc_bin(nuc_t(m, x));
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
