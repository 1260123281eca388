// The sampler's candidates (kernels.hpp:434-447 top_tokens / penalize_row, topk.cuh): per row of the head's logits the
// row's logit_bias and penalties applied in place (repeat multiplies a non-positive logit and divides a positive one,
// then frequency x count and presence once), then its 64 highest, ordered by logit (descending) and token id (ascending)
// on ties, however many tie. err bit 16: a logit was NaN or inf before the penalties.
//
// The reference ranks a row in one block (radix passes over the whole row). Here a row is cut into slices of 2,560
// logits, one block each, so a window's rows fill the chip: a block keeps its slice's 64 best, a second launch keeps the
// 64 best of a row's slices and sorts them. "The 64 best" is always the same selection by a wave over the values its
// lanes hold: the threshold key found by halving (counting in the wave: no memory traffic), ties at the threshold taken by
// lowest id bit by bit; every (key, id) pair is distinct, so the result does not depend on how the row was cut.
#pragma once

#include "k_moe_layer.h"

namespace fnx {

constexpr int SM_N = 64;                                                    // candidates a row (kernels.hpp:440 TOPK_N)
constexpr int SM_THREADS = 256, SM_V = 10, SM_SLICE = SM_THREADS * SM_V;   // a block's slice: 2,560 logits
constexpr int SM_PEN_STEP = 4;                                               // a thread's penalized tokens in flight
constexpr int SM_PEN_CAP = 4096;                                            // penalized tokens a row, at most (engine.hpp:73 PEN_CAP)
constexpr int SM_MAXS = 128;                                                // slices a row, at most (327,680 logits)
constexpr int SM_MERGE_THREADS = 1024, SM_MERGE_V = SM_MAXS * SM_N / SM_MERGE_THREADS;   // 8 candidates a lane
// the slices' candidates between the two launches: one top_tokens in flight per device
__device__ unsigned long long g_topk_cand[FNX_MAXT * SM_MAXS * SM_N];

// order-preserving key of a float's bits: a larger float, a larger key (topk.cuh:13-16)
__device__ __forceinline__ unsigned tk_key(float v) {
    const unsigned u = __float_as_uint(v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// a small count summed over the wave's lanes with DPP adds; every lane gets the total. (Counting with a ballot a value
// costs a trip from the vector to the scalar unit each, one after another through the one condition register.)
__device__ __forceinline__ int wave_total(int v) {
#define FNX_DPP_ADDI(ctrl, rmask) v += __builtin_amdgcn_update_dpp(0, v, ctrl, rmask, 0xF, false)
    FNX_DPP_ADDI(0xB1, 0xF);    // quad_perm [1,0,3,2]
    FNX_DPP_ADDI(0x4E, 0xF);    // quad_perm [2,3,0,1]
    FNX_DPP_ADDI(0x141, 0xF);   // row_half_mirror
    FNX_DPP_ADDI(0x140, 0xF);   // row_mirror
    FNX_DPP_ADDI(0x142, 0xA);   // row_bcast15 into rows 1 and 3
    FNX_DPP_ADDI(0x143, 0xC);   // row_bcast31 into rows 2 and 3
#undef FNX_DPP_ADDI
    return __builtin_amdgcn_readlane(v, 63);
}

// The 64 greatest of a wave's 64 V (key, idf) pairs, as a mask of each lane's slots. Real pairs are distinct and have
// idf != 0 (idf = 0xffffffff - id); empty slots are (0, 0), lose to every real pair and are only "selected" by being
// left over when fewer than 64 pairs are real. Greater key first, then greater idf (= the lower id).
// The threshold is looked for by halving between the least of the lanes' greatest keys (64 keys, one a lane, are no smaller) and
// the greatest key of all: a slice's best lie within a few powers of two, some 2^24 keys, of which a search by the keys' bits from
// the top would take the first seven or eight steps for nothing (16 rows of 151,936 logits: the slices 12.8 -> 11.4 us, their
// merge 9.7 -> 9.1; the sampled head of 5 rows 110.2 -> 107.8).
template <int V>
__device__ __forceinline__ unsigned wave_select64(const unsigned (&key)[V], const unsigned (&idf)[V]) {
    // 64 real pairs or fewer (a short tail slice, a wave past the row's end): all of them
    int mine = 0;
    unsigned all = 0;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        mine += idf[v] != 0u;
        all |= (idf[v] != 0u ? 1u : 0u) << v;
    }
    const int real = wave_total(mine);
    if (real <= SM_N) return all;
    const auto count_ge = [&](unsigned th) {
        int c = 0;
#pragma unroll
        for (int v = 0; v < V; ++v) c += key[v] >= th;
        return wave_total(c);
    };
    // the greatest k with at least 64 keys >= k; a threshold with exactly 64 at or above it ends the search
    unsigned top = key[0];
#pragma unroll
    for (int v = 1; v < V; ++v) top = max(top, key[v]);
    unsigned k = ~wave_umax(~top), hi = wave_umax(top);
    // With little more than 64 real pairs there are often just 64 at the lower end itself, which halving comes to last: there the
    // key after the lower end is tried first (one row of 2,561 logits 19.1 -> 14.5 us, 16.3 bit by bit; tried everywhere it
    // costs 1.4 us of 20)
    unsigned shift = real < 2 * SM_N ? 31u : 1u;
    while (k < hi) {
        const unsigned th = k + 1u + ((hi - k - 1u) >> shift);   // k < th <= hi
        const int c = count_ge(th);
        shift = 1u;
        if (c == SM_N) {
            unsigned sel = 0;
#pragma unroll
            for (int v = 0; v < V; ++v) sel |= (key[v] >= th ? 1u : 0u) << v;
            return sel;
        }
        if (c > SM_N) k = th;
        else hi = th - 1u;
    }
    // more than 64 keys >= k, fewer than 64 above it: the rest come from the pairs at k, the greatest idf first
    int above = 0, at = 0;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        above += key[v] > k;
        at += key[v] == k;
    }
    above = wave_total(above);
    at = wave_total(at);
    const int want = SM_N - above;
    unsigned f = 0;   // all of them: every idf >= 0
    if (at > want) {
        // the greatest f with at least `want` pairs (k, idf >= f): idfs are distinct, so exactly `want` at the end
        for (unsigned bit = 0x80000000u; bit; bit >>= 1) {
            int c = 0;
#pragma unroll
            for (int v = 0; v < V; ++v) c += key[v] == k && idf[v] >= (f | bit);
            c = wave_total(c);
            if (c >= want) f |= bit;
            if (c == want) break;
        }
    }
    unsigned sel = 0;
#pragma unroll
    for (int v = 0; v < V; ++v) sel |= (key[v] > k || (key[v] == k && idf[v] >= f) ? 1u : 0u) << v;
    return sel;
}
// the selected pairs, packed (key << 32 | idf), to out[0 .. 64) in (slot, lane) order
template <int V>
__device__ __forceinline__ void wave_emit64(const unsigned (&key)[V], const unsigned (&idf)[V], unsigned sel, unsigned long long* out) {
    const int lane = threadIdx.x & 63;
    int base = 0;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const bool on = (sel >> v) & 1u;
        const unsigned long long b = __ballot(on);
        if (on) out[base + __popcll(b & ((1ull << lane) - 1ull))] = (unsigned long long) key[v] << 32 | idf[v];
        base += __popcll(b);
    }
    if (base + lane < SM_N) out[base + lane] = 0ull;   // fewer than 64 real pairs: the rest are empty
}

struct TopArgs {
    float* logits;
    int n, v0, nslice;
    const int *pen_tok, *pen_cnt, *pen_n;
    int pen_stride;
    const float* pen_par;
    const int* bias_tok;
    const float* bias_val;
    const int *bias_off, *bias_n;
    unsigned* err;
};
// launch 1: block (slice, row). Bound by its trips to memory and the selections' steps one after the other: 5 rows of
// 151,936 logits, 600 penalised tokens each, 14.5 -> 11.5 us with the penalties' loads together and beside the logits', 9.7 with the threshold halved.
__global__ void __launch_bounds__(SM_THREADS) k_top_slices(const TopArgs a) {
    __shared__ float vals[SM_SLICE];
    __shared__ unsigned long long cand[SM_THREADS / 64][SM_N];
    const int row = blockIdx.y, s = blockIdx.x, tid = threadIdx.x, wave = uniform(tid >> 6);
    const int i0 = s * SM_SLICE, len = min(SM_SLICE, a.n - i0);
    float* L = a.logits + (size_t) row * a.n + i0;
    float x[SM_V];
#pragma unroll
    for (int v = 0; v < SM_V; ++v) x[v] = L[min(v * SM_THREADS + tid, len - 1)];
    const int nb = a.bias_n ? min(max(a.bias_n[row], 0), SM_PEN_CAP) : 0, np = a.pen_n ? min(max(a.pen_n[row], 0), a.pen_stride) : 0;
    // the penalised tokens SM_PEN_STEP at a time, the first of them asked for with the logits (a list walked entry by entry,
    // and once more to write the row, was ten trips to memory one after the other for 600 tokens)
    int ptok[SM_PEN_STEP], pcnt[SM_PEN_STEP];
    auto pens = [&](int p0) {
#pragma unroll
        for (int k = 0; k < SM_PEN_STEP; ++k) {
            const size_t at = (size_t) row * a.pen_stride + min(p0 + k * SM_THREADS + tid, np - 1);
            ptok[k] = a.pen_tok[at];
            pcnt[k] = a.pen_cnt[at];
        }
    };
    float repeat = 1.f, freq = 0.f, present = 0.f;
    if (np) {
        pens(0);
        repeat = a.pen_par[row * 3], freq = a.pen_par[row * 3 + 1], present = a.pen_par[row * 3 + 2];
    }
    bool bad = false;
#pragma unroll
    for (int v = 0; v < SM_V; ++v) {
        const int i = v * SM_THREADS + tid;
        if (i >= len) x[v] = 0.f;
        bad = bad || !isfinite(x[v]);
        vals[i] = x[v];
    }
    if (__any(bad) && (tid & 63) == 0) atomicOr(a.err, 16u);
    __syncthreads();
    // the row's logit_bias on this slice's tokens (each token once in a list), before its penalties (topk.cuh:31-37)
    if (nb) {   // (the same for the whole block)
        for (int i = tid; i < nb; i += SM_THREADS) {
            const int at = a.bias_off[row] + i, tok = a.bias_tok[at] - a.v0 - i0;
            if (tok >= 0 && tok < len) vals[tok] += a.bias_val[at];
        }
        __syncthreads();
    }
    for (int p0 = 0; p0 < np; p0 += SM_PEN_STEP * SM_THREADS) {
        if (p0) pens(p0);
#pragma unroll
        for (int k = 0; k < SM_PEN_STEP; ++k) {
            const int tok = ptok[k] - a.v0 - i0, cnt = pcnt[k];
            if (p0 + k * SM_THREADS + tid >= np || tok < 0 || tok >= len || cnt <= 0) continue;
            float l = vals[tok];
            l = l <= 0.f ? l * repeat : l / repeat;
            l = l - (float) cnt * freq - present;
            vals[tok] = l;
            if (!nb) L[tok] = l;   // the changed logits go back to the row (the operator changes it in place)
        }
    }
    __syncthreads();
    if (nb) {   // (a token may be in both lists: the row is written when both have been applied)
        for (int i = tid; i < nb; i += SM_THREADS) {
            const int tok = a.bias_tok[a.bias_off[row] + i] - a.v0 - i0;
            if (tok >= 0 && tok < len) L[tok] = vals[tok];
        }
        for (int i = tid; i < np; i += SM_THREADS) {
            const int tok = a.pen_tok[(size_t) row * a.pen_stride + i] - a.v0 - i0;
            if (tok >= 0 && tok < len) L[tok] = vals[tok];
        }
    }
    unsigned key[SM_V], idf[SM_V];
#pragma unroll
    for (int v = 0; v < SM_V; ++v) {
        const int i = v * SM_THREADS + tid;
        key[v] = i < len ? tk_key(vals[i]) : 0u;
        idf[v] = i < len ? 0xffffffffu - (unsigned) (i0 + i) : 0u;
    }
    wave_emit64<SM_V>(key, idf, wave_select64<SM_V>(key, idf), cand[wave]);
    __syncthreads();
    if (wave != 0) return;
    constexpr int W = SM_THREADS / 64;
    unsigned k2[W], f2[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const unsigned long long c = cand[j][tid];
        k2[j] = (unsigned) (c >> 32);
        f2[j] = (unsigned) c;
    }
    wave_emit64<W>(k2, f2, wave_select64<W>(k2, f2), g_topk_cand + ((size_t) row * a.nslice + s) * SM_N);
}
// launch 2: a block per row: the 64 best of its slices' candidates, sorted. The same rows: 12.7 -> 9.5 us with the
// search between two ends and places counted instead of a sorting network. V: candidates a lane, no more than the row's slices
// make, since the search goes through all of them at every step (both launches over 5 rows, us, always eight / as many as needed: 32,000
// logits 17.1 / 16.7, 81,920 19.9 / 19.2, 151,936 20.7 / 19.9, 163,840 21.3 / 20.1).
template <int V>
__global__ void __launch_bounds__(SM_MERGE_THREADS) k_top_merge(const float* __restrict__ logits, int n, int v0, int nslice, float* __restrict__ out_v,
                                                               int* __restrict__ out_i) {
    __shared__ unsigned long long cand[SM_MERGE_THREADS / 64][SM_N];
    const int row = blockIdx.x, tid = threadIdx.x, wave = uniform(tid >> 6), lane = tid & 63;
    const unsigned long long* C = g_topk_cand + (size_t) row * nslice * SM_N;
    const int total = nslice * SM_N;
    {
        unsigned key[V], idf[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const int i = v * SM_MERGE_THREADS + tid;
            const unsigned long long c = i < total ? C[i] : 0ull;
            key[v] = (unsigned) (c >> 32);
            idf[v] = (unsigned) c;
        }
        wave_emit64<V>(key, idf, wave_select64<V>(key, idf), cand[wave]);
    }
    __syncthreads();
    if (wave != 0) return;
    constexpr int W = SM_MERGE_THREADS / 64;
    __shared__ unsigned long long best[SM_N];
    {
        unsigned key[W], idf[W];
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const unsigned long long c = cand[j][lane];
            key[j] = (unsigned) (c >> 32);
            idf[j] = (unsigned) c;
        }
        wave_emit64<W>(key, idf, wave_select64<W>(key, idf), best);
    }
    // one pair a lane; a pair's place is the number of greater ones (the 64 are distinct: a row has 64 logits at least), every
    // lane's pair handed round through scalar registers: half the time of a sorting network of exchanges between lanes
    const unsigned long long c = best[lane];
    int place = 0;
#pragma unroll
    for (int l = 0; l < 64; ++l) {
        const unsigned lo = (unsigned) __builtin_amdgcn_readlane((int) (unsigned) c, l), hi = (unsigned) __builtin_amdgcn_readlane((int) (unsigned) (c >> 32), l);
        place += ((unsigned long long) hi << 32 | lo) > c;
    }
    const int j = (int) (0xffffffffu - (unsigned) c);
    out_i[row * SM_N + place] = v0 + j;
    out_v[row * SM_N + place] = logits[(size_t) row * n + j];
}

// penalize_row (kernels.hpp:434-436): pen = {k, k indexes into the row, their k counts}, par = {repeat, freq, present}
__global__ void k_penalize_row(float* __restrict__ L, int n, const int* __restrict__ pen, const float* __restrict__ par) {
    const int k = min(max(pen[0], 0), SM_PEN_CAP);   // a count past the cap is not a list: never walk off the buffer on its word
    const float repeat = par[0], freq = par[1], present = par[2];
    for (int i = threadIdx.x; i < k; i += blockDim.x) {
        const int j = pen[1 + i], cnt = pen[1 + k + i];
        if (j < 0 || j >= n || cnt <= 0) continue;
        float l = L[j];
        l = l <= 0.f ? l * repeat : l / repeat;
        L[j] = l - (float) cnt * freq - present;
    }
}

}  // namespace fnx
