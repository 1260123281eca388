// The prompt path's MoE: routing into jobs of up to FNX_PF_JOB rows per expert, and the routed experts on the matrix
// cores with f16 weights and activations and fp32 accumulation (the numerics of the reference's moe_mma.cuh:1-11).
//
// Matrix-core kernel, CDNA4 form. A wave owns 16 (or 32) weight rows of one job and walks K; v_mfma_f32_16x16x32_f16
// wants from lane l the operand row l % 16 and eight consecutive k "slots" of group l / 16. Which k a slot means is
// free as long as both operands agree, so group g is given the sub-blocks sb = 4 q + g: a lane then decodes one whole
// IQ3_S sub-block (32 weights, exactly what a lane of the mat-vec kernels decodes) straight into the A operands of four
// MFMAs, and the B operand of MFMA i is the 16 contiguous bytes x[token][32 sb + 8 i ..]. The dequantised weights
// never pass through LDS; LDS holds only the signed codebook as f16 (8192 entries of 4 halves, 64 KiB).
// A weight becomes f16 as (grid * (1 + 2 s)) * d: the first product is an integer below 2048, exact in f16, so the
// second rounds once - the same value as the reference's f32 product rounded to f16 (moe_mma_iq.cuh:136-149).
#pragma once

#include "gemv_rows_plan.h"
#include "k_moe_layer.h"

namespace fnx {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- routing (prefill.cu:288-377)
// a wave per row: top-k of its logits, the weights. The blocks past the rows' (cvt_n > 0) turn cvt_n floats at cvt_x into
// f16 at cvt_y: the activations' copy for the matrix cores, which waits for nothing, rides along instead of a launch.
constexpr int PF_TOPK_WAVES = 4;
__global__ void __launch_bounds__(PF_TOPK_WAVES * 64) k_pf_topk(const float* __restrict__ logits, int ls, int C, int nexp, int topk,
                                                               int* __restrict__ topi, float* __restrict__ topw, const float* __restrict__ cvt_x,
                                                               size_t cvt_n, uint16_t* __restrict__ cvt_y) {
    __shared__ int ex[PF_TOPK_WAVES][64];
    const int row_blocks = (C + PF_TOPK_WAVES - 1) / PF_TOPK_WAVES;
    if ((int) blockIdx.x >= row_blocks) {   // four values a thread and step
        const size_t nb = gridDim.x - row_blocks, stride = nb * blockDim.x * 4;
        for (size_t i = ((size_t) (blockIdx.x - row_blocks) * blockDim.x + threadIdx.x) * 4; i < cvt_n; i += stride) {
            if (i + 3 < cvt_n && ((uintptr_t) cvt_x & 15) == 0 && ((uintptr_t) cvt_y & 7) == 0) {
                const float4 v = *reinterpret_cast<const float4*>(cvt_x + i);
                uint2 h;
                h.x = (uint32_t) float_to_half_bits(v.x) | (uint32_t) float_to_half_bits(v.y) << 16;
                h.y = (uint32_t) float_to_half_bits(v.z) | (uint32_t) float_to_half_bits(v.w) << 16;
                *reinterpret_cast<uint2*>(cvt_y + i) = h;
            } else {
                for (size_t j = i; j < i + 4 && j < cvt_n; ++j) cvt_y[j] = float_to_half_bits(cvt_x[j]);
            }
        }
        return;
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, t = blockIdx.x * PF_TOPK_WAVES + wave;
    if (t >= C) return;
    if (nexp <= 512) wave_topk<8>(logits + (size_t) t * ls, nexp, topk, lane, ex[wave], topi + (size_t) t * topk, topw + (size_t) t * topk);
    else wave_topk<16>(logits + (size_t) t * ls, nexp, topk, lane, ex[wave], topi + (size_t) t * topk, topw + (size_t) t * topk);
}
// A block of NW waves takes EPB experts and puts their pairs in ascending order into the slots of their jobs (a pair always lands
// in the same job and slot, prefill.cu:340-343). Each of its waves goes through an NWth of all picks twice, PF_ROUNDS loads in
// flight: first every expert's pairs are counted (in LDS, by all waves) and how many of the block's experts' the wave has
// (ballots), then, with the waves' counts added up, the slots follow from the ballots; an expert's picks of 64 PF_ROUNDS are
// packed in LDS on the way, so that a busy expert's jobs are written 64 slots a store. So a block meets three times, however many
// pairs there are. Blocks past the experts write the shared expert's jobs (every row: gate|up reads row t, writes row P + t; down
// reads and writes row P + t) and their count. Where its jobs start a block works out for itself - every expert's pair count,
// ceil(count / FNX_PF_JOB) jobs each, the jobs of the experts before it - instead of waiting for a launch of one block that does
// it for all; it leaves its experts' counts and first jobs (cnt, jbase), the last expert's block the job count.
// Bound by the passes over the picks (LDS atomics and round trips to L2), which is why a block has the most waves there are and
// two experts, unless four waves have all picks in one batch each (PF_FEW): then four waves' meetings are shorter (77 rows:
// 5.3 us against 5.6, a launch's own latency). 512 experts, ten picks a row, some experts in most rows: 4096 rows 18 us,
// 512 rows 6.2; blocks of four waves that met every 2048 picks took 81 and 12.8, and without the packing 4096 rows take 28.
constexpr int PF_ROUNDS = 8, PF_MAXE = 1024, PF_FEW = 4 * 64 * PF_ROUNDS;   // (PF_MAXE: the most experts)
template <int NW, int EPB>
__global__ void __launch_bounds__(NW * 64) k_pf_fill(const int* __restrict__ topi, int P, int topk, int nexp, int* __restrict__ cnt,
                                                     int* __restrict__ jbase, int* __restrict__ njobs, fnx_bigjob* __restrict__ gu,
                                                     fnx_bigjob* __restrict__ dn, int cap, int C, fnx_bigjob* __restrict__ sh_gu,
                                                     fnx_bigjob* __restrict__ sh_dn, int* __restrict__ nsh) {
    constexpr int THREADS = NW * 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, eblocks = (nexp + EPB - 1) / EPB;
    if ((int) blockIdx.x >= eblocks) {
        if (!sh_gu) return;
        const int t = ((int) blockIdx.x - eblocks) * THREADS + tid;
        if (t == 0) *nsh = (C + FNX_PF_JOB - 1) / FNX_PF_JOB;
        if (t >= C) return;
        const int j = t / FNX_PF_JOB, k = t % FNX_PF_JOB;
        sh_gu[j].y[k] = t;
        sh_gu[j].out[k] = P + t;
        sh_dn[j].y[k] = P + t;
        sh_dn[j].out[k] = P + t;
        if (k == 0) {
            sh_gu[j].w = sh_dn[j].w = 0;
            sh_gu[j].n = sh_dn[j].n = min(FNX_PF_JOB, C - j * FNX_PF_JOB);
        }
        return;
    }
    const int e0 = blockIdx.x * EPB;
    __shared__ int hist[PF_MAXE], wjobs[NW], wcnt[EPB][NW], found[NW][64 * PF_ROUNDS];
    for (int i = tid; i < nexp; i += THREADS) hist[i] = 0;
    __syncthreads();
    const int span = (P + THREADS - 1) / THREADS * 64;   // a wave's picks: whole ballots
    const int p_lo = wave * span, p_hi = min(P, p_lo + span);
    int mine[EPB];
#pragma unroll
    for (int x = 0; x < EPB; ++x) mine[x] = 0;
    for (int p0 = p_lo; p0 < p_hi; p0 += 64 * PF_ROUNDS) {
        int pick[PF_ROUNDS];
#pragma unroll
        for (int r = 0; r < PF_ROUNDS; ++r) {
            const int p = p0 + 64 * r + lane;
            pick[r] = p < p_hi ? topi[p] : -1;
        }
#pragma unroll
        for (int r = 0; r < PF_ROUNDS; ++r) {
            if (pick[r] >= 0) atomicAdd(&hist[pick[r]], 1);
#pragma unroll
            for (int x = 0; x < EPB; ++x) mine[x] += __popcll(__ballot(pick[r] == e0 + x));
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int x = 0; x < EPB; ++x) wcnt[x][wave] = mine[x];
    }
    __syncthreads();
    int before_me = 0;   // jobs of the experts before this block's
    for (int i = tid; i < e0; i += THREADS) before_me += (hist[i] + FNX_PF_JOB - 1) / FNX_PF_JOB;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) before_me += __shfl_xor(before_me, o, 64);
    if (lane == 0) wjobs[wave] = before_me;
    __syncthreads();
    int jb[EPB], ce[EPB], at[EPB], some = 0;   // an expert's first job, its pairs, those before this wave's picks
    jb[0] = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) jb[0] += wjobs[w];
#pragma unroll
    for (int x = 0; x < EPB; ++x) {
        ce[x] = e0 + x < nexp ? hist[e0 + x] : 0;
        if (x) jb[x] = jb[x - 1] + (ce[x - 1] + FNX_PF_JOB - 1) / FNX_PF_JOB;
        at[x] = 0;
        for (int w = 0; w < wave; ++w) at[x] += wcnt[x][w];
        some += mine[x];
        if (tid == 0 && e0 + x < nexp) {
            cnt[e0 + x] = ce[x];
            jbase[e0 + x] = jb[x];
            if (e0 + x == nexp - 1) njobs[0] = jb[x] + (ce[x] + FNX_PF_JOB - 1) / FNX_PF_JOB;
        }
    }
    if (some == 0) return;
    for (int p0 = p_lo; p0 < p_hi; p0 += 64 * PF_ROUNDS) {
        int pick[PF_ROUNDS];
#pragma unroll
        for (int r = 0; r < PF_ROUNDS; ++r) {
            const int p = p0 + 64 * r + lane;
            pick[r] = p < p_hi ? topi[p] : -1;
        }
#pragma unroll
        for (int x = 0; x < EPB; ++x) {   // an expert's picks among these, packed in LDS first: a busy expert's go out 64 a store
            int n = 0;
#pragma unroll
            for (int r = 0; r < PF_ROUNDS; ++r) {
                const unsigned long long m = __ballot(pick[r] == e0 + x);
                if (pick[r] == e0 + x) found[wave][n + __popcll(m & ((1ull << lane) - 1ull))] = p0 + 64 * r + lane;
                n += __popcll(m);
            }
            for (int i = lane; i < n; i += 64) {
                const int p = found[wave][i], s = at[x] + i, j = jb[x] + s / FNX_PF_JOB, k = s % FNX_PF_JOB;
                if (j < cap) {
                    gu[j].y[k] = p / topk;
                    gu[j].out[k] = p;
                    dn[j].y[k] = p;
                    dn[j].out[k] = p;
                    if (k == 0) {
                        gu[j].w = dn[j].w = e0 + x;
                        gu[j].n = dn[j].n = min(FNX_PF_JOB, ce[x] - (s / FNX_PF_JOB) * FNX_PF_JOB);
                    }
                }
            }
            at[x] += n;
        }
    }
}

// ---------------------------------------------------------------- element-wise
__global__ void k_f32_f16(const float* __restrict__ x, size_t n, uint16_t* __restrict__ y) {
    for (size_t i = blockIdx.x * (size_t) blockDim.x + threadIdx.x; i < n; i += (size_t) gridDim.x * blockDim.x) y[i] = float_to_half_bits(x[i]);
}
// moe_mma.cuh:500-507
__global__ void k_swiglu_h16(const float* __restrict__ gu, int ffs, size_t total, uint16_t* __restrict__ h) {
    for (size_t e = blockIdx.x * (size_t) blockDim.x + threadIdx.x; e < total; e += (size_t) gridDim.x * blockDim.x) {
        const size_t r = e / ffs, i = e % ffs;
        const float g = gu[r * 2 * ffs + i];
        h[e] = float_to_half_bits(silu_f(g) * gu[r * 2 * ffs + ffs + i]);
    }
}

// ---------------------------------------------------------------- router logits of a chunk
// The same sums for many activation rows (the prompt path's router logits): a wave takes GR_ROWS weight rows x a group
// of FNX_MAXT activation rows, lane l the float4 chunks l, l + 64, ... of all of them, so every activation chunk it
// loads (coalesced, straight from the caches: no LDS, no barriers) feeds GR_ROWS chains. Order per sum as above.
constexpr int GM_WAVES = 8, GR_ROWS = 4, GM_BATCH = 8;
static_assert(GR_ROWS * FNX_MAXT == 64, "64 sums a wave, one per lane in the end");
// one wave: weight rows row0 .. row0 + GR_ROWS - 1 against the activation rows FNX_MAXT tgroup ..
template <bool BF>
__device__ __forceinline__ void gemv_rows_many_wave(const void* __restrict__ Wv, const float* __restrict__ x, float* __restrict__ y, int rows, int n,
                                                    int T, int row0, int tgroup, int lane) {
    x += (size_t) tgroup * FNX_MAXT * n;
    y += (size_t) tgroup * FNX_MAXT * rows;
    T = min(FNX_MAXT, T - tgroup * FNX_MAXT);
    if (row0 >= rows || T <= 0) return;
    float acc[GR_ROWS][FNX_MAXT];
#pragma unroll
    for (int r = 0; r < GR_ROWS; ++r)
#pragma unroll
        for (int t = 0; t < FNX_MAXT; ++t) acc[r][t] = 0.f;
    const float4* xr[FNX_MAXT];
#pragma unroll
    for (int t = 0; t < FNX_MAXT; ++t) xr[t] = reinterpret_cast<const float4*>(x + (size_t) min(t, T - 1) * n) + lane;
    for (int c0 = 0; c0 < n / 4; c0 += 64) {
        float4 w[GR_ROWS];
#pragma unroll
        for (int r = 0; r < GR_ROWS; ++r) {
            const size_t row = (size_t) min(row0 + r, rows - 1);
            if constexpr (BF) {
                const uint2 u = reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(Wv) + row * n)[c0 + lane];
                w[r] = make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                                   __uint_as_float(u.y & 0xffff0000u));
            } else {
                w[r] = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(Wv) + row * n)[c0 + lane];
            }
        }
        // GM_BATCH activation chunks in flight at a time (left to itself the compiler loads them one by one, each a cache
        // round trip before its 16 fmaf)
#pragma unroll
        for (int t0 = 0; t0 < FNX_MAXT; t0 += GM_BATCH) {
            float4 b[GM_BATCH];
#pragma unroll
            for (int t = 0; t < GM_BATCH; ++t) b[t] = xr[t0 + t][c0];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < GM_BATCH; ++t)
#pragma unroll
                for (int r = 0; r < GR_ROWS; ++r) {
                    float a = acc[r][t0 + t];
                    a = fmaf(w[r].x, b[t].x, a);
                    a = fmaf(w[r].y, b[t].y, a);
                    a = fmaf(w[r].z, b[t].z, a);
                    a = fmaf(w[r].w, b[t].w, a);
                    acc[r][t0 + t] = a;
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // The 64 sums (value j = 16 r + t) over the 64 lanes, all at once: at the butterfly's level for lane bit b a lane
    // keeps the half of its values whose index has bit b equal to its own and adds its partner's copy of them - the
    // same pairwise adds, level by level, as group_sum<64> makes for each value, in 63 exchanges instead of 384.
    // Lane l ends with value l.
    float v32[32], v16[16], v8[8];
#pragma unroll
    for (int i = 0; i < 32; ++i) v32[i] = swap32_add(acc[i >> 4][i & 15], acc[2 + (i >> 4)][i & 15]);
#pragma unroll
    for (int i = 0; i < 16; ++i) v16[i] = swap16_add(v32[i], v32[i + 16]);
    auto fold = [&](const float lo, const float hi, int o) {
        const bool up = lane & o;
        return (up ? hi : lo) + __shfl_xor(up ? lo : hi, o, WAVE);
    };
#pragma unroll
    for (int i = 0; i < 8; ++i) v8[i] = fold(v16[i], v16[i + 8], 8);
    const float a0 = fold(v8[0], v8[4], 4), a1 = fold(v8[1], v8[5], 4), a2 = fold(v8[2], v8[6], 4), a3 = fold(v8[3], v8[7], 4);
    const float b0 = fold(a0, a2, 2), b1 = fold(a1, a3, 2);
    const float v = fold(b0, b1, 1);
    const int r = lane >> 4, t = lane & 15;
    if (t < T && row0 + r < rows) y[(size_t) t * rows + row0 + r] = v;
}
template <bool BF>
__global__ void __launch_bounds__(GM_WAVES * 64) k_gemv_rows_many(const void* __restrict__ Wv, const float* __restrict__ x, float* __restrict__ y,
                                                                 int rows, int n, int T, int row_begin) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    gemv_rows_many_wave<BF>(Wv, x, y, rows, n, T, row_begin + (blockIdx.x * GM_WAVES + wave) * GR_ROWS, blockIdx.y, lane);
}

// ---------------------------------------------------------------- the same sums in tiles of 16 x 16, for a short chunk
// A chunk of a few hundred rows leaves the kernel below (tiles of 32 x 32: 48 blocks for 77 rows against 513 weight rows) with
// CUs that have no tile or one, and a tile's chain of 256 MFMAs of 64 cycles a wave is its time. Here a tile is 16 x 16
// and the instruction v_mfma_f32_16x16x1_4b_f32: its four blocks take lanes l, l + 16, l + 32 and l + 48 of the fixed order
// (the butterfly's levels 32 and 16 are adds within the accumulator), wave w of four takes l = 4 w + j, four independent chains
// of n / 64 MFMAs of 32 cycles that it goes through together - a quarter of the tile's work in a quarter of the time, on
// four times the blocks. Levels 8 and 4 add the waves' sums, levels 2 and 1 the chains', through LDS at the end.
// Operands: a stage is 256 columns of the tile's 16 + 16 rows, a row 1 KiB and a wave instruction (two loader waves, straight
// into LDS, two stages ahead, one of three buffers); rows lie 1,040 bytes apart, so that the 16 rows an operand read
// touches fall on 16 different bank groups. The waves multiply a stage while the next one's operands are read.
// Bound by what the XCDs' L2s hand over (256 KB a tile; some 10 TB/s in all) once every CU has a tile: 77 rows x 513 of 2048,
// 13.8 -> 5.5 us over one set of weights; 7.5 inside a layer, whose other launches have the caches in between.
typedef float rs_v16f __attribute__((ext_vector_type(16)));
constexpr int RS_WAVES = 4, RS_LOADERS = 2, RS_THREADS = (RS_WAVES + RS_LOADERS) * 64, RS_ROWLD = RS_COLS * 4 + 16,
              RS_STAGE = 2 * RS_TILE * RS_ROWLD, RS_BUFS = 3;
__global__ void __launch_bounds__(RS_THREADS) k_gemv_rows_mfma16(const float* __restrict__ W, const float* __restrict__ x, float* __restrict__ y, int rows,
                                                                int n, int T, int ntt, int net) {
    __shared__ __align__(16) uint8_t lds[RS_BUFS * RS_STAGE];
    __shared__ __align__(16) float red[RS_WAVES][4][64][4];   // [wave][chain][lane][row of the lane's four]
    const int wave = uniform((int) (threadIdx.x >> 6)), lane = threadIdx.x & 63;
    // an XCD's blocks (every eighth) take neighbouring tiles, a tile of W against all of x's: its L2 then holds what they share
    const int lin = ((int) blockIdx.x % 8) * ((int) gridDim.x / 8) + (int) blockIdx.x / 8, et = lin / ntt, tt = lin - et * ntt;
    if (et >= net) return;
    const int t0 = tt * RS_TILE, e0 = et * RS_TILE, S = n / RS_COLS;   // stages: an even number, two at least
    const uint32_t lds_at = (uint32_t) (size_t) (__attribute__((address_space(3))) uint8_t*) lds;
    auto meet = [&](bool newest_in_flight) {   // (see k_gemv_rows_mfma's)
        __builtin_amdgcn_sched_barrier(0);
        if (newest_in_flight) __builtin_amdgcn_s_waitcnt(0x4070);   // vmcnt(16) lgkmcnt(0)
        else __builtin_amdgcn_s_waitcnt(0x0070);                    // vmcnt(0) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wave >= RS_WAVES) {   // a loader: the first takes the stages' rows of W, the second those of x
        const int lw = wave - RS_WAVES;
        const uint8_t* from[RS_TILE];
#pragma unroll
        for (int j = 0; j < RS_TILE; ++j)   // (past the last row: that one again)
            from[j] = reinterpret_cast<const uint8_t*>(lw == 0 ? W + (size_t) min(e0 + j, rows - 1) * n : x + (size_t) min(t0 + j, T - 1) * n);
        auto fetch = [&](int k, int buf) {
#pragma unroll
            for (int j = 0; j < RS_TILE; ++j)
                lds_load16(from[j] + (size_t) k * (RS_COLS * 4), 16u * lane, lds_at + buf * RS_STAGE + (lw * RS_TILE + j) * RS_ROWLD);
        };
        fetch(0, 0);
        fetch(1, 1);
        int buf = 2;
        for (int k = 0; k < S; ++k) {
            meet(k + 1 < S);   // stage k has landed; stage k - 1 has been read
            if (k + 2 < S) fetch(k + 2, buf);
            buf = buf == RS_BUFS - 1 ? 0 : buf + 1;
        }
        return;   // (a wave that has ended counts as arrived at the last meeting)
    }
    const int i = lane & 15, b = lane >> 4;
    const uint8_t* row = lds + i * RS_ROWLD + 16 * (16 * b + 4 * wave);   // row i of W (of x: 16 rows on), chains 4 wave .. + 3 of block b
    float4 A[2][4], B[2][4];
    rs_v16f acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
    int at = 0;   // the buffer that is read next
    auto read = [&](float4(&a)[4], float4(&bb)[4]) {
        meet(false);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            a[j] = *reinterpret_cast<const float4*>(row + at + 16 * j);
            bb[j] = *reinterpret_cast<const float4*>(row + at + RS_TILE * RS_ROWLD + 16 * j);
        }
        at = at == (RS_BUFS - 1) * RS_STAGE ? 0 : at + RS_STAGE;
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const float4(&a)[4], const float4(&bb)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x1f32(a[j].x, bb[j].x, acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x1f32(a[j].y, bb[j].y, acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x1f32(a[j].z, bb[j].z, acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x1f32(a[j].w, bb[j].w, acc[j], 0, 0, 0);
    };
    read(A[0], B[0]);
    for (int k = 0; k < S; k += 2) {
        read(A[1], B[1]);
        multiply(A[0], B[0]);
        if (k + 2 < S) read(A[0], B[0]);
        multiply(A[1], B[1]);
    }
    // block q's sums lie in registers 4 q .. 4 q + 3: weight rows 4 b .. 4 b + 3 of the tile against row i of x
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float f[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) f[r] = (acc[j][r] + acc[j][8 + r]) + (acc[j][4 + r] + acc[j][12 + r]);
        *reinterpret_cast<float4*>(red[wave][j][lane]) = make_float4(f[0], f[1], f[2], f[3]);
    }
    meet(false);
    const int e = e0 + 4 * b + wave, t = t0 + i;   // this wave's row of each lane's four
    float s[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = (red[0][j][lane][wave] + red[2][j][lane][wave]) + (red[1][j][lane][wave] + red[3][j][lane][wave]);
    if (e < rows && t < T) y[(size_t) t * rows + e] = (s[0] + s[2]) + (s[1] + s[3]);
}

// ---------------------------------------------------------------- the same sums on the matrix cores
// v_mfma_f32_32x32x1_2b_f32 is D = fma(a, b, D) element by element with one rounding - the fmaf of the chains above
// (checked bit for bit on this GPU, products in the denormal range included). A chain of them over the chunks
// l, l + 64, ... therefore leaves lane l's partial sum of 32 activation rows x 32 weight rows at once; the instruction's
// two blocks take l and l + 32, the pair that the butterfly adds first. A block owns such a tile of 32 x 32 sums; wave w of four
// takes the lanes l = 16 h + 4 w + j: for h = 0 and then h = 1 the four chains of j side by side, so that an MFMA never waits for
// the one before it. Level 16 of the butterfly adds the two halves' accumulators, levels 8 and 4 the waves', levels 2 and 1 the four
// chains', through LDS at the end.
// Operands (f32 weights only): a step is a chunk of each of the wave's chains of 32 + 32 rows, a row's four chunks (and those of
// l + 32) 64 bytes in a row: eight kilobytes that the wave sends to a ring of its own in LDS (global_load_lds_dwordx4, sixteen
// such runs an instruction), RM_RING - 1 steps ahead, and nobody else reads: no wave meets another before the end, and a
// wait is for its own loads, counted. A step's sixteen MFMAs (64 cycles each) hide the eight reads of the next step's operands and
// the eight loads of the ring's next step, one behind each MFMA. Run r of eight rows' runs lies at place p = 4 r + (j ^ f), f of the row,
// so that the 16 rows an operand read touches fall on 16 different bank groups.
// A CU has one block (its rings fill the LDS), which takes its tiles one after another (MANY): the next tile's first steps come in
// behind the last ones of the tile before, and its sums go through a place of their own, so that a tile's start is not waited for and
// its end is the exchange alone. With a block a tile the CU stood still from one tile's last MFMA to the next one's first: 513 rows of 2,048
// columns, 4,096 rows of x 95 -> 88 us over weights in turn, 1,900 51.5 -> 45.1 (the launch alone); two tiles a block the same (700: 24.4), and where
// every block has one tile that form is 4 % behind the plain one (its sums in the ring, nothing asked for past the end).
// Bound by the MFMAs and the loads behind them: of a chain of tiles some 11 us each (eight a CU: 88), where the MFMAs alone take 6.8, the operands'
// reads 0.7; a tile alone 14.9 with the launch's start and end.
// The weight rows past the last full 32 (the router's 513th) are items of such a row against one row of x, added up while the first
// steps are on their way: where a row of tiles has a wave for each of its items, and a block one tile, those, one a wave at most; else dealt to all
// waves of the grid (SPREAD), T / 1,024 a wave for the router's one row: 8,192 rows of x 195 -> 176 us against a launch of a block a tile, 65,535 1,516 -> 1,401.
typedef float v32f __attribute__((ext_vector_type(32)));
constexpr int RM_WAVES = 4, RM_THREADS = RM_WAVES * 64, RM_STEP = 8 * 1024, RM_RING = 4, RM_PART = 2 * 4 * 64 * 16;   // (RM_PART: a wave's sums of two chains)
template <bool MANY, bool SPREAD>
__global__ void __launch_bounds__(RM_THREADS) __attribute__((amdgpu_waves_per_eu(1, 1))) k_gemv_rows_mfma(const float* __restrict__ W, const float* __restrict__ x,
                                                                                                         float* __restrict__ y, int rows, int n, int T, int ntt,
                                                                                                         int net, int items) {
    __shared__ __align__(16) uint8_t lds[RM_WAVES * RM_RING * RM_STEP];
    __shared__ __align__(16) uint8_t red[MANY ? RM_WAVES * RM_PART : 16];   // the waves' sums of two chains at a tile's end
    const int wave = uniform((int) (threadIdx.x >> 6)), lane = threadIdx.x & 63;
    // Which tiles: block ids go round the eight XCDs, each with an L2 of its own, so an XCD's blocks are given an eighth of the tiles in
    // patches of 4 x 8 (1 MB of x and 2 MB of W for rows of 2048: its L2 holds them), a patch's tiles side by side. Several tiles a block: the patches
    // go along x, so that an XCD keeps its rows of W. A block a tile: along W (513 x 512 along x 15.2 us, along W 14.9, as with a grid of whole patches,
    // whose blocks without a tile left most CUs idle where W has few rows: 33 weight rows, 8,192 of x 71 us, 35 without them).
    const int total = ntt * net, xcd = (int) blockIdx.x % 8, per = (int) gridDim.x / 8;
    int L = (total * xcd >> 3) + (int) blockIdx.x / 8;   // (total < 2^28: x and W lie below 4 GiB each)
    const int Lend = total * (xcd + 1) >> 3;
    int t0 = 0, e0 = 0;
    auto tile_of = [&](int l) {   // (no divisions where a patch is a whole one: a block does this before its first load)
        if (!MANY && net % 8 == 0 && ntt % 4 == 0) {
            const int a = (l >> 5) / (net >> 3);
            t0 = (4 * a + ((l & 31) >> 3)) * RM_TILE, e0 = (8 * ((l >> 5) - a * (net >> 3)) + (l & 7)) * RM_TILE;
            return;
        }
        int p = 0;
        for (; l >= 8 * ntt; l -= 8 * ntt) ++p;
        const int w = min(8, net - 8 * p), q = w == 8 ? l >> 5 : l / (4 * w), r = l - 4 * w * q, d = w == 8 ? r >> 3 : r / w;
        t0 = (4 * q + d) * RM_TILE, e0 = (8 * p + r - w * d) * RM_TILE;
    };
    const bool any = L < Lend;   // (a block without a tile helps with the items where they are spread)
    if (!SPREAD && !any) return;
    tile_of(any ? L : 0);
    const int half = n / 256, S = 2 * half;   // steps: a multiple of 16
    uint8_t* ring = lds + wave * (RM_RING * RM_STEP);
    const uint32_t ring_at = (uint32_t) (size_t) (__attribute__((address_space(3))) uint8_t*) ring;
    uint32_t xoff[4], woff[4];   // instruction g: rows 8 g .. 8 g + 7, this lane's piece
    auto point = [&]() {
        const int r7 = (lane >> 2) & 7, b = lane >> 5;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint32_t piece = 512u * b + 16u * ((lane & 3) ^ ((r7 >> 2) | ((g & 1) << 1)));
            xoff[g] = (uint32_t) min(t0 + 8 * g + r7, T - 1) * (uint32_t) n * 4u + piece;
            woff[g] = (uint32_t) (e0 + 8 * g + r7) * (uint32_t) n * 4u + piece;
        }
    };
    point();
    auto from_of = [&](int s) { return 64 * wave + (s >= half ? 256 + 1024 * (s - half) : 1024 * s); };
    auto fetch = [&](int op, int from, int slot) {   // one of a step's eight instructions
        const int g = op & 3;
        if (op < 4) lds_load16(reinterpret_cast<const uint8_t*>(x) + from, xoff[g], ring_at + slot * RM_STEP + g * 1024);
        else lds_load16(reinterpret_cast<const uint8_t*>(W) + from, woff[g], ring_at + slot * RM_STEP + 4096 + g * 1024);
    };
    if (any) {
#pragma unroll
        for (int s = 0; s < RM_RING; ++s)   // (S >= 16)
#pragma unroll
            for (int op = 0; op < 8; ++op) fetch(op, from_of(s), s);
    }
    // The weight rows past the last full tile: items of such a row against one row of x. SPREAD: all of them over the waves of the grid;
    // else a row of tiles' items go to its waves, one at most, whose x the L2 has.
    auto item_of = [&](int it, int irow, bool on) {
        const float4 *wp = reinterpret_cast<const float4*>(W + (size_t) irow * n) + lane, *xp = reinterpret_cast<const float4*>(x + (size_t) it * n) + lane;
        float v = 0.f;
        for (int c0 = 0; c0 < n / 4; c0 += 8 * 64) {
            float4 wv[8], xv[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) wv[k] = wp[c0 + 64 * k], xv[k] = xp[c0 + 64 * k];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                v = fmaf(wv[k].x, xv[k].x, v);
                v = fmaf(wv[k].y, xv[k].y, v);
                v = fmaf(wv[k].z, xv[k].z, v);
                v = fmaf(wv[k].w, xv[k].w, v);
            }
        }
        v = group_sum<64>(v);
        if (lane == 0 && on) y[(size_t) it * rows + irow] = v;
    };
    if constexpr (SPREAD) {
        const int left = rows - net * RM_TILE;
        if (items > 0) {
            for (int item = (int) blockIdx.x * RM_WAVES + wave; item < items; item += (int) gridDim.x * RM_WAVES) {
                const int it = left == 1 ? item : item / left;
                item_of(it, net * RM_TILE + item - it * left, true);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the counts below are of the steps' loads alone)
        }
    } else if (const int item = RM_WAVES * (e0 / RM_TILE) + wave; items > 0 && item < RM_TILE * (rows - net * RM_TILE)) {
        const int it = t0 + item % RM_TILE;
        item_of(min(it, T - 1), net * RM_TILE + item / RM_TILE, it < T);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    if (!any) return;   // the same for the whole block
    const int i = lane & 31, b = lane >> 5;
    const int rd = (i >> 3) * 1024 + 64 * ((i & 7) + 8 * b), f = ((i & 7) >> 2) | (((i >> 3) & 1) << 1);
    const uint8_t* at[4];   // this lane's pieces of a step: row i of x (of W: 4 KiB on), chunk j of its block
#pragma unroll
    for (int j = 0; j < 4; ++j) at[j] = ring + rd + 16 * (j ^ f);
    float4 A[2][4], B[2][4];
    v32f acc[4];
    float held[4][16];
    auto wait = [&](int steps) {   // until only the newest so many steps' loads may be on their way
        __builtin_amdgcn_sched_barrier(0);
        if (steps == 2) __builtin_amdgcn_s_waitcnt(0x4F70);        // vmcnt(16)
        else if (steps == 1) __builtin_amdgcn_s_waitcnt(0x0F78);   // vmcnt(8)
        else __builtin_amdgcn_s_waitcnt(0x0F70);                   // vmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // A step: its sixteen MFMAs over the operands a, bb, and behind one of them each the reads of the next step's (READ, from slot
    // rs) and the loads of the step RM_RING on (FETCH, into the slot this step was read from). FIRST: a half's first step,
    // whose chains start from zero; the half before is folded (the instruction's two blocks, level 32) into held ahead of its chain.
    auto step = [&](const float4 (&a)[4], const float4 (&bb)[4], float4 (&na)[4], float4 (&nb)[4], int rs, int from, auto first_c, auto fold_c, auto read_c, auto fetch_c) {
        constexpr bool FIRST = decltype(first_c)::value, FOLD = decltype(fold_c)::value, READ = decltype(read_c)::value, FETCH = decltype(fetch_c)::value;
        const int ro = rs * RM_STEP, fs = (rs + RM_RING - 1) % RM_RING;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int j = m & 3, c = m >> 2;
            if (FOLD && c == 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) held[j][v] = acc[j][v] + acc[j][16 + v];
            }
            const float av = c == 0 ? a[j].x : c == 1 ? a[j].y : c == 2 ? a[j].z : a[j].w, bv = c == 0 ? bb[j].x : c == 1 ? bb[j].y : c == 2 ? bb[j].z : bb[j].w;
            if (FIRST && c == 0) {
                v32f z;
#pragma unroll
                for (int v = 0; v < 32; ++v) z[v] = 0.f;
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x1f32(av, bv, z, 0, 0, 0);
            } else {
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x1f32(av, bv, acc[j], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (READ && m < 8) {
                if (m < 4) na[m] = *reinterpret_cast<const float4*>(at[m] + ro);
                else nb[m & 3] = *reinterpret_cast<const float4*>(at[m & 3] + ro + 4096);
            }
            if (FETCH && m >= 8) fetch(m - 8, from, fs);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto meet = [] {   // (the loads on their way stay there)
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    using std::integral_constant;
    constexpr integral_constant<bool, true> yes{};
    constexpr integral_constant<bool, false> no{};
    wait(2);   // (the first two steps have landed)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        A[0][j] = *reinterpret_cast<const float4*>(at[j]);
        B[0][j] = *reinterpret_cast<const float4*>(at[j] + 4096);
    }
    // step k reads step k + 1's operands and fetches step k + RM_RING; RM_RING steps a trip, so that the ring's places are constants
    auto trip = [&](int k, auto first_c, auto fold_c, auto last_c) {
        constexpr bool LAST = decltype(last_c)::value;
        constexpr integral_constant<bool, !LAST> on{};
        wait(2);
        step(A[0], B[0], A[1], B[1], 1, from_of(k + 4), first_c, fold_c, yes, on);
        wait(LAST ? 1 : 2);
        step(A[1], B[1], A[0], B[0], 2, from_of(k + 5), no, no, yes, on);
        wait(LAST ? 0 : 2);
        step(A[0], B[0], A[1], B[1], 3, from_of(k + 6), no, no, yes, on);
        if constexpr (!LAST) wait(2);
        step(A[1], B[1], A[0], B[0], 0, from_of(k + 7), no, no, on, on);
    };
    while (true) {
        const int tt0 = t0, te0 = e0;
        const bool more = MANY && L + per < Lend;
        trip(0, yes, no, no);
        for (int k = RM_RING; k < half; k += RM_RING) trip(k, no, no, no);
        trip(half, yes, yes, no);
        for (int k = half + RM_RING; k + RM_RING < S; k += RM_RING) trip(k, no, no, no);
        if constexpr (MANY) {   // the next tile's first steps come in behind this one's last (after the last tile its own again: no form without them)
            L += more ? per : 0;
            tile_of(L);
            point();
            trip(-RM_RING, no, no, no);
        } else {
            trip(0, no, no, yes);
        }
        // levels 32 and 16 here, 8 and 4 over the waves, 2 and 1 over the chains: wave w the accumulator's registers 4 w .. 4 w + 3. The sums
        // go through the waves' own rings (each has been read by its wave), or, where the next tile's steps are coming in there, two chains at a time
        // through a place of their own.
        constexpr int CH = MANY ? 2 : 4;
        uint8_t* const to = MANY ? red + wave * RM_PART : ring;
        const uint8_t* const from = MANY ? red : lds;
        constexpr int part = MANY ? RM_PART : RM_RING * RM_STEP;
        static_assert(CH * 4 * 64 * 16 <= part, "a wave's sums fit their place");
        float s[4][4];
#pragma unroll
        for (int j0 = 0; j0 < 4; j0 += CH) {
            if (j0) meet();   // the sums before have been read
#pragma unroll
            for (int j = j0; j < j0 + CH; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float u[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v) u[v] = held[j][4 * q + v] + (acc[j][4 * q + v] + acc[j][16 + 4 * q + v]);
                    *reinterpret_cast<float4*>(to + (((j - j0) * 4 + q) * 64 + lane) * 16) = make_float4(u[0], u[1], u[2], u[3]);
                }
            meet();
#pragma unroll
            for (int j = j0; j < j0 + CH; ++j) {
                float4 u[4];
#pragma unroll
                for (int w = 0; w < 4; ++w) u[w] = *reinterpret_cast<const float4*>(from + w * part + (((j - j0) * 4 + wave) * 64 + lane) * 16);
                s[j][0] = (u[0].x + u[2].x) + (u[1].x + u[3].x);
                s[j][1] = (u[0].y + u[2].y) + (u[1].y + u[3].y);
                s[j][2] = (u[0].z + u[2].z) + (u[1].z + u[3].z);
                s[j][3] = (u[0].w + u[2].w) + (u[1].w + u[3].w);
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = tt0 + 8 * wave + 4 * b + v;
            if (t < T) y[(size_t) t * rows + te0 + i] = (s[0][v] + s[2][v]) + (s[1][v] + s[3][v]);
        }
        if (!more) break;
        meet();   // (the next tile's sums go to the same place)
    }
    if constexpr (MANY) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing is on its way into LDS when the block leaves

}

// ---------------------------------------------------------------- the routed experts on the matrix cores
struct MmaArgs {
    const uint8_t* w;       // the experts' matrices: expert e at w + e * stride, or ep[e]
    size_t stride;
    const void* const* ep;
    int nrows, ncols;
    const fnx_bigjob* jobs;
    const int* njobs;
    int cap;
    const uint16_t* x;      // f16 activation rows of ldx values
    int ldx;
    float* out;             // rows of nrows
    // a second job list over one more matrix (the shared expert's, whatever its jobs' w says), in the same launch: alone
    // its few jobs fill a quarter of the chip (the wave forms)
    const uint8_t* w2 = nullptr;
    const fnx_bigjob* jobs2 = nullptr;
    const int* njobs2 = nullptr;
    int cap2 = 0;
    // wave form, stacked gate|up matrices: a wave's two tiles are 16 gate rows and the 16 up rows that go with them, and
    // what is written is h = silu(gate) * up as f16 rows of nrows / 2 (k_swiglu_h16's values) instead of the products themselves
    uint16_t* h16 = nullptr;
};
constexpr int MM_THREADS = 512, MM_WAVES = MM_THREADS / 64, MM_TT = FNX_PF_JOB / 16;

struct SubFields {   // one sub-block as loaded: four words of codes, the scale nibble, d's bits
    uint32_t q0, q1, q2, q3, sc, d;
};
// loads through address-space-1 pointers: global_load, which (unlike flat_load) does not tie up the LDS counter that
// the codebook reads wait on
template <bool PACKED>
__device__ __forceinline__ SubFields sub_load(const uint8_t* __restrict__ we, int row, int sb, int ks) {
    typedef __attribute__((address_space(1))) const v2u g64;
    typedef __attribute__((address_space(1))) const uint32_t g32;
    typedef __attribute__((address_space(1))) const unsigned short g16;
    SubFields r;
    if constexpr (PACKED) {
        const uint32_t L = (uint32_t) row * ks + sb, l = L & 63u;
        const gbytes u = as_global(we + (size_t) (L >> 6) * UNIT_BYTES);
        const v2u a = *(g64*) (u + 8 * l);
        r.q0 = a.x;
        r.q1 = a.y;
        r.q2 = *(g32*) (u + UNIT_B_AT + 4 * l);
        r.q3 = u[UNIT_C_AT + l];
        r.sc = u[UNIT_SCALES_AT + (l >> 1)] >> (4 * (l & 1));
        r.d = *(g16*) (u + UNIT_D_AT + 2 * (l >> 3));
    } else {
        const int ib = sb & 7;
        const gbytes b = as_global(we + ((size_t) row * (ks >> 3) + (sb >> 3)) * 110);
        const g16* q = (g16*) (b + 2 + 8 * ib);
        r.q0 = q[0] | (uint32_t) q[1] << 16;
        r.q1 = q[2] | (uint32_t) q[3] << 16;
        const g16* sg = (g16*) (b + 74 + 4 * ib);
        r.q2 = sg[0] | (uint32_t) sg[1] << 16;
        r.q3 = b[66 + ib];
        r.sc = b[106 + (ib >> 1)] >> (4 * (ib & 1));
        r.d = *(g16*) b;
    }
    return r;
}
// LDS byte offset of group j's entry in the f16 codebook (entries of 8 bytes)
template <bool PACKED>
__device__ __forceinline__ uint32_t sub_entry(const SubFields& f, int j) {
    if constexpr (PACKED) {
        const uint32_t q[4] = {f.q0, f.q1, f.q2, f.q3};
        const int bit = 13 * j, w = bit >> 5, s = bit & 31;
        uint32_t v;
        if (s + 13 <= 32) v = s >= 3 ? q[w] >> (s - 3) : q[w] << (3 - s);
        else v = __builtin_amdgcn_alignbit(q[w + 1], q[w], s - 3);
        return v & 0xFFF8u;
    } else {
        const uint32_t code = ((j < 4 ? f.q0 >> (8 * j) : f.q1 >> (8 * (j - 4))) & 0xFFu) | (((f.q3 >> j) & 1u) << 8);
        return (((f.q2 >> (4 * j)) & 0xFu) << 12) | (code << 3);
    }
}
__device__ __forceinline__ v2h as_v2h(uint32_t u) { return __builtin_bit_cast(v2h, u); }

// A task = (job, RG * 16 weight rows, MM_TP token tiles of 16): uniform pieces, so a static split over the waves
// balances; consecutive waves take the same job's next rows and share its activation rows in the caches.
// Order of a k-step's loads matters because loads return in order: first this step's activation operands (from L2,
// consumed after the decode), then the weights of two steps ahead (from HBM) - a wait for the former never waits for
// the latter.
constexpr int MM_TP = 2;
template <bool PACKED, int RG>
__global__ void __launch_bounds__(MM_THREADS) __attribute__((amdgpu_waves_per_eu(4, 4))) k_moe_mma(const MmaArgs a) {
    typedef __attribute__((address_space(1))) const v4u gx4;
    __shared__ uint2 tab[SGRID_WORDS];
    const uint32_t tab0 = g_sgrid.v[threadIdx.x];   // (512 threads: a thread's code, its sixteen signed entries made here)
#pragma unroll
    for (int i = threadIdx.x; i < SGRID_WORDS; i += MM_THREADS) {
        const uint32_t g = signed_entry(tab0, i >> 9);
        v2h lo, hi;
        lo.x = (_Float16) (int) (int8_t) (g & 0xFFu);
        lo.y = (_Float16) (int) (int8_t) ((g >> 8) & 0xFFu);
        hi.x = (_Float16) (int) (int8_t) ((g >> 16) & 0xFFu);
        hi.y = (_Float16) (int) (int8_t) (g >> 24);
        tab[i] = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int nj = min(a.cap, uniform(*a.njobs));
    const int ks = a.ncols >> 5, groups = a.nrows / (16 * RG), steps = ks >> 2;
    constexpr int HALVES = MM_TT / MM_TP;
    const int nwaves = gridDim.x * MM_WAVES, per_job = groups * HALVES;
    for (int task = uniform(blockIdx.x * MM_WAVES + (threadIdx.x >> 6)); task < nj * per_job; task += nwaves) {
        const int ji = task / per_job, rem = task - ji * per_job, t0 = (rem / groups) * MM_TP, row0 = (rem % groups) * 16 * RG;
        const fnx_bigjob* jb = a.jobs + ji;
        const int n = min(FNX_PF_JOB, uniform(jb->n)), e = uniform(jb->w), nt = (n + 15) >> 4;
        if (t0 >= nt) continue;
        const int ntile = min(MM_TP, nt - t0);
        const uint8_t* we = a.ep ? (const uint8_t*) a.ep[e] : a.w + (size_t) e * a.stride;
        const uint16_t* xr[MM_TP];
#pragma unroll
        for (int tt = 0; tt < MM_TP; ++tt) xr[tt] = a.x + (size_t) jb->y[min((t0 + tt) * 16 + r, n - 1)] * a.ldx + 32 * g;
        v4f acc[RG][MM_TP];
#pragma unroll
        for (int q = 0; q < RG; ++q)
#pragma unroll
            for (int tt = 0; tt < MM_TP; ++tt) acc[q][tt] = v4f{0.f, 0.f, 0.f, 0.f};
        SubFields w0[RG], w1[RG];
#pragma unroll
        for (int q = 0; q < RG; ++q) w0[q] = sub_load<PACKED>(we, row0 + 16 * q + r, g, ks);
        // one k-step: cur holds its weights' fields; nxt receives the next step's (no register copies between steps: a
        // copy of a loaded register would wait for the load)
        auto step = [&](SubFields (&cur)[RG], SubFields (&nxt)[RG], int st) {
            v4u B[MM_TP][4];
#pragma unroll
            for (int tt = 0; tt < MM_TP; ++tt)
                if (tt < ntile) {
                    const gx4* xp = (gx4*) (uintptr_t) (xr[tt] + 128 * st);
#pragma unroll
                    for (int i = 0; i < 4; ++i) B[tt][i] = xp[i];
                }
            const int sbn = 4 * min(st + 1, steps - 1) + g;   // past the end: the last step's again
#pragma unroll
            for (int q = 0; q < RG; ++q) nxt[q] = sub_load<PACKED>(we, row0 + 16 * q + r, sbn, ks);
            // this lane's sub-block of each row group as 32 f16 weights: the A operands of four MFMAs
            v8h A[RG][4];
#pragma unroll
            for (int q = 0; q < RG; ++q) {
                const _Float16 sc = (_Float16) (int) (1 + 2 * (cur[q].sc & 0xFu)), d = __builtin_bit_cast(_Float16, (unsigned short) cur[q].d);
                const v2h s2 = {sc, sc}, d2 = {d, d};
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint2 en = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(tab) + sub_entry<PACKED>(cur[q], j));
                    const v2h lo = (as_v2h(en.x) * s2) * d2, hi = (as_v2h(en.y) * s2) * d2;
                    A[q][j >> 1][4 * (j & 1) + 0] = lo.x;
                    A[q][j >> 1][4 * (j & 1) + 1] = lo.y;
                    A[q][j >> 1][4 * (j & 1) + 2] = hi.x;
                    A[q][j >> 1][4 * (j & 1) + 3] = hi.y;
                }
            }
#pragma unroll
            for (int tt = 0; tt < MM_TP; ++tt)
                if (tt < ntile) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int q = 0; q < RG; ++q)
                            acc[q][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[q][i], __builtin_bit_cast(v8h, B[tt][i]), acc[q][tt], 0, 0, 0);
                }
        };
        for (int st = 0; st < steps; st += 2) {   // steps = ncols / 128, even for whole 256-column blocks
            step(w0, w1, st);
            step(w1, w0, st + 1);
        }
        // lane: token r of each tile, weight rows 4 g .. 4 g + 3 of each group
#pragma unroll
        for (int tt = 0; tt < MM_TP; ++tt) {
            const int tok = (t0 + tt) * 16 + r;
            if (tt < ntile && tok < n) {
                float* o = a.out + (size_t) jb->out[tok] * a.nrows + row0 + 4 * g;
#pragma unroll
                for (int q = 0; q < RG; ++q) *reinterpret_cast<float4*>(o + 16 * q) = make_float4(acc[q][tt].x, acc[q][tt].y, acc[q][tt].z, acc[q][tt].w);
            }
        }
    }
}

// ---------------------------------------------------------------- a lane's four consecutive sub-blocks of a row
// What limits the wave-a-task kernel above (what is left to it: raw blocks, and unit64 rows of widths that are not 256, 512, 1,024 or whole 2,048s) on MI355X is the vector-memory front end: every wave gathers its weights 32
// bytes per row at a time, so each cache line is fetched four times. A lane that owns four consecutive sub-blocks of its
// row per super-step of 512 columns (sub-block 16 S + 4 g + p at step p) loads whole 32/16/4/2-byte runs of the planes,
// 6 loads per row and super-step, each line of a plane touched once: the loads of the tile16 re-laying below and of the
// wave forms (k_moe_mma_wave16.h), which read the same fields from the tile16 layout.
struct SuperFields {   // a lane's four sub-blocks of one row as loaded
    v4u a0, a1, b;
    uint32_t c, sc, d;
};
__device__ __forceinline__ SuperFields super_load(const uint8_t* __restrict__ we, int row, int sb0, int ks) {
    typedef __attribute__((address_space(1))) const v4u g128;
    typedef __attribute__((address_space(1))) const uint32_t g32;
    typedef __attribute__((address_space(1))) const unsigned short g16;
    const uint32_t L = (uint32_t) row * ks + sb0, l = L & 63u;   // l: a multiple of 4
    const gbytes u = as_global(we + (size_t) (L >> 6) * UNIT_BYTES);
    SuperFields r;
    r.a0 = *(g128*) (u + 8 * l);
    r.a1 = *(g128*) (u + 8 * l + 16);
    r.b = *(g128*) (u + UNIT_B_AT + 4 * l);
    r.c = *(g32*) (u + UNIT_C_AT + l);
    r.sc = *(g16*) (u + UNIT_SCALES_AT + (l >> 1));
    r.d = *(g16*) (u + UNIT_D_AT + 2 * (l >> 3));
    return r;
}
template <int P>
__device__ __forceinline__ SubFields super_sub(const SuperFields& f) {
    SubFields s;
    s.q0 = P < 2 ? f.a0[2 * (P & 1)] : f.a1[2 * (P & 1)];
    s.q1 = P < 2 ? f.a0[2 * (P & 1) + 1] : f.a1[2 * (P & 1) + 1];
    s.q2 = f.b[P];
    s.q3 = (f.c >> (8 * P)) & 0xFFu;
    s.sc = (f.sc >> (4 * P)) & 0xFu;
    s.d = f.d;
    return s;
}
// The same fields from the prompt path's own layout ("tile16", FNX_T_IQ3S_TILE16): a matrix as tiles of 16 rows x 512
// columns, tile (row / 16, column / 512) at ((row / 16) * (ncols / 512) + column / 512) * TILE16_BYTES, and in a tile the
// 64 lanes' shares side by side, plane by plane: lane (row % 16) + 16 g holds sub-blocks 4 g .. 4 g + 3 of the tile's 16 -
// A 32 bytes a lane, B 16, C 4, the scale nibbles 2, d 2. Every load of a wave is then one contiguous run (2 KiB, 1 KiB,
// 256, 128, 128 bytes) and a wave's super-steps follow each other in memory, where the unit64 planes give the matrix
// cores' lanes - sixteen different rows - a cache line each. 3,584 bytes per 8,192 weights (unit64: 3,520; d is held by
// both lanes of a super-block).
constexpr int TILE16_BYTES = 3584, TILE16_B_AT = 2048, TILE16_C_AT = 3072, TILE16_SC_AT = 3328, TILE16_D_AT = 3456;
__device__ __forceinline__ SuperFields tile16_load(const uint8_t* __restrict__ we, int row, int S, int nsuper) {   // row: the lane's row
    typedef __attribute__((address_space(1))) const v4u g128;
    typedef __attribute__((address_space(1))) const uint32_t g32;
    typedef __attribute__((address_space(1))) const unsigned short g16;
    const int lane = (row & 15) | (int) (threadIdx.x & 48u);
    const gbytes u = as_global(we + ((size_t) (row >> 4) * nsuper + S) * TILE16_BYTES);
    SuperFields r;
    r.a0 = *(g128*) (u + 32 * lane);
    r.a1 = *(g128*) (u + 32 * lane + 16);
    r.b = *(g128*) (u + TILE16_B_AT + 16 * lane);
    r.c = *(g32*) (u + TILE16_C_AT + 4 * lane);
    r.sc = *(g16*) (u + TILE16_SC_AT + 2 * lane);
    r.d = *(g16*) (u + TILE16_D_AT + 2 * lane);
    return r;
}
// The same through a buffer descriptor over a row of tiles (rows 16 t .. 16 t + 15: wave-uniform), tile S of it by a scalar
// offset: the lane's offsets are 32-bit and the planes' places ride in the instructions, where tile16_load keeps a 64-bit
// address a plane in vector registers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile16_rsrc(const uint8_t* __restrict__ we, int t, int nsuper) {
    return __builtin_amdgcn_make_buffer_rsrc((void*) uniform_ptr(we + (size_t) t * nsuper * TILE16_BYTES), 0, -1, 0x00020000);
}
__device__ __forceinline__ SuperFields tile16_load_buf(__amdgpu_buffer_rsrc_t m, int S) {
    const int lane = threadIdx.x & 63, at = S * TILE16_BYTES;
    SuperFields r;
    r.a0 = __builtin_amdgcn_raw_buffer_load_b128(m, 32 * lane, at, 0);
    r.a1 = __builtin_amdgcn_raw_buffer_load_b128(m, 32 * lane + 16, at, 0);
    r.b = __builtin_amdgcn_raw_buffer_load_b128(m, 16 * lane + TILE16_B_AT, at, 0);
    r.c = __builtin_amdgcn_raw_buffer_load_b32(m, 4 * lane + TILE16_C_AT, at, 0);
    r.sc = __builtin_amdgcn_raw_buffer_load_b16(m, 2 * lane + TILE16_SC_AT, at, 0);
    r.d = __builtin_amdgcn_raw_buffer_load_b16(m, 2 * lane + TILE16_D_AT, at, 0);
    return r;
}
// unit64 -> tile16 (once, at load; out of place): a wave a tile, every lane reads its four sub-blocks of its row
__global__ void __launch_bounds__(256) k_iq3s_tile16(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int nrows, int ncols, long tiles) {
    const long t = (long) blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= tiles) return;
    const int lane = threadIdx.x & 63, nsuper = ncols >> 9, ks = ncols >> 5;
    const long per = (long) (nrows >> 4) * nsuper;   // tiles a matrix
    const long m = t / per, tl = t - m * per;
    const int R = (int) (tl / nsuper), S = (int) (tl - (long) R * nsuper);
    const uint8_t* we = src + (size_t) m * ((size_t) nrows * ks / 64 * UNIT_BYTES);
    const SuperFields f = super_load(we, 16 * R + (lane & 15), 16 * S + 4 * (lane >> 4), ks);
    uint8_t* u = dst + (size_t) t * TILE16_BYTES;
    *reinterpret_cast<v4u*>(u + 32 * lane) = f.a0;
    *reinterpret_cast<v4u*>(u + 32 * lane + 16) = f.a1;
    *reinterpret_cast<v4u*>(u + TILE16_B_AT + 16 * lane) = f.b;
    *reinterpret_cast<uint32_t*>(u + TILE16_C_AT + 4 * lane) = f.c;
    *reinterpret_cast<unsigned short*>(u + TILE16_SC_AT + 2 * lane) = (unsigned short) f.sc;
    *reinterpret_cast<unsigned short*>(u + TILE16_D_AT + 2 * lane) = (unsigned short) f.d;
}
// tokens of a job's tile that the wave forms (k_moe_mma_wave16.h) multiply at a time: four tiles of 16
constexpr int MB_TP = 4, MB_TOK64 = 16 * MB_TP;

}  // namespace fnx
