// Jobs of many rows over tile16 matrices, on the matrix cores, with no decoded weight in LDS.
//
// k_iq3s_jobs_mma (unit64: a lane = a sub-block of one row) has to turn its decoded rows by way of LDS before the matrix
// cores can take 16 rows of a sub-block at once, and the 16 waves' partial sums meet there too: the LDS is its limit.
// The prompt path's layout gives lane (r, g) of a wave four consecutive sub-blocks of row r of a tile of 16 rows - at
// step p sub-block 4 g + p of the tile's 16. v_mfma_i32_16x16x32_i8 wants a sub-block of 16 rows as lane (r, G): row r,
// bytes 8 G .. 8 G + 7. What the four lane groups hold after a step's decode - four sub-blocks, 32 bytes a lane - is
// that, for all four sub-blocks, up to a 4 x 4 transpose of 8-byte pairs between lane group and register pair: eight
// permlane swaps. Then one MFMA a sub-block gives the 16 x 16 integer sums, which take their scales and are added; no
// decoded weight ever reaches LDS. What is left for the LDS: the codebook lookups, the job's int8 activations (staged
// once a job, four 8-byte reads a lane and step), and the sixteen rows' scales of a sub-block, which go from the
// decoding lanes (row r) to the accumulator's (rows 4 G .. 4 G + 3) through a few words of the wave's own. A wave takes
// whole tiles of 16 rows and all the columns: no sums to add between waves, no barrier but those around a job's staging.
// out[job.out[j]][r] = W[job.w][r] . y[job.y[j]] as kernels.hpp:49 and moe.cuh:613-658 define it, a term as in
// k_iq3s_jobs_mma: d_w (1 + 2 s) d_x sumi; a row's sub-blocks are added in the order the steps give them
// (16 S + p + 4 j for S, then p, then j ascending), whatever the job's rows are.
#pragma once

#include "k_prefill.h"

namespace fnx {

constexpr int J16_THREADS = 1024, J16_WAVES = 16, J16_MAXCOLS = 2048;
constexpr int J16_XLD = J16_MAXCOLS + 32;   // bytes of a token's int8 row in LDS: a wave's 8-byte reads of a sub-block then take the two passes their 512 bytes need
typedef int j16_v4i __attribute__((ext_vector_type(4)));
// x's lanes 32 .. 63 <-> y's lanes 0 .. 31; x's 16-lane rows 1, 3 <-> y's rows 0, 2 (as instructions: see swap32_add)
__device__ __forceinline__ void swap32(uint32_t& x, uint32_t& y) { asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(x), "+v"(y)); }
__device__ __forceinline__ void swap16(uint32_t& x, uint32_t& y) { asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(x), "+v"(y)); }
// The signed codebook twice, entry i's two copies side by side (words 2 i and 2 i + 1): even lanes read the even words,
// odd lanes the odd ones, so the 64 random lookups of a wave instruction are two sets of 32 over 32 banks each.
template <int TOKS>   // tokens a unit
struct J16Lds {
    uint32_t tab[2 * SGRID_WORDS];
    __attribute__((aligned(16))) uint8_t xq[TOKS * J16_XLD];
    __attribute__((aligned(16))) float dx[(J16_MAXCOLS / 128) * TOKS * 4];   // [super-step][step p][token][lane group g]: the activations' block scales
    __attribute__((aligned(16))) float sw[J16_WAVES][4][16];                 // [wave][lane group][row]: a step's weight scales d (1 + 2 s)
};

// tiles [g0, g1) of 16 rows of matrix `we` (ncols columns) against the job's tokens, NT tiles of sixteen, staged in L: the whole block,
// after a barrier. f: the fields of the wave's first super-step. A step is decoded once for all NT tiles; a token's sums are the
// same whatever NT.
template <int NT, int TOKS>
__device__ __forceinline__ void j16_segment(J16Lds<TOKS>& L, const uint8_t* __restrict__ we, int g0, int g1, int ncols, const int* __restrict__ outs, int n,
                                            float* __restrict__ out, int out_stride, SuperFields f) {
    const int lane = threadIdx.x & 63, wave = uniform((int) (threadIdx.x >> 6));
    const int r = lane & 15, grp = lane >> 4;   // decoding: row r of the tile, lane group grp; accumulating: token r, rows 4 grp .. 4 grp + 3
    const int nsuper = ncols / 512;
    int oi[NT];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) oi[tt] = 16 * tt + r < n ? outs[16 * tt + r] : 0;
    const uint8_t* xrow = L.xq + r * J16_XLD + 8 * grp;   // bytes 8 grp .. of sub-block 16 S + 4 j + p of token r lie 512 S + 128 j + 32 p further
    float* myw = &L.sw[wave][grp][r];
    const uint32_t copy_at = 4u * (lane & 1);
    if (g0 + wave >= g1) return;
    for (int g = g0 + wave; g < g1; g += J16_WAVES) {
        float acc[NT][4];
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) acc[tt][0] = acc[tt][1] = acc[tt][2] = acc[tt][3] = 0.f;
        for (int S = 0; S < nsuper; ++S) {
            // the next super-step's fields (past the tile's last: the next tile of this wave, or this one again)
            const int gn = S + 1 < nsuper ? g : (g + J16_WAVES < g1 ? g + J16_WAVES : g);
            const SuperFields nf = tile16_load_buf(tile16_rsrc(we, gn, nsuper), S + 1 < nsuper ? S + 1 : 0);
            auto step = [&](auto p_c) {
                constexpr int p = decltype(p_c)::value;
                const SubFields s = super_sub<p>(f);
                const v4u idx = {s.q0, s.q1, s.q2, s.q3};
                uint32_t w8[8];   // this lane's sub-block (row r, 16 S + 4 grp + p): 32 int8
#pragma unroll
                for (int j = 0; j < 8; ++j) w8[j] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(L.tab) + 2 * packed_addr(idx, j) + copy_at);
                *myw = half_bits_to_float(s.d) * (float) (int) (1u + 2u * s.sc);
                // pair P_k = bytes 8 k .. 8 k + 7 of the lane's sub-block; afterwards pair j holds bytes 8 grp .. of lane group j's
                swap32(w8[0], w8[4]);
                swap32(w8[1], w8[5]);
                swap32(w8[2], w8[6]);
                swap32(w8[3], w8[7]);
                swap16(w8[0], w8[2]);
                swap16(w8[1], w8[3]);
                swap16(w8[4], w8[6]);
                swap16(w8[5], w8[7]);
                float4 fw[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) fw[j] = *reinterpret_cast<const float4*>(&L.sw[wave][j][4 * grp]);
#pragma unroll
                for (int tt = 0; tt < NT; ++tt) {
                    long b[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const long*>(xrow + 16 * tt * J16_XLD + 512 * S + 128 * j + 32 * p);
                    const float4 dxv = *reinterpret_cast<const float4*>(&L.dx[((S * 4 + p) * TOKS + 16 * tt + r) * 4]);
                    const float dxs[4] = {dxv.x, dxv.y, dxv.z, dxv.w};
#pragma unroll
                    for (int j = 0; j < 4; ++j) {   // lane group j's sub-block, 16 S + 4 j + p
                        const long a = (long) ((unsigned long) w8[2 * j] | (unsigned long) w8[2 * j + 1] << 32);
                        const j16_v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b[j], j16_v4i{0, 0, 0, 0}, 0, 0, 0);
                        acc[tt][0] = fmaf(fw[j].x * dxs[j], (float) d[0], acc[tt][0]);
                        acc[tt][1] = fmaf(fw[j].y * dxs[j], (float) d[1], acc[tt][1]);
                        acc[tt][2] = fmaf(fw[j].z * dxs[j], (float) d[2], acc[tt][2]);
                        acc[tt][3] = fmaf(fw[j].w * dxs[j], (float) d[3], acc[tt][3]);
                    }
                }
            };
            step(std::integral_constant<int, 0>{});
            step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{});
            step(std::integral_constant<int, 3>{});
            f = nf;
        }
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
            if (16 * tt + r < n) {
                float* op = out + (size_t) oi[tt] * out_stride + 4 * grp + 16 * g;
                op[0] = acc[tt][0], op[1] = acc[tt][1], op[2] = acc[tt][2], op[3] = acc[tt][3];
            }
    }
}

// tile16 matrices of up to 2048 columns (a multiple of 512), rows in 16s.
// MODE 0: jobs of up to FNX_MAXT rows (kernels.hpp:18-23) over q8_1 rows: the blocks split the (job, tile of 16 rows) items of all jobs
// evenly and walk them in order; a job's activations are staged when the block comes to it.
// (A job's first weights are asked for ahead of its activations: 160 jobs of one row gate|up 39.9 -> 38.5 us and down 30.9 -> 29.8, ten of 16
// rows 17.6 -> 16.7 and 14.4 as before.)
// MODE 1: the prompt path's jobs of up to FNX_PF_JOB rows (kernels.hpp:324, moe_gate_up_big): a job's rows in units of up to two
// token tiles, so that a weight is decoded once for both. A unit of nt token tiles costs J16_DEC + J16_MUL nt for each of its
// rounds, J16_ROUND tiles of 16 rows; the blocks split the costs of all rounds evenly (a prefix sum over the jobs in LDS) and each
// takes the rounds that begin in its share. Lists of so few tiles that the blocks have no more than J16_SINGLE each are bound by a
// tile's chain of steps and by what comes before it: there a unit is one token tile, and up to a tile a wave a round is as many
// tiles as leave every block a round of one unit, where that can be - a second unit would be staged after the first.
// MODE 2 (kernels.hpp:325, moe_down_big): the same with the unit's activations made on the way from the rows [gate | up] of 2 ncols floats:
// h = silu(gate) * up quantised as k_swiglu_q8_1 does it, four threads a sub-block.
constexpr int J16_MAXJOBS = 4096;   // big jobs a launch (their token counts and costs live in LDS)
// us a chunk of 512 experts, Zipf (a decode for every sixteen tokens, jobs' starts looked up in memory as their turn came / this), 300
// rows: 192 / 171, 1,024: 389 / 335, 4,096: 1,302 / 1,014; 77 rows, uniform: 234 / 210; the shared expert's launches over 300 rows 23.6 / 18.1 and
// 30.5 / 20.5. Rounds of 8 tiles are the same within the noise (173, 336, 1,019, 212), of 16 slower (182, 337, 1,026, 219): a unit's
// last tiles and the block's run come out less even. Four token tiles a unit (of up to 1024 columns; sums spill) were slower: 40.9 -> 46
// us a down launch of 300 rows.
// J16_SINGLE: us a launch of gate|up (1,024 x 2,048) and down (2,048 x 512), units of one token tile up to 16 / 24 / 32 tiles a block: 17
// jobs of 64 rows 29.5 / 26.9 / 26.8 and 27, ten 17.1 and 24.8 / 17.7 / 17.7, 24 of them 29.7 / 29.1 / 29.1 and 28, 32 26.3 / 26.6 / 33.4 and
// 24.2. What comes before a block's first tile is a launch of its own size: a job of one row 11.5 and 8.7 us with the costs' sums
// exchanged through LDS and a division for each rule, 10.0 and 7.3 with DPP moves and divisions only where a list needs them.
constexpr int J16_SINGLE = 24, J16_ROUND = 4, J16_DEC = 3, J16_MUL = 2;
static_assert(J16_MAXJOBS * (FNX_PF_JOB / 32) * (J16_DEC + 2 * J16_MUL) < 65536, "the costs' sum in 16 bits");

// the sum of the wave's lanes up to and including this one (DPP moves: an exchange through LDS is a trip of its own a step)
__device__ __forceinline__ uint32_t wave_running(uint32_t v) {
#define FNX_DPP_ADDU(ctrl, rmask) v += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) v, ctrl, rmask, 0xF, false)
    FNX_DPP_ADDU(0x111, 0xF);   // row_shr:1, 2, 4, 8
    FNX_DPP_ADDU(0x112, 0xF);
    FNX_DPP_ADDU(0x114, 0xF);
    FNX_DPP_ADDU(0x118, 0xF);
    FNX_DPP_ADDU(0x142, 0xA);   // row_bcast15 into rows 1 and 3
    FNX_DPP_ADDU(0x143, 0xC);   // row_bcast31 into rows 2 and 3
#undef FNX_DPP_ADDU
    return v;
}
// a unit's activations (n tokens, toks places) to LDS
template <int MODE, int TOKS>
__device__ __forceinline__ void j16_stage(J16Lds<TOKS>& L, const RowsArgs& a, const uint8_t* y, const int* ys, int n, int toks) {
    const int nsb = a.ncols / 32;
    if constexpr (MODE == 2) {
        for (int q = threadIdx.x; q < 4 * toks * nsb; q += J16_THREADS) {   // (token, sub-block, quarter): 8 values (the four threads of a sub-block are neighbours)
            const int s = q >> 2, part = q & 3, t = s / nsb, sb = s - t * nsb;
            uint32_t v[2] = {0u, 0u};
            float d = 0.f;
            if (t < n) {
                const float* gp = a.gu + (size_t) ys[t] * (2 * a.ncols) + 32 * sb + 8 * part;
                float4 gv[2], uv[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) gv[k] = reinterpret_cast<const float4*>(gp)[k], uv[k] = reinterpret_cast<const float4*>(gp + a.ncols)[k];
                float h[8], amax = 0.f;
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    h[4 * k] = silu_f(gv[k].x) * uv[k].x, h[4 * k + 1] = silu_f(gv[k].y) * uv[k].y;
                    h[4 * k + 2] = silu_f(gv[k].z) * uv[k].z, h[4 * k + 3] = silu_f(gv[k].w) * uv[k].w;
                }
#pragma unroll
                for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(h[k]));
                amax = fmaxf(amax, __shfl_xor(amax, 1));
                amax = fmaxf(amax, __shfl_xor(amax, 2));
                const float dq = amax / 127.0f;   // q8_1_store's arithmetic (kernels.cu:131-145)
                d = half_bits_to_float(float_to_half_bits(dq));
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    uint32_t word = 0;
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const int8_t qv = amax == 0.0f ? (int8_t) 0 : (int8_t) roundf(h[4 * k + b] / dq);
                        word |= (uint32_t) (uint8_t) qv << (8 * b);
                    }
                    v[k] = word;
                }
            }
            *reinterpret_cast<uint2*>(L.xq + t * J16_XLD + 32 * sb + 8 * part) = make_uint2(v[0], v[1]);
            if (part == 0) L.dx[(((sb >> 4) * 4 + (sb & 3)) * TOKS + t) * 4 + ((sb >> 2) & 3)] = d;
        }
    } else {
        for (int q = threadIdx.x; q < toks * nsb; q += J16_THREADS) {   // (token, sub-block): its 32 int8 and its scale
            const int t = q / nsb, sb = q - t * nsb;
            uint32_t v[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
            float d = 0.f;
            if (t < n) {
                const uint8_t* yb = y + ((size_t) ys[t] * nsb + sb) * FNX_Q8_1_BLOCK;
                d = half_bits_to_float(*reinterpret_cast<const unsigned short*>(yb));
#pragma unroll
                for (int k = 0; k < 8; ++k) v[k] = *reinterpret_cast<const uint32_t*>(yb + 4 + 4 * k);
            }
            uint32_t* dst = reinterpret_cast<uint32_t*>(L.xq + t * J16_XLD + 32 * sb);
#pragma unroll
            for (int k = 0; k < 8; ++k) dst[k] = v[k];
            L.dx[(((sb >> 4) * 4 + (sb & 3)) * TOKS + t) * 4 + ((sb >> 2) & 3)] = d;
        }
    }
}

template <int MODE>
__global__ void __launch_bounds__(J16_THREADS) k_iq3s_jobs_mma16(const RowsArgs a) {
    __shared__ J16Lds<MODE ? 2 * FNX_MAXT : FNX_MAXT> L;
    __shared__ uint8_t jn[MODE ? J16_MAXJOBS : 1];            // the jobs' tokens
    __shared__ unsigned short before[MODE ? J16_MAXJOBS + 2 : 1];   // costs of the jobs before job j, a round of each of their units
    __shared__ int tiles_sum;
    const int lane = threadIdx.x & 63, wave = uniform((int) (threadIdx.x >> 6));
    const int nj_raw = a.njobs ? *a.njobs : a.njobs_max;
    const uint32_t code0 = g_sgrid.v[threadIdx.x & 511];
    const int nj = max(0, min(min(uniform(nj_raw), a.njobs_max), MODE ? J16_MAXJOBS : a.njobs_max));
    // the token counts of the jobs that count, on their way while the codebook is written
    int hn[MODE ? J16_MAXJOBS / J16_THREADS : 1] = {};
    if constexpr (MODE != 0) {
#pragma unroll
        for (int i = 0; i < J16_MAXJOBS / J16_THREADS; ++i) {
            const int j = (int) threadIdx.x + i * J16_THREADS;
            if (j < nj) hn[i] = a.big[j].n;
        }
    }
    if (threadIdx.x < 512) {   // a code's sixteen signed entries from its unsigned one
        const int g = threadIdx.x;
#pragma unroll
        for (int sg = 0; sg < 16; ++sg) L.tab[2 * (sg * 512 + g)] = L.tab[2 * (sg * 512 + g) + 1] = signed_entry(code0, sg);
    }
    const uint32_t gpj = (uint32_t) a.nrows / 16;   // items per unit
    const uint8_t* y = a.y ? a.y : g_moe_hq;
    const int nsuper = a.ncols / 512;
    if constexpr (MODE == 0) {
        const unsigned long long total = (unsigned long long) nj * gpj;
        uint32_t i = (uint32_t) (total * blockIdx.x / gridDim.x);
        const uint32_t i1 = (uint32_t) (total * (blockIdx.x + 1) / gridDim.x);
        while (i < i1) {
            const uint32_t ui = i / gpj;
            const int g0 = (int) (i - ui * gpj), g1 = (int) min(gpj, g0 + (i1 - i));
            const fnx_job* jb = a.jobs + ui;
            const int n = uniform(min(jb->n, FNX_MAXT)), w = uniform(jb->w);
            i += (uint32_t) (g1 - g0);
            if (n < 1) continue;   // the same for the whole block; a job without rows names no matrix
            const uint8_t* we = a.ep ? uniform_ptr(a.ep[w]) : a.wbase + (size_t) w * a.w_stride;
            const SuperFields f = tile16_load_buf(tile16_rsrc(we, min(g0 + wave, g1 - 1), nsuper), 0);
            __syncthreads();   // the unit before has been read (and the codebook written)
            j16_stage<0>(L, a, y, jb->y, n, FNX_MAXT);
            __syncthreads();
            j16_segment<1>(L, we, g0, g1, a.ncols, jb->out, n, a.out, a.out_stride, f);
        }
    } else {
#pragma unroll
        for (int i = 0; i < J16_MAXJOBS / J16_THREADS; ++i) {
            const int j = (int) threadIdx.x + i * J16_THREADS;
            if (j < nj) jn[j] = (uint8_t) min(max(hn[i], 0), FNX_PF_JOB);
        }
        __syncthreads();
        constexpr uint32_t C1 = J16_DEC + J16_MUL, C2 = J16_DEC + 2 * J16_MUL;   // a round's cost in a unit of one token tile, of two
        if (wave == 0) {
            // the jobs' token tiles (high half) and their costs as units of two token tiles (low half), their running sums made
            // together: a lane takes a run of jobs
            const int per = (nj + 63) / 64, j0 = min(nj, lane * per), j1 = min(nj, j0 + per);
            auto of_job = [&](int j) {
                const uint32_t t = (jn[j] + 15u) >> 4;
                return t << 16 | ((t >> 1) * C2 + (t & 1) * C1);
            };
            uint32_t mine = 0;
            for (int j = j0; j < j1; ++j) mine += of_job(j);
            const uint32_t incl = wave_running(mine);
            const uint32_t tiles = (uint32_t) __builtin_amdgcn_readlane((int) incl, 63) >> 16;
            const int half = (unsigned long long) tiles * gpj <= (unsigned long long) J16_SINGLE * gridDim.x ? 16 : 0;   // units of one token tile count as one
            uint32_t run = incl - mine;
            if (lane == 0) before[0] = 0, tiles_sum = (int) tiles;
            for (int j = j0; j < j1; ++j) {
                run += of_job(j);
                before[j + 1] = (unsigned short) (run >> half);
            }
        }
        __syncthreads();
        const uint32_t tiles = (uint32_t) uniform(tiles_sum);
        const bool single = (unsigned long long) tiles * gpj <= (unsigned long long) J16_SINGLE * gridDim.x;
        uint32_t round = J16_ROUND, rpu = (gpj + J16_ROUND - 1) / J16_ROUND;   // tiles a round, rounds a unit
        if (single && tiles * gpj <= J16_WAVES * gridDim.x) {   // the smallest with a round a block at most, or a tile a wave
            round = 1, rpu = gpj;
            if (tiles * gpj > gridDim.x) {
                round = (tiles * gpj + gridDim.x - 1) / gridDim.x, rpu = (gpj + round - 1) / round;
                for (; round < (uint32_t) J16_WAVES && tiles * rpu > gridDim.x; rpu = (gpj + round - 1) / round) ++round;
            }
        }
        const int ut = single ? 1 : 2;   // token tiles a unit
        const uint32_t whole = (single ? 1u : C2) * rpu;
        // the block's share of the costs: the blocks' shares differ by one at most
        const unsigned long long total = (unsigned long long) before[nj] * rpu;
        const unsigned long long each = total >> 32 ? total / gridDim.x : total < gridDim.x ? 0u : (uint32_t) total / gridDim.x, rest = total - each * gridDim.x;
        unsigned long long c = each * blockIdx.x + min((unsigned long long) blockIdx.x, rest);
        const unsigned long long c1 = c + each + (blockIdx.x < rest ? 1u : 0u);
        while (c < c1) {   // the same for the whole block
            int lo = 0, hi = nj - 1;   // the job that c falls in: before[j] rpu <= c < before[j + 1] rpu
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if ((unsigned long long) before[mid + 1] * rpu <= c) lo = mid + 1;
                else hi = mid;
            }
            lo = uniform(lo);
            const fnx_bigjob* jb = a.big + lo;
            // its unit q, which begins at `at`, and the unit's rounds from the first that begins at or after c
            const unsigned long long jat = (unsigned long long) before[lo] * rpu;
            const int nall = uniform((int) jn[lo]), q = nall > 16 * ut ? uniform((int) ((uint32_t) (c - jat) / whole)) : 0;
            const unsigned long long at = jat + (unsigned long long) q * whole;
            const int n = min(nall - 16 * ut * q, 16 * ut), nt = (n + 15) / 16, w = uniform(jb->w);
            const uint32_t end = (single ? 1u : nt == 1 ? C1 : C2) * rpu;   // the unit's costs
            uint32_t k0 = (uint32_t) (c - at), k1 = c1 - at >= end ? end : (uint32_t) (c1 - at);
            if (!single) {
                k0 = nt == 1 ? (k0 + C1 - 1) / C1 : (k0 + C2 - 1) / C2;
                k1 = nt == 1 ? (k1 + C1 - 1) / C1 : (k1 + C2 - 1) / C2;
            }
            c = at + end;
            const int g0 = uniform((int) (k0 * round)), g1 = uniform((int) min(gpj, k1 * round));
            if (g0 >= g1) continue;
            const int *ys = jb->y + 16 * ut * q, *outs = jb->out + 16 * ut * q;
            const uint8_t* we = a.ep ? uniform_ptr(a.ep[w]) : a.wbase + (size_t) w * a.w_stride;
            const SuperFields f = tile16_load_buf(tile16_rsrc(we, min(g0 + wave, g1 - 1), nsuper), 0);
            __syncthreads();   // the unit before has been read (and the codebook written)
            j16_stage<MODE>(L, a, y, ys, n, 16 * nt);
            __syncthreads();
            if (nt == 1) j16_segment<1>(L, we, g0, g1, a.ncols, outs, n, a.out, a.out_stride, f);
            else j16_segment<2>(L, we, g0, g1, a.ncols, outs, n, a.out, a.out_stride, f);
        }
    }
}

}  // namespace fnx
