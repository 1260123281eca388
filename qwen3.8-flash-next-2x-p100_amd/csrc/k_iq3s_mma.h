// Jobs of many rows over unit64 matrices of 2048 columns (a unit = one weight row), on the matrix cores.
//
// The vector-ALU job kernel dots a decoded sub-block with one or two tokens; with sixteen tokens a job that is eight
// decodes of every weight, or sixteen dot products a decode. Here a block of 16 waves takes 16 weight rows at a time:
//   1. wave w decodes row 16 g + w as the mat-vec kernels do (lane = sub-block, 8 codebook lookups: 32 int8 weights a lane)
//      and stores them, the sub-block's integer scale and the row's d in LDS;
//   2. wave w then owns sub-blocks 4 w .. 4 w + 3 of all 16 rows: v_mfma_i32_16x16x32_i8 takes the 16 rows x 32 columns
//      of one sub-block as A (8 bytes a lane from LDS) and the job's up to 16 tokens' int8 activations of that sub-block
//      as B (in registers for the whole job), and leaves every lane four exact integer dot products; each takes its
//      scales (the reference's term (d_w * d_x) * (float) (sumi * (1 + 2 s)), moe.cuh's vec_dot, as d_w (1 + 2 s) * d_x * sumi) and
//      is added to the lane's four sums;
//   3. the waves' sums (each over 128 columns) meet in LDS and one wave adds them in wave order and stores the 16 x 16 tile.
// A weight is decoded once per job whatever the job's rows. Jobs of one row keep the vector-ALU path (its waves
// share a block's run of units). (kernels.hpp:49, moe.cuh:613-658 give the semantics: out[job.out[j]][r] =
// W[job.w][r] . y[job.y[j]].)
#pragma once

#include "k_iq3s_packed.h"

namespace fnx {

constexpr int JM_THREADS = 1024, JM_WAVES = 16, JM_ROWS = 16;
constexpr int JM_ROWLD = 2048 + 32;   // bytes of a decoded row in LDS: 64 sub-blocks x 32 int8, padded so that rows m and m + 1 start 8 banks apart
constexpr int JM_SLD = 20;            // floats of a sub-block's scale record: its 16 rows + 4 (records 16-byte aligned, 20 words apart)
constexpr int JM_MIN = 2;             // rows from which a job goes to the matrix cores (two tokens a pass on the vector ALU does not fit 128 registers with four units in flight)
constexpr int JM_AHEAD = 3;           // units a wave has in flight beyond the one it decodes
typedef int jm_v4i __attribute__((ext_vector_type(4)));

constexpr int JM_NI = 2;   // groups of 16 rows between two barriers: each wave decodes JM_NI rows, then multiplies its sub-blocks of JM_NI tiles
struct JmLds {
    uint32_t tab[SGRID_WORDS];
    __attribute__((aligned(16))) uint8_t tile[JM_NI][JM_ROWS * JM_ROWLD];
    __attribute__((aligned(16))) float sw[JM_NI][64][JM_SLD];   // [sub-block][row]: d (1 + 2 s), exact in f32 (11 + 5 bits): a lane's four rows are one 16-byte read
    __attribute__((aligned(16))) float red[JM_NI][JM_WAVES][64][4];
};
template <int SBR>
struct JmOneLds {   // for one group of 16 units: 71 to 74 KB, two blocks a CU
    union {
        uint32_t tab[SGRID_WORDS];
        __attribute__((aligned(16))) float red[1][JM_WAVES][64][4];   // (when every row has been decoded)
    };
    __attribute__((aligned(16))) uint8_t tile[1][JM_ROWS * (64 / SBR) * (32 * SBR + 32)];
    __attribute__((aligned(16))) float sw[1][64][JM_SLD];
};

// the job's activations of a wave's four sub-blocks: token col's bytes 8 kg .. 8 kg + 7 and its block scale. A lane past the job's tokens
// loads the first one's, and its column of the products is thrown away: loads under a condition go out one by one, a trip to
// memory each. (The first one's row is taken by the whole wave: read under the condition it would be the first lane's past the job's
// tokens, and what an entry past a job's rows holds names no row)
struct JmActs {
    uint32_t lo[4], hi[4], dh[4];
    // (sub-blocks sb0, sb0 + step, ..)
    template <int SBR = 64>
    __device__ __forceinline__ void load(const uint8_t* __restrict__ y, int yi, bool on, int sb0, int kg, int step = 1) {
        const int first = uniform(yi);
        const uint8_t* yr = y + ((size_t) (on ? yi : first) * SBR + sb0) * FNX_Q8_1_BLOCK;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const uint8_t* yb = yr + s * step * FNX_Q8_1_BLOCK;
            lo[s] = *reinterpret_cast<const uint32_t*>(yb + 4 + 8 * kg);
            hi[s] = *reinterpret_cast<const uint32_t*>(yb + 8 + 8 * kg);
            dh[s] = *reinterpret_cast<const unsigned short*>(yb);
        }
    }
};
// 1. this wave's unit of group i: 32 int8 weights a lane (SBR sub-blocks a row: row wave of the group, or its 64 / SBR rows from there on)
template <int SBR = 64, class Lds>
__device__ __forceinline__ void jm_decode(Lds& L, int i, int wave, int lane, const PackedSub& cur) {
    v4u lo, hi;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        lo[j] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(L.tab) + packed_addr(cur.idx, j));
        hi[j] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(L.tab) + packed_addr(cur.idx, 4 + j));
    }
    const int row = wave * (64 / SBR) + lane / SBR, sb = lane % SBR;
    uint8_t* dst = L.tile[i] + row * (32 * SBR + 32) + sb * 32;
    *reinterpret_cast<v4u*>(dst) = lo;
    *reinterpret_cast<v4u*>(dst + 16) = hi;
    const uint32_t sc = 1u + 2u * ((cur.sc >> (4 * (lane & 1))) & 0xFu);
    float* sw = &L.sw[i][row / JM_ROWS * SBR + sb][row % JM_ROWS];
    if constexpr (SBR < 64) *reinterpret_cast<uint32_t*>(sw) = (uint32_t) (unsigned short) cur.d | sc << 16;
    else *sw = half_bits_to_float(cur.d) * (float) (int) sc;
}
// 2. this wave's four sub-blocks of group i's 16 rows against the tokens. Shorter rows: of the 16 rows that W = SBR / 4 waves share, sub-blocks
// w, w + W, w + 2 W, w + 3 W, whose terms, formed as the mat-vec kernels form them, meet in the first two levels of the butterfly over a row;
// jm_store goes through the others. A row's bits are then those of the kernels for jobs of one and two rows and of the streaming ones,
// whatever the job's length. (In the order that the rows of 2,048 columns have they depended on it, at the same speed.)
template <int SBR = 64, class Lds>
__device__ __forceinline__ void jm_multiply(Lds& L, int i, int wave, int lane, const JmActs& x, const float (&dx)[4]) {
    const int col = lane & 15, kg = lane >> 4;
    if constexpr (SBR < 64) {
        constexpr int W = SBR / 4;
        const int rg = wave / W;
        float term[4][4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int sb = wave % W + s * W;
            const long a = *reinterpret_cast<const long*>(L.tile[i] + (JM_ROWS * rg + col) * (32 * SBR + 32) + sb * 32 + 8 * kg);
            const v4u f = *reinterpret_cast<const v4u*>(&L.sw[i][rg * SBR + sb][4 * kg]);
            const long xb = (long) ((unsigned long) x.lo[s] | (unsigned long) x.hi[s] << 32);
            const jm_v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, xb, jm_v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) term[s][v] = (half_bits_to_float(f[v]) * dx[s]) * (float) __mul24(d[v], (int) (f[v] >> 16));
        }
        float z[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) z[v] = (term[0][v] + term[2][v]) + (term[1][v] + term[3][v]);
        *reinterpret_cast<float4*>(L.red[i][wave][lane]) = make_float4(z[0], z[1], z[2], z[3]);
        return;
    }
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int sb = 4 * wave + s;
        const long a = *reinterpret_cast<const long*>(L.tile[i] + col * JM_ROWLD + sb * 32 + 8 * kg);
        const float4 f = *reinterpret_cast<const float4*>(&L.sw[i][sb][4 * kg]);
        const long xb = (long) ((unsigned long) x.lo[s] | (unsigned long) x.hi[s] << 32);
        const jm_v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, xb, jm_v4i{0, 0, 0, 0}, 0, 0, 0);
        // a term is d_w (1 + 2 s) d_x sumi: the reference's (d_w d_x) (float) (sumi (1 + 2 s)) with the factors taken in another order
        acc[0] = fmaf(f.x * dx[s], (float) d[0], acc[0]);
        acc[1] = fmaf(f.y * dx[s], (float) d[1], acc[1]);
        acc[2] = fmaf(f.z * dx[s], (float) d[2], acc[2]);
        acc[3] = fmaf(f.w * dx[s], (float) d[3], acc[3]);
    }
    *reinterpret_cast<float4*>(L.red[i][wave][lane]) = make_float4(acc[0], acc[1], acc[2], acc[3]);
}
// 3. one wave adds group i's sums of the sixteen in wave order (shorter rows: of the SBR / 4 from wave w0 on, in the butterfly's) and stores the tile
template <int SBR = 64, class Lds>
__device__ __forceinline__ void jm_store(const Lds& L, int i, int lane, float* op, int w0 = 0) {
    constexpr int W = SBR / 4;
    auto sum_of = [&](int w) { return *reinterpret_cast<const float4*>(L.red[i][w0 + w][lane]); };
    auto plus = [](float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); };
    float4 z;
    if constexpr (SBR == 64) {
        z = sum_of(0);
#pragma unroll
        for (int w = 1; w < W; ++w) z = plus(z, sum_of(w));
    } else {
        float4 p[W];
#pragma unroll
        for (int w = 0; w < W; ++w) p[w] = sum_of(w);
#pragma unroll
        for (int o = W / 2; o >= 1; o /= 2)
#pragma unroll
            for (int w = 0; w < o; ++w) p[w] = plus(p[w], p[w + o]);
        z = p[0];
    }
    op[0] = z.x, op[1] = z.y, op[2] = z.z, op[3] = z.w;
}

// rows [16 g0, 16 g1) of matrix `we` against the job's tokens: the whole block. between() runs when the first weights and the activations
// are on their way (the block's first run writes the codebook there)
template <class Between>
__device__ __forceinline__ void jm_segment(JmLds& L, const uint8_t* __restrict__ we, int g0, int g1, const fnx_job* jb, int n,
                                           const uint8_t* __restrict__ y, float* __restrict__ out, int out_stride, Between between) {
    const int lane = threadIdx.x & 63, wave = uniform((int) (threadIdx.x >> 6));
    const int col = lane & 15, kg = lane >> 4;   // as B column / accumulator column: token col; as A row: weight row col of the 16
    const int yi = jb->y[col], oi = jb->out[col];   // (they mean something below n; asked for before the weights, or waiting for them waits for those too)
    const PackedVOffs o = packed_voffs(lane);
    const __amdgpu_buffer_rsrc_t mtx = matrix_rsrc(we);
    auto load = [&](int g) { return load_packed_buf(mtx, (JM_ROWS * min(g, g1 - 1) + wave) * UNIT_BYTES, o); };   // past the end: the last group again
    constexpr int RING = JM_AHEAD + 1;
    static_assert(RING % JM_NI == 0, "a round takes whole slots of the ring");
    PackedSub ring[RING];
#pragma unroll
    for (int i = 0; i < RING; ++i) ring[i] = load(g0 + i);
    JmActs x;
    x.load(y, yi, col < n, 4 * wave, kg);
    float* orow = out + (size_t) (col < n ? oi : 0) * out_stride + 4 * kg;   // token col's row of the output, this lane's four rows of a tile
    between();
    float dx[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) dx[s] = half_bits_to_float(x.dh[s]);
    for (int gb = g0; gb < g1; gb += RING)
#pragma unroll
    for (int rb = 0; rb < RING; rb += JM_NI) {   // the ring's slots in turn: no register moves
        const int g = gb + rb;   // this round: groups g .. g + JM_NI - 1 (those below g1)
        if (g >= g1) break;
#pragma unroll
        for (int i = 0; i < JM_NI; ++i) {
            const PackedSub cur = ring[rb + i];
            ring[rb + i] = load(g + i + RING);
            jm_decode(L, i, wave, lane, cur);
        }
        __syncthreads();   // the rows are in LDS
#pragma unroll
        for (int i = 0; i < JM_NI; ++i) jm_multiply(L, i, wave, lane, x, dx);
        __syncthreads();   // the waves' sums are in LDS (and the tiles have been read: the next decode may overwrite them)
#pragma unroll
        for (int i = 0; i < JM_NI; ++i)   // (the waves take turns)
            if (g + i < g1 && wave == ((g + i - g0) & (JM_WAVES - 1)) && col < n) jm_store(L, i, lane, orow + JM_ROWS * (g + i));
    }
}

// 16 units of a matrix of nunits (16 rows, or 64 / SBR times as many shorter ones) against the job's tokens, and nothing after them: a wave
// decodes one, no ring and no second group. Past the last unit: that one again, its rows not stored. Over rows of 2,048 columns the sums are
// jm_segment's bit for bit, over shorter ones butterfly_sum's.
template <int SBR, class Between>
__device__ __forceinline__ void jm_group(JmOneLds<SBR>& L, const uint8_t* __restrict__ we, int g, int nunits, const fnx_job* jb, int n, const uint8_t* __restrict__ y,
                                         float* __restrict__ out, int out_stride, Between between) {
    const int lane = threadIdx.x & 63, wave = uniform((int) (threadIdx.x >> 6));
    const int col = lane & 15, kg = lane >> 4;
    const int yi = jb->y[col], oi = jb->out[col];
    const PackedSub cur = load_packed_buf(matrix_rsrc(we), min(16 * g + wave, nunits - 1) * UNIT_BYTES, packed_voffs(lane));
    JmActs x;
    if constexpr (SBR < 64) x.load<SBR>(y, yi, col < n, wave % (SBR / 4), kg, SBR / 4);
    else x.load<SBR>(y, yi, col < n, 4 * wave, kg);
    between();
    jm_decode<SBR>(L, 0, wave, lane, cur);
    __syncthreads();   // the rows are in LDS
    float dx[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        asm volatile("" : "+v"(x.dh[s]));   // (converted here: before, the decode would wait for the activations)
        dx[s] = half_bits_to_float(x.dh[s]);
    }
    jm_multiply<SBR>(L, 0, wave, lane, x, dx);
    __syncthreads();   // the waves' sums are in LDS
    const int row = JM_ROWS * (64 / SBR * g + wave / (SBR / 4)) + 4 * kg;
    if (wave % (SBR / 4) == 0 && col < n && row < 64 / SBR * nunits) jm_store<SBR>(L, 0, lane, out + (size_t) oi * out_stride + row, wave);
}

// units [u0, u1) of matrix `we` for a job of one row: the block's waves share them, each a contiguous run. between(): as in jm_segment
template <class Between>
__device__ __forceinline__ void jm_narrow(const uint32_t* tab, const uint8_t* we, int u0, int u1, const fnx_job* jb, const uint8_t* y,
                                          float* out, int out_stride, Between between) {
    const int wave = uniform((int) (threadIdx.x >> 6)), per = (u1 - u0 + JM_WAVES - 1) / JM_WAVES;
    const int ua = u0 + wave * per, ub = min(u1, ua + per);
    PackedSub cur[4];
    if (ua < ub) packed_first(we, ua, ub, cur);
    between();
    if (ua >= ub) return;
    packed_units<64, 1>(tab, we, ua, ub, cur, JobPrep<64, 1>{jb, 0, y, out, out_stride});
}

// The same for a block's first run where it leaves a wave U rows or fewer (a matrix of up to 1024 U rows a CU's block has
// alone: the lone mat-vec). There is nothing to stream: the time is the launch and the trips to memory one after the other, so the rows
// and the activations are asked for before the codebook is written to LDS (between() does that, and meets), and only the U rows are
// decoded - the loop above decodes four, asks for four more, and with sixteen waves a CU that was a third of the launch.
template <int U, int SBR = 64, class Between>
__device__ __forceinline__ void jm_few(const uint32_t* tab, const uint8_t* we, int u0, int u1, int yi, int oi, const uint8_t* y, float* out, int out_stride,
                                       Between between) {
    const int lane = threadIdx.x & 63, wave = uniform((int) (threadIdx.x >> 6)), ua = u0 + wave * U;
    const PackedOffs o = packed_offs(lane);
    PackedSub cur[U];
#pragma unroll
    for (int r = 0; r < U; ++r) cur[r] = load_packed(as_global(uniform_ptr(we + (size_t) min(ua + r, u1 - 1) * UNIT_BYTES)), o);
    const uint8_t* yb = y + ((size_t) yi * SBR + lane % SBR) * FNX_Q8_1_BLOCK;
    int xs[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) xs[j] = reinterpret_cast<const int*>(yb + 4)[j];
    const float dx = half_bits_to_float(*reinterpret_cast<const unsigned short*>(yb));
    between();
    float v[U];
#pragma unroll
    for (int r = 0; r < U; ++r) {
        int sum = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            sum = __builtin_amdgcn_sdot4(*reinterpret_cast<const int*>(reinterpret_cast<const uint8_t*>(tab) + packed_addr(cur[r].idx, j)), xs[j], sum, false);
        v[r] = (half_bits_to_float(cur[r].d) * dx) * (float) __mul24(sum, 1 + 2 * (int) ((cur[r].sc >> (4 * (lane & 1))) & 0xFu));
    }
    float* orow = out + (size_t) oi * out_stride;
    if constexpr (U == 4) {   // (packed_units' sums)
        const int ur = reduce4_unit_of_row(lane >> 4);
        const float z = reduce4_units(v[0], v[1], v[2], v[3]);
        if ((lane & 15) == 0 && ua + ur < u1) orow[ua + ur] = z;
    } else {
#pragma unroll
        for (int r = 0; r < U; ++r) {
            const float z = butterfly_sum<SBR>(v[r]);
            if (lane % SBR == SBR - 1 && ua + r < u1) orow[(size_t) (ua + r) * (64 / SBR) + lane / SBR] = z;
        }
    }
}

// A unit a wave against two rows of activations, over rows of SBR < 64 sub-blocks: no trip of the decoded weights through LDS and no second meeting
// (9,600 rows of 1,024 columns, two rows, with their quantisation: 8.9 us by jm_group, 7.6 here, 8.5 before)
template <int SBR, class Between>
__device__ __forceinline__ void jm_two(const uint32_t* tab, const uint8_t* we, int u, int nunits, const fnx_job* jb, const uint8_t* y, float* out, int out_stride,
                                       Between between) {
    const int lane = threadIdx.x & 63, y0 = uniform(jb->y[0]), y1 = uniform(jb->y[1]), o0 = uniform(jb->out[0]), o1 = uniform(jb->out[1]);
    const PackedSub cur = load_packed(as_global(uniform_ptr(we + (size_t) min(u, nunits - 1) * UNIT_BYTES)), packed_offs(lane));
    int xs[2][8];
    float dx[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint8_t* yb = y + ((size_t) (t ? y1 : y0) * SBR + lane % SBR) * FNX_Q8_1_BLOCK;
#pragma unroll
        for (int j = 0; j < 8; ++j) xs[t][j] = reinterpret_cast<const int*>(yb + 4)[j];
        dx[t] = half_bits_to_float(*reinterpret_cast<const unsigned short*>(yb));
    }
    between();
    int sum[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int w4 = *reinterpret_cast<const int*>(reinterpret_cast<const uint8_t*>(tab) + packed_addr(cur.idx, j));
#pragma unroll
        for (int t = 0; t < 2; ++t) sum[t] = __builtin_amdgcn_sdot4(w4, xs[t][j], sum[t], false);
    }
    const float dw = half_bits_to_float(cur.d);
    const int sc = 1 + 2 * (int) ((cur.sc >> (4 * (lane & 1))) & 0xFu);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const float z = butterfly_sum<SBR>((dw * dx[t]) * (float) __mul24(sum[t], sc));
        if (lane % SBR == SBR - 1 && u < nunits) out[(size_t) (t ? o1 : o0) * out_stride + u * (64 / SBR) + lane / SBR] = z;
    }
}

// A block has one group of 16 rows of one job. For launches of about a group a CU (a matrix of up to 4,096 rows alone): such a launch is
// its chain of trips to memory, and the kernel below, whose blocks stream, decodes and loads ahead for groups that are not
// there. And for a few jobs over short matrices, whose groups a CU do not come out even: the streaming kernel's runs then cross
// from one job to the next, each job with its activations to fetch, where two of these blocks run on a CU side by side.
// Over weights nobody has read lately, us (streaming / this), jobs of 1 row, 2, 5, 16: 4,096 rows, one job 4.4 / 3.8, 7.7 / 5.9, 8.0 / 6.4,
// 9.5 / 7.7; 1,024 rows, five jobs 8.1 / 4.5, 11.8 / 7.5, 12.6 / 8.2, 15.6 / 11.5; ten 8.6 / 6.1, 12.3 / 10.2, 13.1 / 11.2, 16.4 / 15.7. Not for the
// others: every block fetches its job's activations, 8,192 rows, sixteen rows of one job 9.7 / 11.7; 1,024 rows, twenty jobs 19.4 / 24.1.
// SBR < 64: a mat-vec call of up to eight jobs over shorter rows, 16 64 / SBR of them a block. The vector-ALU kernel that took them loads and
// decodes a weight once for every two rows of a job, or four. Us a call with its quantisation, before / now, jobs of 1 row, 5, 16: 8,192
// rows of 512 columns 7.5 / 7.4, 10.5 / 7.4, 15.6 / 8.3, of 1,024 columns 7.8 / 7.4, 11.1 / 7.7, 16.8 / 9.1; two blocks on some CUs: 12,288
// rows of 1,024 columns 8.0 / 7.3, 11.4 / 9.8, 17.7 / 13.2. Past two blocks a CU the streaming kernel's runs stay.
template <int SBR>
__global__ void __launch_bounds__(JM_THREADS) k_iq3s_jobs_mma_one(const RowsArgs a) {
    __shared__ JmOneLds<SBR> L;
    const uint32_t code = g_sgrid.v[threadIdx.x & 511];   // a code's sixteen signed entries from its unsigned one, by two threads
    const int nj = a.njobs ? min(uniform(*a.njobs), a.njobs_max) : a.njobs_max;
    const int nunits = a.nrows / (64 / SBR);
    const uint32_t gpj = (uint32_t) (nunits + 15) / 16, ji = blockIdx.x / gpj;
    if ((int) ji >= nj) return;   // the same for the whole block
    const int g = (int) (blockIdx.x - ji * gpj);
    const fnx_job* jb = a.jobs + ji;
    const int n = uniform(min(jb->n, FNX_MAXT)), w = uniform(jb->w), y0 = uniform(jb->y[0]), out0 = uniform(jb->out[0]);
    if (n < 1) return;
    const uint8_t* y = a.y ? a.y : g_moe_hq;
    const uint8_t* we = a.ep ? uniform_ptr(a.ep[w]) : a.wbase + (size_t) w * a.w_stride;
    auto codebook = [&] {
        uint32_t code_v = code;
        asm volatile("" : "+v"(code_v));   // (the entries are worked out here: before, they would wait for the code ahead of the loads)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int sg = 2 * k + (int) (threadIdx.x >> 9);
            L.tab[sg * 512 + (threadIdx.x & 511)] = signed_entry(code_v, sg);
        }
        __syncthreads();
    };
    if (n == 1) jm_few<1, SBR>(L.tab, we, 16 * g, min(16 * (g + 1), nunits), y0, out0, y, a.out, a.out_stride, codebook);
    else if (SBR < 64 && n == 2) jm_two<SBR>(L.tab, we, 16 * g + uniform((int) (threadIdx.x >> 6)), nunits, jb, y, a.out, a.out_stride, codebook);
    else jm_group<SBR>(L, we, g, nunits, jb, n, y, a.out, a.out_stride, codebook);
}

// rows of 2048 columns, a multiple of 16 of them; unit64. The blocks split the (job, 16 rows) items of all jobs evenly and
// walk them in order, so a block streams a contiguous range of memory and changes job a few times at most. The first run's job
// is looked up and its first weights are asked for while the codebook's entries are on their way. Sixteen waves a CU ask for
// the codebook's 2 KiB in every block at once, so half of them do.
// 8,192 rows, one job, us (against a kernel that writes the codebook first): one row 6.8 -> 5.3, 2 rows 8.7 -> 7.9, 5 rows 8.6 -> 8.2,
// 16 rows 9.4 -> 9.7; 32,768 rows 10.8 -> 11.0, 17.5 -> 16.5, 17.4 -> 16.7, 18.7 -> 18.1.
__global__ void __launch_bounds__(JM_THREADS) k_iq3s_jobs_mma(const RowsArgs a) {
    __shared__ JmLds L;
    uint32_t code = 0;   // a code's sixteen signed entries from its unsigned one, by the lower half's threads
    if (threadIdx.x < 512) code = g_sgrid.v[threadIdx.x];
    const int nj = a.njobs ? min(uniform(*a.njobs), a.njobs_max) : a.njobs_max;
    const uint32_t gpj = (uint32_t) a.nrows / JM_ROWS;   // items per job
    const unsigned long long total = (unsigned long long) nj * gpj;
    uint32_t i = (uint32_t) (total * blockIdx.x / gridDim.x);
    const uint32_t i1 = (uint32_t) (total * (blockIdx.x + 1) / gridDim.x);
    if (i >= i1) return;   // the same for the whole block
    const uint8_t* y = a.y ? a.y : g_moe_hq;
    uint32_t ji = i / gpj;
    int g0 = (int) (i - ji * gpj), g1 = (int) min(gpj, g0 + (i1 - i));
    const fnx_job* jb = a.jobs + ji;
    int n = uniform(min(jb->n, FNX_MAXT)), w = uniform(jb->w);
    const int y0 = uniform(jb->y[0]), out0 = uniform(jb->out[0]);
    auto codebook = [&] {
        uint32_t code_v = code;
        asm volatile("" : "+v"(code_v));   // (the entries are worked out here: before, they would wait for the code ahead of the loads)
        if (threadIdx.x < 512) {
#pragma unroll
            for (int sg = 0; sg < 16; ++sg) L.tab[sg * 512 + threadIdx.x] = signed_entry(code_v, sg);
        }
        __syncthreads();
    };
    auto matrix = [&] { return a.ep ? uniform_ptr(a.ep[w]) : a.wbase + (size_t) w * a.w_stride; };
    const int few = n == 1 ? g1 - g0 : 0;
    bool done = few >= 1 && few <= 4;   // the first run is made
    if (__builtin_expect(done, 0)) {   // (out of the way of the others' code)
        if (few <= 2) jm_few<2>(L.tab, matrix(), JM_ROWS * g0, JM_ROWS * g1, y0, out0, y, a.out, a.out_stride, codebook);
        else jm_few<4>(L.tab, matrix(), JM_ROWS * g0, JM_ROWS * g1, y0, out0, y, a.out, a.out_stride, codebook);
    }
    bool table = done;   // the codebook is in LDS
    auto between = [&] {
        if (!table) codebook();   // (the same for the whole block)
        table = true;
    };
    while (true) {
        if (!done) {
            const uint8_t* we = matrix();
            if (n >= JM_MIN) jm_segment(L, we, g0, g1, jb, n, y, a.out, a.out_stride, between);
            else if (n >= 1) jm_narrow(L.tab, we, JM_ROWS * g0, JM_ROWS * g1, jb, y, a.out, a.out_stride, between);
        }
        done = false;
        i += (uint32_t) (g1 - g0);
        if (i >= i1) break;
        ji = i / gpj;
        g0 = (int) (i - ji * gpj), g1 = (int) min(gpj, g0 + (i1 - i));
        jb = a.jobs + ji;
        n = uniform(min(jb->n, FNX_MAXT)), w = uniform(jb->w);
    }
}

}  // namespace fnx
