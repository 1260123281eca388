// The routed experts' down projection on the matrix cores over matrices of up to 512 columns (tile16, unit64), a wave a tile of 16 rows.
//
// A block that takes one (job, 256 rows) task at a time, its activations staged per step, meets at two barriers a stage:
// with rows of 512 columns a task is a single stage, the eight waves of such a block meet four times per 32 rows each, and
// at two waves a SIMD little covers the codebook lookups' latency. Here the whole activation tile of a job - up to 64 tokens x 512
// columns of f16, 64 KiB - is put in LDS once (by loads that write LDS directly, a token's row per wave instruction), and
// after that a wave needs nothing from the others: it takes tiles of 16 rows, a lane decodes its four sub-blocks of its
// row from one contiguous load of the tile16 layout, and the sixteen waves of a block (four a SIMD) meet only where the
// block goes from one phase of jobs to the next. The blocks split the (job, sixteen tiles) units of all jobs by cost - a tile's
// decode and its job's token tiles of multiplications - into contiguous runs.
// part[job.out[t]][row] = W[job.w][row] . h16[job.y[t]] as kernels.hpp:330 (moe_down_mma) defines it, with the weights as
// f16 (d (1 + 2 s) g, the f32 value rounded once, as k_moe_mma rounds it) and a row's sub-blocks accumulated super-step by
// super-step (S, then the four steps, then a step's four operands).
#pragma once

#include "k_prefill.h"

namespace fnx {

constexpr int W16_THREADS = 1024, W16_WAVES = 16, W16_COLS = 512;
constexpr int W16_XROW = 2 * W16_COLS + 16;   // bytes of a token's f16 row in LDS (260 words: the 16 tokens of a 16-byte operand read fall on 64 different banks)
constexpr int W16_DEC = 3, W16_MUL = 1;   // an item's cost: W16_DEC for its decode and W16_MUL a token tile of its job (measured: 2.7 us a round of
                                          // sixteen tiles with one token tile, 4.7 us with four)
constexpr int W16_HELD = 2048;  // jobs of a list whose token counts and matrices are read into LDS at once, ahead of the split
struct Wave16Lds {
    uint2 tab[SGRID_WORDS];
    __attribute__((aligned(16))) uint8_t xt[MB_TOK64 * W16_XROW];
    int first_job, first_tile, last_job, last_tile;   // the block's run: from (first_job, first_tile) up to but not including (last_job, last_tile)
    uint8_t jn[2][W16_HELD];                          // the token counts of the two lists' jobs, as far as they fit
    int jw[W16_HELD];                                 // the first list's matrices
};

// f16(a0 b0) | f16(a1 b1) << 16, each product rounded once and a product that vanishes a positive zero: what the compiler makes
// of k_swiglu_h16's expression. Left to itself it takes a multiplication and a conversion in one place and this in the next,
// and a row's h would depend on the size of the job it falls in.
__device__ __forceinline__ uint32_t h16_pair(float a0, float b0, float a1, float b1) {
    uint32_t v;
    // (a half register's write is not forwarded: a wait state before the next instruction that uses the register)
    asm("v_fma_mixlo_f16 %0, %1, %2, 0\n\ts_nop 0\n\tv_fma_mixhi_f16 %0, %3, %4, 0\n\ts_nop 0" : "=&v"(v) : "v"(a0), "v"(b0), "v"(a1), "v"(b1));
    return v;
}
// A lane's half of a sub-block (fields s) as two f16 operands: weights 16 h .. 16 h + 15
__device__ __forceinline__ void w16_half(const uint2* tab, const SubFields& s, int h, v8h (&A)[2]) {
    const _Float16 c = (_Float16) (int) (1 + 2 * s.sc), d = __builtin_bit_cast(_Float16, (unsigned short) s.d);
    const v2h s2 = {c, c}, d2 = {d, d};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint2 en = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(tab) + sub_entry<true>(s, 4 * h + k));
        const v2h lo = (as_v2h(en.x) * s2) * d2, hi = (as_v2h(en.y) * s2) * d2;
        A[k >> 1][4 * (k & 1) + 0] = lo.x;
        A[k >> 1][4 * (k & 1) + 1] = lo.y;
        A[k >> 1][4 * (k & 1) + 2] = hi.x;
        A[k >> 1][4 * (k & 1) + 3] = hi.y;
    }
}
// A tile's super-step: the lane's four sub-blocks of its row (fields f) as f16 operands, against the nt token tiles of
// the activation tile in LDS (xlane: token r's row at this lane group's sub-blocks), added to acc
template <int PS = 4>
__device__ __forceinline__ void w16_super_step(const uint2* tab, const uint8_t* xlane, const SuperFields& f, int nt, v4f (&acc)[MB_TP]) {
    // the token tiles two at a time against the sub-block's operands
    auto pair = [&](const v8h (&A)[4], int p, auto t0_tag, auto cnt_tag) {
        constexpr int T0 = decltype(t0_tag)::value, CNT = decltype(cnt_tag)::value;
#pragma unroll
        for (int h = 0; h < 2; ++h) {   // two of the four operands at a time: the registers of a block of 1024 threads
            v4u B[2][2];
#pragma unroll
            for (int tt = 0; tt < CNT; ++tt)
#pragma unroll
                for (int i = 0; i < 2; ++i) B[tt][i] = *reinterpret_cast<const v4u*>(xlane + (T0 + tt) * 16 * W16_XROW + 64 * p + 32 * h + 16 * i);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int tt = 0; tt < CNT; ++tt)
                    acc[T0 + tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[2 * h + i], __builtin_bit_cast(v8h, B[tt][i]), acc[T0 + tt], 0, 0, 0);
        }
    };
    auto step = [&](auto p_c) {
        constexpr int p = decltype(p_c)::value;
        const SubFields s = super_sub<p>(f);
        const _Float16 sc = (_Float16) (int) (1 + 2 * s.sc), d = __builtin_bit_cast(_Float16, (unsigned short) s.d);
        const v2h s2 = {sc, sc}, d2 = {d, d};
        v8h A[4];   // the lane's sub-block (row r, 4 grp + p) as 32 f16 weights
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint2 en = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(tab) + sub_entry<true>(s, k));
            const v2h lo = (as_v2h(en.x) * s2) * d2, hi = (as_v2h(en.y) * s2) * d2;
            A[k >> 1][4 * (k & 1) + 0] = lo.x;
            A[k >> 1][4 * (k & 1) + 1] = lo.y;
            A[k >> 1][4 * (k & 1) + 2] = hi.x;
            A[k >> 1][4 * (k & 1) + 3] = hi.y;
        }
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        if (nt >= 2) pair(A, p, I0{}, I2{});
        else pair(A, p, I0{}, I1{});
        if (nt == 3) pair(A, p, I2{}, I1{});
        else if (nt == 4) pair(A, p, I2{}, I2{});
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    if constexpr (PS == 4) {
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
    }
}

// Two tiles' super-steps against the same NT token tiles (fields f0 and f1, sums acc0 and acc1): an operand of the activation
// tile read from LDS once for both. Half a sub-block of either tile is decoded at a time, so that the decoded operands take
// the registers that one tile's whole sub-block takes above. between: run between the second and the third of the four
// steps, where the first half of the fields is dead (loads of what comes next find registers there). Every sum is
// accumulated as w16_super_step does it.
template <int NT, class Between>
__device__ __forceinline__ void w16_super_pair(const uint2* tab, const uint8_t* xlane, const SuperFields& f0, const SuperFields& f1, v4f (&acc0)[NT],
                                               v4f (&acc1)[NT], Between between) {
    auto step = [&](auto p_c) {
        constexpr int p = decltype(p_c)::value;
        const SubFields sa = super_sub<p>(f0), sb = super_sub<p>(f1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v8h A0[2], A1[2];
            w16_half(tab, sa, h, A0);
            w16_half(tab, sb, h, A1);
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) {
                v4u B[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) B[i] = *reinterpret_cast<const v4u*>(xlane + tt * 16 * W16_XROW + 64 * p + 32 * h + 16 * i);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    acc0[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A0[i], __builtin_bit_cast(v8h, B[i]), acc0[tt], 0, 0, 0);
                    acc1[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A1[i], __builtin_bit_cast(v8h, B[i]), acc1[tt], 0, 0, 0);
                }
            }
        }
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    __builtin_amdgcn_sched_barrier(0);
    between();
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
}

// Where a lane finds its sub-blocks of a tile of 16 rows: PS of them a super-step of 128 PS columns, PS (lane / 16) .. of its row.
struct W16Tile16 {
    static constexpr int PS = 4;
    int nsuper;
    __device__ __forceinline__ W16Tile16(int ncols) : nsuper(ncols >> 9) {}
    __device__ __forceinline__ int tile_size() const { return nsuper * TILE16_BYTES; }
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t tiles(const uint8_t* we, int t) const { return tile16_rsrc(we, t, nsuper); }
    __device__ __forceinline__ SuperFields load(__amdgpu_buffer_rsrc_t m, int S) const { return tile16_load_buf(m, S); }
};
// unit64: rows of 256 columns (half a super-step: two sub-blocks a lane), 512, 1,024 or whole 2,048s. A lane's loads are runs of 32 (16), 16 (8),
// 4 (2), 2 (1) and 2 bytes of its row's planes, a tile's rows in whole units side by side: some more cache lines an instruction than tile16's
// contiguous planes, at the same speed (512 columns, 64 tokens of 128 jobs 29.0 us against 28.1, 8 tokens of 256 jobs 29.0 against 28.2).
template <int STEPS>
struct W16Unit64 {
    static constexpr int PS = STEPS;
    int nsuper, tile_bytes, a, b, c, sc, d;
    __device__ __forceinline__ W16Unit64(int ncols) : nsuper(ncols / (128 * STEPS)), tile_bytes((ncols >> 5) * (UNIT_BYTES / 4)) {
        const int lane = threadIdx.x & 63, at = (lane & 15) * (ncols >> 5) + STEPS * (lane >> 4), u = (at >> 6) * UNIT_BYTES, l = at & 63;
        a = u + 8 * l, b = u + UNIT_B_AT + 4 * l, c = u + UNIT_C_AT + l, sc = u + UNIT_SCALES_AT + (l >> 1), d = u + UNIT_D_AT + 2 * (l >> 3);
    }
    __device__ __forceinline__ int tile_size() const { return tile_bytes; }
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t tiles(const uint8_t* we, int t) const {
        return __builtin_amdgcn_make_buffer_rsrc((void*) uniform_ptr(we + (size_t) t * tile_bytes), 0, -1, 0x00020000);
    }
    __device__ __forceinline__ SuperFields load(__amdgpu_buffer_rsrc_t m, int S) const {
        SuperFields r;
        if constexpr (STEPS == 4) {
            const int u = (S >> 2) * UNIT_BYTES, s = S & 3;   // 16 sub-blocks further in the unit's planes; a unit after four
            r.a0 = __builtin_amdgcn_raw_buffer_load_b128(m, a, u + 128 * s, 0);
            r.a1 = __builtin_amdgcn_raw_buffer_load_b128(m, a + 16, u + 128 * s, 0);
            r.b = __builtin_amdgcn_raw_buffer_load_b128(m, b, u + 64 * s, 0);
            r.c = __builtin_amdgcn_raw_buffer_load_b32(m, c, u + 16 * s, 0);
            r.sc = __builtin_amdgcn_raw_buffer_load_b16(m, sc, u + 8 * s, 0);
            r.d = __builtin_amdgcn_raw_buffer_load_b16(m, d, u + 4 * s, 0);
        } else {   // (one super-step a row)
            const v2u h = __builtin_amdgcn_raw_buffer_load_b64(m, b, 0, 0);
            r.a0 = __builtin_amdgcn_raw_buffer_load_b128(m, a, 0, 0);
            r.a1 = r.b = v4u{0, 0, 0, 0};
            r.b.x = h.x, r.b.y = h.y;
            r.c = __builtin_amdgcn_raw_buffer_load_b16(m, c, 0, 0);
            r.sc = __builtin_amdgcn_raw_buffer_load_b8(m, sc, 0, 0);
            r.d = __builtin_amdgcn_raw_buffer_load_b16(m, d, 0, 0);
        }
        return r;
    }
};

// (rows of one super-step)
template <class LY>
__global__ void __launch_bounds__(W16_THREADS) k_moe_mma_wave16(const MmaArgs a) {
    constexpr int PS = LY::PS;
    // the block's place in the plan: blocks with neighbouring places run on one XCD (workgroups go to the eight XCDs in turn), so
    // the units of one expert, which the plan deals to neighbouring places, find the expert's weights in that XCD's L2
    const unsigned vb = gridDim.x % 8 == 0 ? (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
    __shared__ Wave16Lds L;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), r = lane & 15, grp = lane >> 4;
    // every job's token count and matrix, a thread a job, both lists at once (entries past a list's count are read too - the
    // arrays hold cap jobs - and not used): one round of loads instead of dependent ones wherever a job's turn comes
    // (asked for ahead of the codebook's entries, made meanwhile)
    int hn[2] = {0, 0}, hn2 = 0, hw[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int j = tid + i * W16_THREADS;
        if (j < min(a.cap, W16_HELD)) hn[i] = a.jobs[j].n, hw[i] = a.jobs[j].w;
    }
    if (a.jobs2 && tid < min(a.cap2, W16_HELD)) hn2 = a.jobs2[tid].n;
    const int nj_raw = *a.njobs, nj2_raw = a.jobs2 ? *a.njobs2 : 0;
    {
        const uint32_t tab0 = g_sgrid.v[tid & 511];   // a thread's code: its sixteen signed entries are made here
#pragma unroll
        for (int i = tid; i < SGRID_WORDS; i += W16_THREADS) {
            const uint32_t g = signed_entry(tab0, i >> 9);
            v2h lo, hi;
            lo.x = (_Float16) (int) (int8_t) (g & 0xFFu);
            lo.y = (_Float16) (int) (int8_t) ((g >> 8) & 0xFFu);
            hi.x = (_Float16) (int) (int8_t) ((g >> 16) & 0xFFu);
            hi.y = (_Float16) (int) (int8_t) (g >> 24);
            L.tab[i] = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int j = tid + i * W16_THREADS;
        if (j < min(a.cap, W16_HELD)) L.jn[0][j] = (uint8_t) max(0, min(FNX_PF_JOB, hn[i])), L.jw[j] = hw[i];
    }
    if (a.jobs2) {
        if (tid < min(a.cap2, W16_HELD)) L.jn[1][tid] = (uint8_t) max(0, min(FNX_PF_JOB, hn2));
        for (int j = tid + W16_THREADS; j < min(a.cap2, W16_HELD); j += W16_THREADS) L.jn[1][j] = (uint8_t) max(0, min(FNX_PF_JOB, a.jobs2[j].n));
    }
    const int nj = min(a.cap, uniform(nj_raw)), nj2 = a.jobs2 ? min(a.cap2, uniform(nj2_raw)) : 0, njall = nj + nj2;
    const int gpj = a.nrows >> 4;   // items a job
    // a unit: a tile for every wave of the block - or, where that would leave blocks without work, a single tile
    const int ut = (long) njall * ((gpj + W16_WAVES - 1) / W16_WAVES) >= 2l * gridDim.x ? W16_WAVES : 1, upj = (gpj + ut - 1) / ut;
    auto job_at = [&](int j) { return j < nj ? a.jobs + j : a.jobs2 + (j - nj); };
    auto n_of = [&](int j) {   // job j's tokens, 0 .. FNX_PF_JOB
        const int l = j < nj ? 0 : 1, k = j < nj ? j : j - nj;
        return k < W16_HELD ? (int) L.jn[l][k] : max(0, min(FNX_PF_JOB, job_at(j)->n));
    };
    __syncthreads();
    // The block's run of items, in units (a run that ended inside a round of the block's waves would leave most of them
    // waiting for the few). A unit of job j costs w_j = W16_DEC + W16_MUL * (token tiles of j), a job upj * w_j;
    // unit (j, u) begins at (the cost of the jobs before j) + u * w_j, and block b takes the units that begin in
    // [total * b / blocks, total * (b + 1) / blocks). One wave finds the run: a lane adds up a stretch of jobs, the
    // stretches' sums are added up over the lanes, and the lanes whose stretch holds an end of the run walk it.
    if (wave == 0) {
        auto weight_of = [&](int j) {
            const int n = n_of(j);
            return n >= 1 ? (uint32_t) (W16_DEC + W16_MUL * ((n + 15) >> 4)) : 0u;
        };
        const int per = (njall + 63) >> 6, j0 = min(njall, lane * per), j1 = min(njall, j0 + per);
        unsigned long long sum = 0;
        for (int j = j0; j < j1; ++j) sum += (unsigned long long) weight_of(j) * (uint32_t) upj;
        unsigned long long incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned long long up = __shfl_up(incl, o);
            if (lane >= o) incl += up;
        }
        const unsigned long long total = __shfl(incl, 63);
        unsigned long long c0, c1;   // (64-bit quotients take a few hundred instructions)
        if (total <= 0xFFFFFFFFull / gridDim.x) c0 = (uint32_t) total * vb / gridDim.x, c1 = (uint32_t) total * (vb + 1) / gridDim.x;
        else c0 = total * vb / gridDim.x, c1 = total * (vb + 1) / gridDim.x;
        if (lane == 0) {   // ends that lie past every job's items
            L.first_job = L.last_job = njall;
            L.first_tile = L.last_tile = 0;
        }
        // the first unit that begins at or after a point inside a job (past its last unit: the next job's first, as a tile past gpj)
        auto find = [&](unsigned long long c, int& job, int& tile) {
            unsigned long long at = incl - sum;   // where this lane's stretch begins
            if (!(at <= c && c < at + sum)) return;
            for (int j = j0; j < j1; ++j) {
                const uint32_t w = weight_of(j);
                const unsigned long long cj = (unsigned long long) w * (uint32_t) upj;
                if (c < at + cj) {
                    job = j;
                    tile = ut * (int) ((uint32_t) (c - at + w - 1) / w);
                    return;
                }
                at += cj;
            }
        };
        find(c0, L.first_job, L.first_tile);
        find(c1, L.last_job, L.last_tile);
    }
    __syncthreads();   // the codebook and the run
    const int jA = uniform(L.first_job), tA = uniform(L.first_tile), jB = uniform(L.last_job), tB = uniform(L.last_tile);
    const uint32_t xt_at = (uint32_t) (size_t) (__attribute__((address_space(3))) uint8_t*) L.xt;
    const LY ly(a.ncols);
    const uint8_t* xlane = L.xt + r * W16_XROW + 64 * PS * grp;   // token r of a tile, this lane group's four sub-blocks of a super-step
    // The run goes in phases: the jobs of it, one after another, whose token tiles find room together in the four that LDS has. A
    // phase's activations come in at once and the waves meet only where it ends; the next one's rows are looked up while they are on
    // their way, and the first weights of a wave's next job, in this phase or the next, asked for behind its last tile of this one. With
    // a job at a time the memory stood still wherever a block went from one to the next (us a launch of 2,048 rows: 512 jobs of two
    // tokens 51.0 -> 47.5, 768 of four 75.5 -> 70.5, 256 of eight 28.1 -> 27.3, 512 of 64 152.3 -> 148.6; a chunk of 29 rows, 8 of 512
    // experts, 93.5 -> 90.5, of 77, 10 picks, 159.5 -> 156.1). The weights are asked for ahead of the rows, which wait for them: behind the rows
    // 0.4 us a launch more; the phase's rows looked up in one place of the code, not two: 0.4 us of cold code.
    auto first_of = [&](int j) { return j == jA ? tA : 0; };   // job j's items of the run
    auto last_of = [&](int j) { return j == jB ? min(tB, gpj) : gpj; };
    struct Job {
        int j, n;
    };
    auto next_job = [&](int j) {   // the first job from j on that has items in the run, and its tokens; past the run: the end
        for (const int end = min(jB, njall - 1); j <= end; ++j) {
            const int n = uniform(n_of(j));
            if (n >= 1 && first_of(j) < last_of(j)) return Job{j, n};
        }
        return Job{njall, 0};
    };
    auto matrix_of = [&](int j) {
        const int e = j >= nj ? 0 : uniform(j < W16_HELD ? L.jw[j] : job_at(j)->w);
        return j >= nj ? a.w2 : a.ep ? uniform_ptr((const uint8_t*) a.ep[e]) : a.w + (size_t) e * a.stride;
    };
    // the phase that begins with a job: where the next one begins; this wave's tokens (tokens wave, wave + 16, .. of every job, past its
    // last that one again) and this lane's place in the output, a token tile each
    auto phase_at = [&](Job c, int (&y)[MB_TP], int (&orow)[MB_TP]) {
        int used = 0, rows[MB_TP];
#pragma unroll
        for (int p = 0; p < MB_TP; ++p) rows[p] = orow[p] = -1;
        while (c.j < njall) {
            const int nt = (c.n + 15) >> 4;
            if (used + nt > MB_TP) break;
            const fnx_bigjob* jb = job_at(c.j);
#pragma unroll
            for (int p = 0; p < MB_TP; ++p)
                if (p >= used && p < used + nt) {
                    const int t0 = 16 * (p - used);
                    rows[p] = jb->y[min(wave + t0, c.n - 1)];
                    if (t0 + r < c.n) orow[p] = jb->out[t0 + r];
                }
            used += nt;
            c = next_job(c.j + 1);
        }
#pragma unroll
        for (int p = 0; p < MB_TP; ++p) y[p] = uniform(rows[p]);   // (waited for together)
        return c;
    };
    Job cur = next_job(jA);
    if (cur.j >= njall) return;   // (the same for the whole block)
    int g = first_of(cur.j) + wave;
    const uint8_t* we = matrix_of(cur.j);
    SuperFields f = ly.load(ly.tiles(we, min(g, last_of(cur.j) - 1)), 0);
    int yn[MB_TP], on[MB_TP];
    uint32_t at[MB_TP] = {0, 0, 0, 0};   // this lane's tokens' places in the output
    bool all_near = true;
    // A tile's results go out as buffer stores that every path issues (a lane without a token: past the buffer's end, where
    // a store is dropped): stores under a condition of their own cannot be counted, and the wait for the next tile's weights,
    // asked for before them, was a wait for the stores too (77 rows, some 400 jobs of two tokens: 59.1 -> 56.7 us a launch, 512 rows
    // 36.0 -> 35.2, 4,096 rows the same 186). The loop stands once for each number of token tiles, so that their stores are counted too.
    // A phase with a row past what 32-bit offsets reach stores under the condition, in one loop for all numbers: with four of
    // them the kernel was 32.7 KB of code instead of 24.9, at the same speed (8 picks of 512 experts, 29 rows 29.7 / 29.1 us a launch).
    const uint32_t rowb = (uint32_t) a.nrows * 4u, end = 0xE0000000u, none = 0xF0000000u;   // (none and a row's bytes: no wrap)
    const int reach = (int) (end / rowb);
    const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc((void*) a.out, 0, (int) end, 0x00020000);
    for (Job pend = cur;;) {   // the phase up to pend is on its way to LDS (at first none)
        const Job begin = pend;
        pend = phase_at(begin, yn, on);
        if (cur.j < begin.j) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
        for (const uint8_t* xl = xlane; cur.j < begin.j;) {
            const int nt = (cur.n + 15) >> 4, g1 = last_of(cur.j);
            // the next job's first tile of this wave (no job: a tile of its own again)
            const Job then = next_job(cur.j + 1);
            const bool any = then.j < njall;
            const int gn = any ? first_of(then.j) + wave : 0, gl = any ? min(gn, last_of(then.j) - 1) : 0;
            const uint8_t* wn = any ? matrix_of(then.j) : we;
            if (g >= g1) f = ly.load(ly.tiles(wn, gl), 0);   // (no tile for this wave)
            int left = (g1 - g + W16_WAVES - 1) / W16_WAVES;   // this wave's tiles
            const uint8_t *tile = we + (size_t) g * ly.tile_size(), *then_tile = any ? wn + (size_t) gl * ly.tile_size() : tile;
            auto rounds = [&](auto ntiles, auto near_tag) {   // (ntiles: a constant, or nt)
                for (; left > 0; --left, g += W16_WAVES) {
                    // The oldest wave of a SIMD goes first, so a block's waves drift apart and the first ones wait at the phase's end
                    // for the last: every wave takes every priority in turn, a tile each
                    switch (((wave >> 2) + left) & 3) {
                        case 0: __builtin_amdgcn_s_setprio(0); break;
                        case 1: __builtin_amdgcn_s_setprio(1); break;
                        case 2: __builtin_amdgcn_s_setprio(2); break;
                        default: __builtin_amdgcn_s_setprio(3); break;
                    }
                    tile = left > 1 ? tile + (size_t) W16_WAVES * ly.tile_size() : then_tile;
                    const SuperFields nf = ly.load(ly.tiles(tile, 0), 0);
                    __builtin_amdgcn_sched_barrier(0);   // (left to itself the compiler asks for them behind the products)
                    v4f acc[MB_TP];
#pragma unroll
                    for (int tt = 0; tt < MB_TP; ++tt) acc[tt] = v4f{0.f, 0.f, 0.f, 0.f};
                    w16_super_step<PS>(L.tab, xl, f, ntiles, acc);
                    // lane: token r of each tile, rows 4 grp .. 4 grp + 3 of the tile
#pragma unroll
                    for (int tt = 0; tt < MB_TP; ++tt) {
                        if constexpr (decltype(near_tag)::value) {
                            if (tt < ntiles) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, acc[tt]), to, at[tt], 64u * g, 0);
                        } else if (16 * tt + r < cur.n && job_at(cur.j)->out[16 * tt + r] >= 0)
                            *reinterpret_cast<float4*>(a.out + (size_t) job_at(cur.j)->out[16 * tt + r] * a.nrows + 16 * g + 4 * grp) = make_float4(acc[tt].x, acc[tt].y, acc[tt].z, acc[tt].w);
                    }
                    f = nf;
                }
            };
            if (!all_near) rounds(nt, std::false_type{});
            else if (nt == 4) rounds(std::integral_constant<int, 4>{}, std::true_type{});
            else if (nt == 3) rounds(std::integral_constant<int, 3>{}, std::true_type{});
            else if (nt == 2) rounds(std::integral_constant<int, 2>{}, std::true_type{});
            else rounds(std::integral_constant<int, 1>{}, std::true_type{});
            // the next job's token tiles to the front
            for (int i = 0; i < nt && then.j < begin.j; ++i) {
#pragma unroll
                for (int tt = 0; tt + 1 < MB_TP; ++tt) at[tt] = at[tt + 1];
            }
            xl += 16 * nt * W16_XROW;
            cur = then, g = gn, we = wn;
        }
        if (begin.j >= njall) break;
        __syncthreads();   // the phase before has been read
#pragma unroll
        for (int p = 0; p < MB_TP; ++p)   // a token's row a wave instruction, 16 bytes a lane
            if (yn[p] >= 0) lds_load16(a.x + (size_t) yn[p] * a.ldx, 16u * (lane & (16 * PS - 1)), xt_at + (wave + 16 * p) * W16_XROW);
        bool near = true;
#pragma unroll
        for (int p = 0; p < MB_TP; ++p) near = near && on[p] < reach, at[p] = on[p] >= 0 ? (uint32_t) on[p] * rowb + 16u * grp : none;
        all_near = __all(near);
    }
}

// ---------------------------------------------------------------- the same form for longer rows (512 S columns): stacked gate|up matrices, and plain ones
// A job's activations are S tiles of 64 tokens x 512 columns here, and LDS holds one: a block takes units of (job, sixteen
// gate tiles and the sixteen up tiles that go with them), a wave one such pair, and walks the S super-steps with the
// pair's accumulators in registers - activation tile S in (two barriers), the gate tile's and the up tile's super-steps
// together, so that an activation operand is read from LDS once for both (4,096 rows of a Zipf chunk: 307 -> 269 us, LDS and
// VALU each busy a little over half the time; reading it for each tile was a third of the LDS's work) - and leaves
// h = silu(gate) * up as f16 (k_swiglu_h16's values). Such a unit is too coarse for runs by cost, and two of even the
// lightest on one block made the launch half as long again as its mean block. So the jobs are ranked by token tiles and the
// units of those with two token tiles and more dealt heaviest first, to and fro over the blocks. The pairs of the jobs of up
// to 16 tokens then fill the blocks up to the mean load: a block stages all the tokens of its stretch's jobs at once, S tiles
// of sixteen places, and its waves take the pairs one by one as they come free (77 rows, some 400 jobs of two tokens: 87 us;
// 114 as units of eight pairs, a wave a tile, with a job's tokens fetched and the block met twice in each of them: of such a
// unit's 16 us the LDS needs 9). A stage with pairs for half of the waves or fewer goes a wave a tile, the up tiles' sums handed to
// the gate tiles' waves (a lone job of 5 tokens 16.0 -> 15.5 us, 125 jobs of 9, some of whose stretches are two stages, 36.3 -> 33.7).
// The weights of the next super-step are asked for in the middle of the one before. Every tile is accumulated in one order (S,
// then the four steps, then a step's four operands) whatever a job's size or the unit it falls in: a row's h does not
// depend on what else is in the chunk.
// Costs, in 1/16 us at S = 4 (measured): a heavy unit of so many token tiles; a light pair, of which a block works on sixteen at a time.
__device__ __forceinline__ int w16_heavy_cost(int nt) { return 320 + 88 * nt; }
constexpr int W16_PAIR_COST = 18;
__device__ __forceinline__ int w16_mean(int heavy, int np, int G) { return (int) (((long) heavy + (long) np * W16_PAIR_COST + G - 1) / G); }
__device__ __forceinline__ double w16_inverse(int all) {   // of a positive count, to the last bits: a step on the unit's estimate
    const double v = __builtin_amdgcn_rcp((double) all);
    return fma(v, fma((double) -all, v, 1.0), v);
}
// where the stretch of n pairs begins whose share starts at c of all (monotone in c, 0 at 0 and n at all)
__device__ __forceinline__ int w16_part(int n, int c, int all, double inv) { return c >= all ? n : min(n, (int) fma((double) n, (double) c * inv, 1e-4)); }
constexpr int W16_SORTJ = 2048, W16_GU_HELD = 2048, W16_PLAN = 4;   // (W16_PLAN: blocks a lane of the planning wave looks after)
struct Wave16GuLds {
    uint2 tab[SGRID_WORDS];
    __attribute__((aligned(16))) uint8_t xt[MB_TOK64 * W16_XROW];
    uint8_t jn[2][W16_GU_HELD];
    int jw[W16_GU_HELD];
    unsigned short jorder[W16_SORTJ];   // the jobs, most token tiles first (the lower index first among equals)
    int orow[FNX_PF_JOB];   // a heavy unit's tokens' places in the output
    float4 xs[W16_WAVES / 2][64];   // up tiles' sums on their way to the gate tiles' waves
    int p_total[MB_TP + 1], p_alone, p_first, p_last;   // the jobs by token tiles, those of 9 .. 16 tokens; the plan where one wave made it: this block's stretch of the light pairs
    int ph_jobs, ph_tokens, ph_next;                      // a phase of light pairs: its jobs, their tokens, the next pair to take
    unsigned short ph_job[16];
    unsigned char ph_first[16];                           // a job's first place in LDS
};
// GU: stacked gate|up matrices, a pair = 16 gate rows and the 16 up rows that go with them, h = silu(gate) * up out as f16; else any matrix, a pair = two
// tiles side by side, the products out as f32 rows.
template <bool GU, class LY>
__global__ void __launch_bounds__(W16_THREADS) k_moe_mma_wave16_pairs(const MmaArgs a) {
    constexpr int PS = LY::PS;
    static_assert(PS == 4, "whole super-steps");
    // the block's place in the plan: blocks with neighbouring places run on one XCD (workgroups go to the eight XCDs in turn), so
    // the units of one expert, which the plan deals to neighbouring places, find the expert's weights in that XCD's L2
    const unsigned vb = gridDim.x % 8 == 0 ? (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
    __shared__ Wave16GuLds L;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), r = lane & 15, grp = lane >> 4;
    const int nj_raw = *a.njobs, nj2_raw = a.jobs2 ? *a.njobs2 : 0;
    const uint32_t tab0 = g_sgrid.v[tid & 511];
    const int nj = min(a.cap, uniform(nj_raw)), nj2 = a.jobs2 ? min(a.cap2, uniform(nj2_raw)) : 0, njall = nj + nj2;
    // the token counts and matrices of the jobs that count, on their way while the codebook is written
    const int held = min(nj, W16_GU_HELD), held2 = min(nj2, W16_GU_HELD);
    int hn[2] = {0, 0}, hn2 = 0, hw[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int j = tid + i * W16_THREADS;
        if (j < held) hn[i] = a.jobs[j].n, hw[i] = a.jobs[j].w;
    }
    if (tid < held2) hn2 = a.jobs2[tid].n;
    {
#pragma unroll
        for (int i = tid; i < SGRID_WORDS; i += W16_THREADS) {
            const uint32_t g = signed_entry(tab0, i >> 9);
            v2h lo, hi;
            lo.x = (_Float16) (int) (int8_t) (g & 0xFFu);
            lo.y = (_Float16) (int) (int8_t) ((g >> 8) & 0xFFu);
            hi.x = (_Float16) (int) (int8_t) ((g >> 16) & 0xFFu);
            hi.y = (_Float16) (int) (int8_t) (g >> 24);
            L.tab[i] = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int j = tid + i * W16_THREADS;
        if (j < held) L.jn[0][j] = (uint8_t) max(0, min(FNX_PF_JOB, hn[i])), L.jw[j] = hw[i];
    }
    if (tid < held2) L.jn[1][tid] = (uint8_t) max(0, min(FNX_PF_JOB, hn2));
    for (int j = tid + W16_THREADS; j < held2; j += W16_THREADS) L.jn[1][j] = (uint8_t) max(0, min(FNX_PF_JOB, a.jobs2[j].n));
    const LY ly(a.ncols);
    const int nsuper = ly.nsuper, ppj = a.nrows >> 5;                                   // pairs of tiles a job
    const int upj = (ppj + W16_WAVES - 1) / W16_WAVES;                                  // heavy units a job
    auto job_at = [&](int j) { return j < nj ? a.jobs + j : a.jobs2 + (j - nj); };
    auto n_of = [&](int j) {
        const int l = j < nj ? 0 : 1, k = j < nj ? j : j - nj;
        return k < W16_GU_HELD ? (int) L.jn[l][k] : max(0, min(FNX_PF_JOB, job_at(j)->n));
    };
    __syncthreads();
    const bool sorted = njall <= W16_SORTJ;
    if (sorted && wave == 0) {   // a counting sort by one wave, 64 jobs a trip: class totals, then every job's place
        int total[MB_TP + 1], alone = 0;   // alone: light jobs of more than half of a phase's places
#pragma unroll
        for (int c = 0; c <= MB_TP; ++c) total[c] = 0;
        for (int j0 = 0; j0 < njall; j0 += 64) {
            const int n = j0 + lane < njall ? n_of(j0 + lane) : -16, kj = (n + 15) >> 4;
            alone += __popcll(__ballot(n > 8 && n <= 16));
#pragma unroll
            for (int c = 0; c <= MB_TP; ++c) total[c] += __popcll(__ballot(kj == c));
        }
        int base[MB_TP + 1];   // where a class starts: the classes in descending order
        base[MB_TP] = 0;
#pragma unroll
        for (int c = MB_TP - 1; c >= 0; --c) base[c] = base[c + 1] + total[c + 1];
        for (int j0 = 0; j0 < njall; j0 += 64) {
            const int kj = j0 + lane < njall ? (n_of(j0 + lane) + 15) >> 4 : -1;
#pragma unroll
            for (int c = 0; c <= MB_TP; ++c) {
                const unsigned long long m = __ballot(kj == c);
                if (kj == c) L.jorder[base[c] + __popcll(m & ((1ull << lane) - 1ull))] = (unsigned short) (j0 + lane);
                base[c] += __popcll(m);
            }
        }
        // The plan. Jobs of two token tiles and more go as units of sixteen pairs (a wave a pair), dealt heaviest first, to
        // and fro over the blocks. The pairs of the jobs of up to 16 tokens (where a row's S <= 4 activation tiles of 16 tokens
        // fit LDS together) fill the blocks up to the mean load: in the order of the blocks from the last one down (the lightest
        // first) each takes the stretch of the list of those pairs that its share, the mean less its heavy units, is of all shares.
        const int G = gridDim.x, ome = G - 1 - (int) vb;
        const bool split = nsuper <= 4;
        const int nbj = total[4] + total[3] + total[2] + (split ? 0 : total[1]), nb = nbj * upj, np = split ? total[1] * ppj : 0;
        if (lane == 0) {
#pragma unroll
            for (int c = 0; c <= MB_TP; ++c) L.p_total[c] = total[c];
            L.p_alone = alone;
        }
        if (nb > G) {   // (heavy units on one block or none: the same plan in closed form, below, by every wave)
            auto load_of = [&](int bb) {   // block bb's heavy units
                int l = 0;
                for (int k = 0; k * G < nb; ++k) {
                    const int u = k * G + ((k & 1) ? G - 1 - bb : bb);
                    if (u < nb) {
                        const int jo = u / upj;
                        l += w16_heavy_cost(jo < total[4] ? 4 : jo < total[4] + total[3] ? 3 : jo < total[4] + total[3] + total[2] ? 2 : 1);
                    }
                }
                return l;
            };
            // a lane looks after W16_PLAN blocks (a grid of up to 64 W16_PLAN), in the order from the last block down
            const int o0 = lane * W16_PLAN;
            int ld[W16_PLAN], mine_sum = 0;
#pragma unroll
            for (int i = 0; i < W16_PLAN; ++i) {
                ld[i] = o0 + i < G ? load_of(G - 1 - (o0 + i)) : 0;
                mine_sum += ld[i];
            }
#pragma unroll
            for (int sh = 32; sh >= 1; sh >>= 1) mine_sum += __shfl_xor(mine_sum, sh);
            const int mean = w16_mean(mine_sum, np, G);
            int kl = 0;
#pragma unroll
            for (int i = 0; i < W16_PLAN; ++i) {
                ld[i] = o0 + i < G ? max(0, mean - ld[i]) : 0;   // from here on: the block's share
                kl += ld[i];
            }
            int incl = kl;
#pragma unroll
            for (int sh = 1; sh < 64; sh <<= 1) {
                const int up = __shfl_up(incl, sh);
                if (lane >= sh) incl += up;
            }
            const int all = __shfl(incl, 63);
            if (o0 <= ome && ome < o0 + W16_PLAN) {
                int c = incl - kl, mine = 0;
#pragma unroll
                for (int i = 0; i < W16_PLAN; ++i) {
                    if (o0 + i < ome) c += ld[i];
                    if (o0 + i == ome) mine = ld[i];
                }
                const double inv = w16_inverse(all);
                L.p_first = w16_part(np, c, all, inv), L.p_last = w16_part(np, c + mine, all, inv);
            }
        }
    }
    __syncthreads();   // the codebook, the order and the plan
    const uint32_t xt_at = (uint32_t) (size_t) (__attribute__((address_space(3))) uint8_t*) L.xt;
    const uint8_t* xlane = L.xt + r * W16_XROW + 64 * PS * grp;
    const uint32_t xl16 = 16u * (lane & (16 * PS - 1));   // a lane's 16 bytes of a row's super-step
    auto first_tile = [&](int pr) { return GU ? pr : 2 * pr; };   // a pair's two tiles
    auto second_tile = [&](int pr) { return GU ? ppj + pr : 2 * pr + 1; };
    auto put = [&](int orow, int pr, v4f gt, v4f up) {   // lane: a token's rows 4 grp .. 4 grp + 3 of the pair's tiles
        if constexpr (GU) {
            uint2 hv;
            hv.x = h16_pair(silu_f(gt.x), up.x, silu_f(gt.y), up.y), hv.y = h16_pair(silu_f(gt.z), up.z, silu_f(gt.w), up.w);
            *reinterpret_cast<uint2*>(a.h16 + (size_t) orow * (a.nrows >> 1) + 16 * pr + 4 * grp) = hv;
        } else {
            float* o = a.out + (size_t) orow * a.nrows + 32 * pr + 4 * grp;
            *reinterpret_cast<float4*>(o) = make_float4(gt.x, gt.y, gt.z, gt.w);
            *reinterpret_cast<float4*>(o + 16) = make_float4(up.x, up.y, up.z, up.w);
        }
    };
    const int G = gridDim.x;
    int tot[MB_TP + 1] = {0, 0, 0, 0, 0};
    if (sorted) {
#pragma unroll
        for (int c = 0; c <= MB_TP; ++c) tot[c] = uniform(L.p_total[c]);
    }
    const bool split = nsuper <= 4;
    const int nbj = sorted ? tot[4] + tot[3] + tot[2] + (split ? 0 : tot[1]) : njall, nb = nbj * upj, np = sorted && split ? tot[1] * ppj : 0;
    int p_first = 0, p_last = 0;   // the block's stretch of the light pairs
    if (nb <= G) {
        // every heavy unit on a block of its own, block b's of the class its place in the order says: the blocks of a class
        // have the same share, and the blocks after b (they come first) are counted class by class
        const int b1 = (int) vb + 1;
        const int hi4 = tot[4] * upj, hi3 = hi4 + tot[3] * upj, hi2 = hi3 + tot[2] * upj;   // where the classes end (class 1: nb)
        const int c4 = w16_heavy_cost(4), c3 = w16_heavy_cost(3), c2 = w16_heavy_cost(2), c1 = w16_heavy_cost(1);
        const int mean = w16_mean(hi4 * c4 + (hi3 - hi4) * c3 + (hi2 - hi3) * c2 + (nb - hi2) * c1, np, G);
        const int s4 = max(0, mean - c4), s3 = max(0, mean - c3), s2 = max(0, mean - c2), s1 = max(0, mean - c1), s0 = mean;
        auto after = [&](int lo, int hi, int b) { return max(0, hi - max(lo, b)); };   // blocks of [lo, hi) from b on
        auto shares = [&](int b) { return after(nb, G, b) * s0 + after(hi2, nb, b) * s1 + after(hi3, hi2, b) * s2 + after(hi4, hi3, b) * s3 + after(0, hi4, b) * s4; };
        const int all = shares(0);
        // A stretch in which two jobs meet whose tokens do not fit the places together is two phases. Where that happens to lists of
        // so few pairs that a block has one phase, the stretches are whole eights of one job instead (us a launch, S = 4; units of
        // eight pairs / as their shares fall / eights): 128 jobs of some 6 tokens, 8 pairs a block, 19.5 / 27.2 / 19.8; 60 jobs of 16
        // tokens, 15 a block, 31.9 / 34.3 / 32.1. Not where few jobs are large (64 of 5 tokens, 8 a block, 19.2 / 19.0) nor at 9 to 13
        // pairs a block (80 jobs of 16 tokens, 10 a block, 31.2 / 26.1 / 31.1; 100, 12.5 a block, 31.4 / 29.6 / 31.0).
        const int most = nb < G ? s0 : hi2 < nb ? s1 : hi3 < hi2 ? s2 : hi4 < hi3 ? s3 : s4, alone = uniform(L.p_alone);
        const long load = (long) np * most;   // the longest stretch is load / all
        const bool eights = ppj % 8 == 0 && (load <= 8l * all ? 16 * alone > tot[1] : load > 13l * all && load <= 16l * all && 2 * alone > tot[1]);
        const int by = eights ? 3 : 0;
        const double inv = w16_inverse(all);
        p_first = uniform(w16_part(np >> by, shares(b1), all, inv) << by), p_last = uniform(w16_part(np >> by, shares(b1 - 1), all, inv) << by);
    } else if (sorted) {
        p_first = uniform(L.p_first), p_last = uniform(L.p_last);
    }
    // The oldest wave of a SIMD goes first and the block's waves drift apart between two barriers: every wave takes each
    // priority in turn, a super-step each
    auto turn = [&](int S) {
        switch (((wave >> 2) + S) & 3) {
            case 0: __builtin_amdgcn_s_setprio(0); break;
            case 1: __builtin_amdgcn_s_setprio(1); break;
            case 2: __builtin_amdgcn_s_setprio(2); break;
            default: __builtin_amdgcn_s_setprio(3); break;
        }
    };
    auto matrix_of = [&](int j, const fnx_bigjob* jb) {
        const int e = j >= nj ? 0 : uniform(j < W16_GU_HELD ? L.jw[j] : jb->w);
        return j >= nj ? a.w2 : a.ep ? uniform_ptr((const uint8_t*) a.ep[e]) : a.w + (size_t) e * a.stride;
    };
    // ---- the heavy units: sixteen pairs of tiles, a pair a wave
    auto heavy = [&](auto nt_tag, const fnx_bigjob* jb, int n, const uint8_t* we, int pr) {
        constexpr int NT = decltype(nt_tag)::value;
        const bool mine = pr < ppj;
        const __amdgpu_buffer_rsrc_t mg = ly.tiles(we, first_tile(min(pr, ppj - 1))), mu = ly.tiles(we, second_tile(min(pr, ppj - 1)));
        const int oput = tid < n ? jb->out[tid] : -1;   // (up to 64 tokens: the first wave)
        int y[NT];   // the wave's tokens' rows: tokens wave, wave + 16, .. (past the job's last: that one again)
#pragma unroll
        for (int i = 0; i < NT; ++i) y[i] = uniform(jb->y[min(wave + 16 * i, n - 1)]);
        v4f accg[NT], accu[NT];
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) accg[tt] = accu[tt] = v4f{0.f, 0.f, 0.f, 0.f};
        SuperFields f = ly.load(mg, 0), fu = ly.load(mu, 0);
        // Super-steps whose activations fit LDS together come in together (jobs of 17 .. 32 tokens two at a time: 256 of them 74.4 -> 72.6 us a launch,
        // of 20 73.4 -> 69.9; 512 rows, eight of 128 experts, 125.0 -> 121.3 a chunk).
        constexpr int SB = MB_TP / NT;
        for (int S0 = 0; S0 < nsuper; S0 += SB) {
            const int cnt = min(SB, nsuper - S0);
            __syncthreads();   // the tile before has been read
            if (S0 == 0 && tid < FNX_PF_JOB) L.orow[tid] = oput;
            for (int s = 0; s < cnt; ++s)
#pragma unroll
                for (int i = 0; i < NT; ++i)   // a token's super-step a wave instruction, 16 bytes a lane
                    lds_load16(a.x + (size_t) y[i] * a.ldx + 128 * PS * (S0 + s), xl16, xt_at + (16 * NT * s + wave + 16 * i) * W16_XROW);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            for (int s = 0; s < cnt; ++s) {
                turn(S0 + s);
                const int Sn = min(S0 + s + 1, nsuper - 1);
                SuperFields nf, nfu;
                w16_super_pair<NT>(L.tab, xlane + 16 * NT * s * W16_XROW, f, fu, accg, accu, [&] { nf = ly.load(mg, Sn), nfu = ly.load(mu, Sn); });
                f = nf, fu = nfu;
            }
        }
        // lane: token r of each tile, rows 4 grp .. 4 grp + 3 of the pair's tiles
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
            const int orow = mine ? L.orow[tt * 16 + r] : -1;
            if (orow >= 0) put(orow, pr, accg[tt], accu[tt]);
        }
    };
    for (int round = 0; round * G < nb; ++round) {
        const int u = round * G + ((round & 1) ? G - 1 - (int) vb : (int) vb);
        if (u >= nb) continue;   // the same for the whole block
        const int jo = u / upj, q = u - jo * upj, j = sorted ? (int) uniform(L.jorder[jo]) : jo;
        const fnx_bigjob* jb = job_at(j);
        const int n = uniform(n_of(j));
        if (n < 1) continue;
        const uint8_t* we = matrix_of(j, jb);
        const int pr = q * W16_WAVES + wave;
        if (n > 48) heavy(std::integral_constant<int, 4>{}, jb, n, we, pr);
        else if (n > 32) heavy(std::integral_constant<int, 3>{}, jb, n, we, pr);
        else if (n > 16) heavy(std::integral_constant<int, 2>{}, jb, n, we, pr);
        else heavy(std::integral_constant<int, 1>{}, jb, n, we, pr);
    }
    // ---- the light pairs, in phases: the jobs of the block's stretch as long as their tokens fit the sixteen places that LDS has for
    // a row's S tiles ([S][place]), all staged at once; the waves then take the phase's pairs one by one as they come free and
    // meet only where a phase ends
    for (int p0 = p_first; p0 < p_last;) {   // the same for the whole block
        __syncthreads();   // the units before have been read
        if (wave == 0) {   // the phase: lane k its k-th job
            const int jo = p0 / ppj + lane;
            const bool in = jo * ppj < p_last && lane < 16;
            const int j = in ? (int) L.jorder[nbj + jo] : 0, n = in ? n_of(j) : 16;   // 1 .. 16
            int incl = n;
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                const int up = __shfl_up(incl, o, 16);
                if ((lane & 15) >= o) incl += up;
            }
            const int jobs = __popcll(__ballot(in && incl <= 16));   // (at least one)
            if (lane < jobs) {
                L.ph_job[lane] = (unsigned short) j;
                L.ph_first[lane] = (unsigned char) (incl - n);
            }
            if (lane == 0) L.ph_jobs = jobs, L.ph_next = p0 + W16_WAVES;
            if (lane == jobs - 1) L.ph_tokens = incl;
        }
        __syncthreads();
        const int jobs = uniform(L.ph_jobs), jo0 = p0 / ppj, pe = min(p_last, (jo0 + jobs) * ppj), tokens = uniform(L.ph_tokens);
        if (wave < tokens) {   // a place a wave: the job it belongs to is the last one that begins at or before it
            const int k = __popcll(__ballot(lane < jobs && (int) L.ph_first[lane & 15] <= wave)) - 1;
            const int y = uniform(job_at((int) L.ph_job[k])->y[wave - (int) L.ph_first[k]]);
            for (int S = 0; S < nsuper; ++S) lds_load16(a.x + (size_t) y * a.ldx + 128 * PS * S, xl16, xt_at + (16 * S + wave) * W16_XROW);
        }
        if (pe - p0 <= W16_WAVES / 2) {   // pairs for half of the waves: a wave a tile, the up tiles' sums go over to the gate tiles' waves
            constexpr int HALF = W16_WAVES / 2;
            const int q = p0 + wave % HALF, up = wave / HALF, jo = min(q, pe - 1) / ppj, pr = min(q, pe - 1) - jo * ppj;
            const int k = jo - jo0, j = uniform((int) L.ph_job[k]), at = uniform((int) L.ph_first[k]);
            const fnx_bigjob* jb = job_at(j);
            const int orow = q < pe && !up && r < n_of(j) ? jb->out[r] : -1;
            const __amdgpu_buffer_rsrc_t m = ly.tiles(matrix_of(j, jb), up ? second_tile(pr) : first_tile(pr));
            SuperFields f = ly.load(m, 0);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            v4f acc[MB_TP] = {};
            const uint8_t* xk = L.xt + min(at + r, 15) * W16_XROW + 64 * PS * grp;
            for (int S = 0; S < nsuper && q < pe; ++S) {
                turn(S);
                const SuperFields nf = ly.load(m, min(S + 1, nsuper - 1));
                w16_super_step<PS>(L.tab, xk + S * 16 * W16_XROW, f, 1, acc);
                f = nf;
            }
            if (up) L.xs[wave % HALF][lane] = make_float4(acc[0].x, acc[0].y, acc[0].z, acc[0].w);
            __syncthreads();
            if (orow >= 0) {
                const float4 ut = L.xs[wave % HALF][lane];
                put(orow, pr, acc[0], v4f{ut.x, ut.y, ut.z, ut.w});
            }
            p0 = pe;
            continue;
        }
        // a wave's pair p: its job's place in the phase, its matrix's two rows of tiles
        int p = p0 + wave;
        __amdgpu_buffer_rsrc_t mg, mu;
        auto tiles_of = [&](int q) {
            const int jo = q / ppj, pr = q - jo * ppj, j = uniform((int) L.ph_job[jo - jo0]);
            const uint8_t* we = matrix_of(j, job_at(j));
            mg = ly.tiles(we, first_tile(pr)), mu = ly.tiles(we, second_tile(pr));
        };
        tiles_of(min(p, pe - 1));
        SuperFields f = ly.load(mg, 0), fu = ly.load(mu, 0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        while (p < pe) {
            int pn = 0;
            if (lane == 0) pn = atomicAdd(&L.ph_next, 1);
            pn = uniform(pn);
            const int jo = p / ppj, pr = p - jo * ppj, k = jo - jo0, j = uniform((int) L.ph_job[k]), at = uniform((int) L.ph_first[k]);
            const fnx_bigjob* jb = job_at(j);
            const int orow = r < n_of(j) ? jb->out[r] : -1;
            const uint8_t* xk = L.xt + min(at + r, 15) * W16_XROW + 64 * PS * grp;   // (a lane without a token: some place's values, its sums not kept)
            v4f accg[1] = {v4f{0.f, 0.f, 0.f, 0.f}}, accu[1] = {v4f{0.f, 0.f, 0.f, 0.f}};
            for (int S = 0; S < nsuper; ++S) {
                turn(S);
                SuperFields nf, nfu;
                w16_super_pair<1>(L.tab, xk + S * 16 * W16_XROW, f, fu, accg, accu, [&] {
                    if (S + 1 == nsuper) tiles_of(min(pn, pe - 1));
                    const int Sn = S + 1 < nsuper ? S + 1 : 0;
                    nf = ly.load(mg, Sn), nfu = ly.load(mu, Sn);
                });
                f = nf, fu = nfu;
            }
            if (orow >= 0) put(orow, pr, accg[0], accu[0]);
            p = pn;
        }
        p0 = pe;
    }
}

}  // namespace fnx
