// What the one-launch verify window (k_moe_window.h) needs to know of a weight type: a unit of 64 sub-blocks of 32 weights
// in memory (rows lie one after the other, so a unit is UNIT contiguous bytes whatever the row's length), a lane's share of
// it as loaded, and the term of the lane's sub-block against its activations. WinUnit64 is the re-laid IQ3_S the window was
// built for; WinQt<type> are the other types of kernels.cu:2454-2471 as the file holds them (block layouts and terms:
// k_qtypes.h), whose lanes read their own block's fields straight from the file's layout: at 1,152 to 2,176 bytes a unit and
// some 40 vector instructions a lane they are bound by memory, not by the decode, and no load-time re-laying is needed.
// Measured (512 experts, width 512, ten picks a row): Q4_K at 7 rows 41 us for 138 MB, at 16 rows 60.5 (operators one by one,
// nine launches: 143 and 261); a window of one row of IQ4_XS experts of width 256, all dependencies and no bytes, 21.6 (37.6).
#pragma once

#include "k_moe_layer.h"
#include "k_qtypes.h"

namespace fnx {

// How a type uses the sum of a block's activations: not at all; the sum of its int8 values (the K-quants' minimum); the
// q8_1 block's own sum field (Q4_0's offset, Q5_1's minimum)
enum { WIN_SUM_NONE = 0, WIN_SUM_CODES = 1, WIN_SUM_FIELD = 2 };

// win_work's least growth of a row's blocks, by type: what a type's loads draw with seven CUs of eight (7 rows at 32 blocks a row; 36 take the rest)
// or three of four (6 rows, 32 or 40). Q8_0 and the 4-bit types without a minimum draw 3.0 to 3.9 TB/s there and want every CU; IQ3_S, the K-quants and
// Q5_1, at 3.7 to 4.6, lose to the second XCD that 36 blocks a row spread a slice over, Q5_1 to the 40 too. us a window, 512 experts of width 1,024,
// 7 rows, at 32 / 36 blocks, 9 picks and 16: Q8_0 124.4 / 119.9, 198.2 / 195.1; Q4_0 75.3 / 73.1, 117.7 / 116.4; IQ4_NL 75.6 / 74.0, 119.3 / 118.3; IQ4_XS 58.1 / 58.5,
// 87.4 / 88.7, but of 256 experts, 10 picks, 60.2 / 59.8; IQ3_S 49.7 / 49.2, 75.4 / 76.4; Q4_K 54.5 / 56.8, 82.9 / 89.3; Q5_K 65.3 / 66.9, 99.7 / 104.0; Q5_1 67.0 /
// 69.7, 103.6 / 109.4. 6 rows, 10 picks, at 32 / 40: Q5_1 66.6 / 68.8, Q4_K 54.2 / 54.7, Q5_K 66.6 / 65.2, IQ3_S 52.8 / 50.3, Q8_0 130.0 / 118.2.
constexpr int win_least_growth(uint32_t type) {
    return type == QT_Q5_1 ? 2 : type == QT_Q8_0 || type == QT_Q4_0 || type == QT_IQ4_NL || type == QT_IQ4_XS ? 0 : 1;
}

struct WinUnit64 {
    static constexpr int UNIT = UNIT_BYTES, SUM = WIN_SUM_NONE;
    static constexpr bool TAB = true;   // decodes through the signed codebook in LDS
    static constexpr int MAXR = 4, NBUF = 3;   // units a wave's trip holds at most; trips' buffers where a trip holds one or two
    typedef PackedSub Raw;
    typedef PackedVOffs Offs;
    typedef __amdgpu_buffer_rsrc_t Mat;
    struct Act {
        int xs[8];
        float dx;
    };
    static __device__ __forceinline__ Offs offs(int lane) { return packed_voffs(lane); }
    static __device__ __forceinline__ Mat matrix(const uint8_t* e) { return matrix_rsrc(e); }   // e: wave-uniform
    static __device__ __forceinline__ Raw load(Mat m, int unit_byte, const Offs& o) { return load_packed_buf(m, unit_byte, o); }
    static __device__ __forceinline__ Act act_x(const uint32_t (*xq)[FNX_Q8_1_BLOCK / 4], int lane) {
        Act r;
        const uint32_t* xb = xq[lane];
        r.dx = half_bits_to_float(xb[0] & 0xFFFFu);
#pragma unroll
        for (int j = 0; j < 8; ++j) r.xs[j] = (int) xb[1 + j];
        return r;
    }
    static __device__ __forceinline__ Act act_h(const uint32_t (*hq)[HQ_WORDS], int kb, int) {
        const uint32_t* hb = hq[kb];
        const uint4 lo = *reinterpret_cast<const uint4*>(hb), hi = *reinterpret_cast<const uint4*>(hb + 4);
        return Act{{(int) lo.x, (int) lo.y, (int) lo.z, (int) lo.w, (int) hi.x, (int) hi.y, (int) hi.z, (int) hi.w}, __uint_as_float(hb[8])};
    }
    static __device__ __forceinline__ float term(const Raw& q, const uint32_t* tab, const Act& x, int sc_shift) {
        int w4[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) w4[j] = *reinterpret_cast<const int*>(reinterpret_cast<const uint8_t*>(tab) + packed_addr(q.idx, j));
        const int sc = 1 + 2 * (int) ((q.sc >> sc_shift) & 0xFu);
        const float dw = half_bits_to_float(q.d);
        int sum = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) sum = __builtin_amdgcn_sdot4(w4[j], x.xs[j], sum, false);
        // one sub-block's term as the reference forms it: (d_w * d_x) * (float) (sumi * (1 + 2 s))
        return (dw * x.dx) * (float) __mul24(sum, sc);
    }
};

typedef __attribute__((address_space(1), aligned(2))) const v4u g_v4u_a2;
typedef __attribute__((address_space(1), aligned(2))) const v2u g_v2u_a2;
typedef __attribute__((address_space(1), aligned(2))) const unsigned short g_u16_a2;

template <uint32_t TYPE>
struct WinQt {
    static constexpr bool K = TYPE == QT_Q4_K || TYPE == QT_Q5_K;
    static constexpr int BLOCK = TYPE == QT_Q4_0 || TYPE == QT_IQ4_NL ? 18 : TYPE == QT_Q5_1 ? 24 : TYPE == QT_Q8_0 ? 34 : TYPE == QT_IQ4_XS ? 136 : TYPE == QT_Q4_K ? 144 : 176;
    static constexpr int UNIT = TYPE == QT_IQ4_XS || K ? 8 * BLOCK : 64 * BLOCK;
    static constexpr int SUM = K ? WIN_SUM_CODES : TYPE == QT_Q4_0 || TYPE == QT_Q5_1 ? WIN_SUM_FIELD : WIN_SUM_NONE;
    static constexpr bool TAB = false;
    static constexpr int MAXR = 2, NBUF = TYPE == QT_Q5_K ? 2 : 3;   // (a lane's share is up to twelve registers: a wave with four units makes them two at a time)
    // head: the block's scale (and minimum, sub-block scales); q: the lane's 16 bytes of values; q2: Q8_0's second half, Q5_K's fifth bits
    static constexpr int HEAD = K ? 4 : TYPE == QT_IQ4_XS || TYPE == QT_Q5_1 ? 2 : 1;
    static constexpr bool SECOND = TYPE == QT_Q8_0 || TYPE == QT_Q5_K;
    struct Raw {
        uint32_t head[HEAD];
        v4u q, q2;
    };
    struct Offs {
        uint32_t head, q;
    };
    typedef const uint8_t* Mat;
    struct Act {
        int xs[8];
        float dx;
        uint32_t sum;   // the codes' sum (an int) or the field (a float's bits)
    };
    static __device__ __forceinline__ Offs offs(int lane) {
        Offs o;
        if constexpr (K) {
            // A K-quant's pair of sub-blocks shares 32 bytes, a nibble each. The pair's lanes split the bytes instead of the
            // sub-blocks - lane 2 i takes the first sixteen of both, lane 2 i + 1 the last - and swap half sums (an integer each).
            o.head = (uint32_t) (lane >> 3) * BLOCK;
            o.q = o.head + (TYPE == QT_Q5_K ? 48 : 16) + 32 * ((lane & 7) >> 1) + 16 * (lane & 1);
        } else if constexpr (TYPE == QT_IQ4_XS) {
            o.head = (uint32_t) (lane >> 3) * BLOCK;
            o.q = o.head + 8 + 16 * (lane & 7);
        } else {
            o.head = (uint32_t) lane * BLOCK;
            o.q = o.head + (TYPE == QT_Q5_1 ? 8 : 2);
        }
        return o;
    }
    static __device__ __forceinline__ Mat matrix(const uint8_t* e) { return e; }
    static __device__ __forceinline__ Raw load(Mat m, int unit_byte, const Offs& o) {
        const gbytes u = as_global(uniform_ptr(m + unit_byte));
        uint32_t oh = o.head, oq = o.q;
        asm volatile("" : "+v"(oh), "+v"(oq));   // keeps the zero-extensions next to the loads (SGPR-base addressing)
        Raw r;
        if constexpr (HEAD == 4) {
            const v4u h = *(g_v4u_a2*) (u + oh);
            r.head[0] = h.x, r.head[1] = h.y, r.head[2] = h.z, r.head[3] = h.w;
        } else if constexpr (HEAD == 2) {
            const v2u h = *(g_v2u_a2*) (u + oh);
            r.head[0] = h.x, r.head[1] = h.y;
        } else {
            r.head[0] = *(g_u16_a2*) (u + oh);
        }
        r.q = *(g_v4u_a2*) (u + oq);
        if constexpr (TYPE == QT_Q8_0) r.q2 = *(g_v4u_a2*) (u + oq + 16);
        else if constexpr (TYPE == QT_Q5_K) {
            uint32_t o5 = o.head + 16 + 16 * (threadIdx.x & 1);
            asm volatile("" : "+v"(o5));
            r.q2 = *(g_v4u_a2*) (u + o5);
        } else r.q2 = v4u{0u, 0u, 0u, 0u};
        return r;
    }
    // a lane's activations: its sub-block's 32 codes - for a K-quant its half of the pair's, first sub-block then second. word(sb, j):
    // word j of sub-block sb's codes
    template <class W>
    static __device__ __forceinline__ void codes(int (&xs)[8], int kb, W word) {
        if constexpr (K) {
            const int h = 4 * (kb & 1), e = kb & ~1;
#pragma unroll
            for (int j = 0; j < 4; ++j) xs[j] = (int) word(e, h + j), xs[4 + j] = (int) word(e + 1, h + j);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) xs[j] = (int) word(kb, j);
        }
    }
    static __device__ __forceinline__ Act act_x(const uint32_t (*xq)[FNX_Q8_1_BLOCK / 4], int lane) {
        Act r;
        const uint32_t head = xq[lane][0];
        r.dx = half_bits_to_float(head & 0xFFFFu);
        r.sum = 0;
        codes(r.xs, lane, [&](int sb, int j) { return xq[sb][1 + j]; });
        if constexpr (SUM == WIN_SUM_FIELD) r.sum = __float_as_uint(half_bits_to_float(head >> 16));
        if constexpr (SUM == WIN_SUM_CODES) {
            int s = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) s = __builtin_amdgcn_sdot4(0x01010101, (int) xq[lane][1 + j], s, false);
            r.sum = (uint32_t) s;
        }
        return r;
    }
    static __device__ __forceinline__ Act act_h(const uint32_t (*hq)[HQ_WORDS], int kb, int) {   // (word 8: the scale; word 9: the sum, as the type wants it)
        Act r;
        if constexpr (K) {
            const int h = 4 * (kb & 1), e = kb & ~1;
            const uint4 a = *reinterpret_cast<const uint4*>(&hq[e][h]), b = *reinterpret_cast<const uint4*>(&hq[e + 1][h]);
            r = Act{{(int) a.x, (int) a.y, (int) a.z, (int) a.w, (int) b.x, (int) b.y, (int) b.z, (int) b.w}, 0.f, 0u};
        } else {
            const uint4 a = *reinterpret_cast<const uint4*>(&hq[kb][0]), b = *reinterpret_cast<const uint4*>(&hq[kb][4]);
            r = Act{{(int) a.x, (int) a.y, (int) a.z, (int) a.w, (int) b.x, (int) b.y, (int) b.z, (int) b.w}, 0.f, 0u};
        }
        r.dx = __uint_as_float(hq[kb][8]);
        if constexpr (SUM != WIN_SUM_NONE) r.sum = hq[kb][9];
        return r;
    }
    // the sub-block's term: k_qtypes.h's qt_decode and qt_term over the loaded fields
    static __device__ __forceinline__ float term(const Raw& q, const uint32_t*, const Act& x, int) {
        const float d = half_bits_to_float(q.head[0] & 0xFFFFu);
        if constexpr (K) {
            const int sb = threadIdx.x & 7;
            int pe = 0, po = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t lo = q.q[j] & 0x0F0F0F0Fu, hi = (q.q[j] >> 4) & 0x0F0F0F0Fu;
                if constexpr (TYPE == QT_Q5_K) {
                    const uint32_t f = q.q2[j] >> (sb & 6);   // bit 0: the pair's first sub-block, bit 1: its second
                    lo |= (f & 0x01010101u) << 4;
                    hi |= ((f >> 1) & 0x01010101u) << 4;
                }
                pe = __builtin_amdgcn_sdot4((int) lo, x.xs[j], pe, false);
                po = __builtin_amdgcn_sdot4((int) hi, x.xs[4 + j], po, false);
            }
            const bool odd = sb & 1;
            const int other = __builtin_amdgcn_update_dpp(0, odd ? pe : po, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
            const int dot = (odd ? po : pe) + other;
            // ggml's get_scale_min_k4 from the three words of packed scales
            const uint32_t s0 = q.head[1] >> (8 * (sb & 3)), s1 = q.head[2] >> (8 * (sb & 3)), s2 = q.head[3] >> (8 * (sb & 3));
            const bool up = sb >= 4;
            const int sc = (int) (up ? (s2 & 0xFu) | ((s0 >> 2) & 0x30u) : s0 & 63u), m = (int) (up ? ((s2 >> 4) & 0xFu) | ((s1 >> 2) & 0x30u) : s1 & 63u);
            const float dmin = half_bits_to_float(q.head[0] >> 16);
            return d * (x.dx * (float) (dot * sc)) - dmin * (x.dx * (float) ((int) x.sum * m));
        } else {
            int w4[8];
            if constexpr (TYPE == QT_Q8_0) {
#pragma unroll
                for (int j = 0; j < 4; ++j) w4[j] = (int) q.q[j], w4[4 + j] = (int) q.q2[j];
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {   // low nibbles: values 0..15; high nibbles: 16..31
                    uint32_t lo = q.q[j] & 0x0F0F0F0Fu, hi = (q.q[j] >> 4) & 0x0F0F0F0Fu;
                    if constexpr (TYPE == QT_IQ4_NL || TYPE == QT_IQ4_XS) lo = iq4_values4(lo), hi = iq4_values4(hi);
                    if constexpr (TYPE == QT_Q5_1) {   // bit 4 j + b of qh to bit 4 of byte b: one multiply spreads four bits
                        lo |= (((q.head[1] >> (4 * j)) & 0xFu) * 0x00204081u & 0x01010101u) << 4;
                        hi |= (((q.head[1] >> (16 + 4 * j)) & 0xFu) * 0x00204081u & 0x01010101u) << 4;
                    }
                    w4[j] = (int) lo, w4[4 + j] = (int) hi;
                }
            }
            int dot = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) dot = __builtin_amdgcn_sdot4(w4[j], x.xs[j], dot, false);
            if constexpr (TYPE == QT_Q4_0) return d * ((float) dot * x.dx - 8.0f * __uint_as_float(x.sum));
            else if constexpr (TYPE == QT_Q5_1) return (float) dot * (d * x.dx) + half_bits_to_float(q.head[0] >> 16) * __uint_as_float(x.sum);
            else if constexpr (TYPE == QT_IQ4_XS) {
                const int ib = threadIdx.x & 7;
                const int sc = (int) (((q.head[1] >> (4 * ib)) & 0xFu) | (((q.head[0] >> (16 + 2 * ib)) & 3u) << 4)) - 32;
                return (d * x.dx) * (float) (dot * sc);
            } else return (d * x.dx) * (float) dot;
        }
    }
};

}  // namespace fnx
