// How the one-launch verify window (k_moe_window.h) cuts a window's work over the grid: which row a block belongs to, its
// router rows, its run of gate|up items, its units of the down matrices, and how many blocks each of a row's two
// hand-overs waits for. Plain functions of integers, compiled for the device and (by the plan test) for the host, so
// that every count a block waits for can be checked against the blocks that arrive without running a kernel.
#pragma once

#include <stddef.h>

#if defined(__HIPCC__)
#define FNX_HOST_DEVICE __host__ __device__
#else
#define FNX_HOST_DEVICE
#endif

namespace fnx {

constexpr int WN_WAVES = 16;   // waves a block

// The even cut. (nk, k0, per_row, ipb, nbi: its gate|up items in runs of [shared, picks ..]. The window deals them otherwise, win_work below, and
// these are for the host check of the cut alone.)
struct WinPlan {
    int Tl;        // rows of the window that count
    int G;         // blocks a row, a power of two (win_work below: not always); block b belongs to row b / G and is the row's block b % G
    int nk, k0;    // matrices a row's gate|up items walk (the shared expert's if k0 == 0, then the picks'), the first one
    int qpp;       // blocks of 32 h values a pair
    int per_row;   // gate|up items a row: qpp * nk, numbered (block of 32, matrix)
    int ipb;       // items a block: block g takes items [g * ipb, min(per_row, (g + 1) * ipb))
    int nbi;       // blocks of a row that have items: the count the row's h hand-over waits for
    int rpb;       // router rows a block: block g takes rows [g * rpb, min(nexp, (g + 1) * rpb))
    int upb;       // units of a down matrix a block: block g takes units [g * upb, (g + 1) * upb)
    int R;         // of them a wave and trip; wave w < dwaves takes units g * upb + w * R .. + R - 1
    int dwaves;    // waves with units
};

FNX_HOST_DEVICE inline int win_log2(int v) { return 31 - __builtin_clz((unsigned) v); }   // (rounded down, v >= 1)
// nb: blocks of the grid; Tl >= 1 rows that count; nexp experts, topk picks a row; shared: the shared expert's matrices are
// this launch's; ff: expert width (a multiple of 256: the down matrices have 2048 rows of ff columns = ff units of 64 sub-blocks)
FNX_HOST_DEVICE inline WinPlan win_plan(int nb, int Tl, int nexp, int topk, bool shared, int ff) {
    WinPlan p;
    p.Tl = Tl;
    p.G = 1 << win_log2(nb / Tl);
    if (p.G > ff) p.G = ff;   // at least one unit of the down matrices a block (ff is a power of two times 256)
    const int lg = win_log2(p.G);   // (shifts: a block does all of this before its first load, and a division is some thirty instructions)
    p.k0 = shared ? 0 : 1;
    p.nk = topk + 1 - p.k0;
    p.qpp = ff / 32;
    p.per_row = p.qpp * p.nk;
    p.ipb = (p.per_row + p.G - 1) >> lg;
    p.nbi = (p.per_row + p.ipb - 1) / p.ipb;
    p.rpb = (nexp + p.G - 1) >> lg;
    p.upb = ff >> lg;
    p.dwaves = p.upb < WN_WAVES ? p.upb : WN_WAVES;
    p.R = p.upb < WN_WAVES ? 1 : p.upb / WN_WAVES;
    return p;
}
// The work as the window deals it. Two things of the cut above cost time. A power of two of blocks a row leaves up to 44 % of the grid
// without work at 5 .. 7 and 9 .. 15 rows: blocks are taken in fours up to nb / Tl where that makes a block's routed items fewer
// and the even cut leaves it more than half a unit of the down matrices a wave. In fours, since the blocks that take the same router rows and
// shared items then lie on one or two of the eight XCDs, whose L2 they share (252 blocks at 21 a row were slower than 192 at 16: Q4_K, 12 rows
// 47.1 -> 51.0 us, at 20 a row 47.2), and in eights, on one, where that leaves out a block in sixteen at most (3 rows of 5 of 512 experts of width 1,024, us at 64 / 84 /
// 80 blocks a row: IQ3_S 28.2 / 28.4 / 27.9, Q4_K 27.6 / 27.8 / 27.2; of 10 IQ3_S 37.4 / 36.5 / 36.2, but Q8_0 74.7 / 69.7 / 70.5). Not where a row gets
// only a few blocks more, by the type (win_least_growth, k_window_formats.h). And the shared expert's items need no pick, so they are dealt apart from the routed ones, to
// run while the row's logits gather: to the row's last blocks where there are more blocks than items, which have the fewest
// routed ones; the routed ones as evenly as they go, since they are what a block does once its picks are known. us a window, 10 of 512
// experts of width 512 (the even cut in runs of [shared, picks ..] / this): IQ3_S 2 rows 26.8 / 25.8, 7 rows 37.2 / 34.9, 9 rows 46.6 / 38.9, 12 rows
// 47.3 / 44.2, 16 rows 49.7 / 49.0; Q4_K 7 rows 37.0 / 35.8; Q8_0 9 rows 110.8 / 80.4; 3 and 4 rows the same. The
// units of the down matrices no longer divide evenly: the last wave of a block may reach into the next block's, the last block may have fewer or
// none. (The kernel keeps a wave's units inside the matrix; a unit that two waves make has the same value from both.) The launch
// brings the plan of all its rows: made by every block it came before the block's first load (2 rows 26.4 -> 25.8 us).
struct WinWork {
    int Tl, G;               // as above, G not always a power of two
    int routed, ipb, more;   // routed items a row, numbered (block of 32, pick): ipb a block in order, one more for the first `more` blocks
    int shared, spb;         // the shared expert's items a row (0: it runs elsewhere); win_shared_first(g) .. + spb - 1 of them
    int nbi;                 // blocks of a row that have items: the count the row's h hand-over waits for
    int rpb, upb, R, dwaves; // as above; units a block and wave at most
};
FNX_HOST_DEVICE inline int win_row(const WinWork& p, int b) { return (p.G & (p.G - 1)) == 0 ? b >> win_log2(p.G) : b / p.G; }   // block b's
FNX_HOST_DEVICE inline int win_routed_first(const WinWork& p, int g) { return g * p.ipb + (g < p.more ? g : p.more); }
FNX_HOST_DEVICE inline int win_shared_first(const WinWork& p, int g) { return (p.G > p.shared ? p.G - 1 - g : g) * p.spb; }
// least: a row's blocks are taken in fours where that makes them more by over `least` eighths; eights: in eights where the above says so. (The window itself,
// where a row count on the device makes every block work this out before its first load, goes without both: with them eight rounds with a chain of three
// drafts took 6,682 us, 6,652 without, and a window of two rows, whose code only shares its registers with that, 25.98 and 25.85.)
FNX_HOST_DEVICE inline WinWork win_work(int nb, int Tl, int nexp, int topk, bool shared, int ff, int least = 0, bool eights = true) {
    const WinPlan e = win_plan(nb, Tl, nexp, topk, shared, ff);
    const int lg = win_log2(e.G), per = nb / Tl, all = eights && per >= 64 ? per / 8 * 8 : per / 4 * 4, routed = e.qpp * topk;
    WinWork p{Tl, e.G, routed, routed >> lg, 0, shared ? e.qpp : 0, 0, 0, e.rpb, e.upb, e.R, e.dwaves};
    if (8 * (all - e.G) > least * e.G && e.upb > WN_WAVES / 2 && (routed + all - 1) / all < (routed + e.G - 1) >> lg) {
        p.G = all;
        p.ipb = routed / all;
        p.rpb = (nexp + all - 1) / all;
        p.upb = (ff + all - 1) / all;
        p.R = p.upb <= WN_WAVES ? 1 : p.upb <= 2 * WN_WAVES ? 2 : 4;
        p.dwaves = (p.upb + p.R - 1) / p.R;
    }
    p.more = routed - p.ipb * p.G;
    p.spb = p.shared > p.G ? (p.shared + p.G - 1) / p.G : p.shared > 0;
    const int with_routed = p.ipb ? p.G : p.more, with_shared = p.spb > 1 ? (p.shared + p.spb - 1) / p.spb : p.shared;
    // the blocks with routed items come first; those with shared ones are the first, or (one each) the last
    p.nbi = p.G > p.shared ? (with_routed + with_shared < p.G ? with_routed + with_shared : p.G) : with_routed > with_shared ? with_routed : with_shared;
    return p;
}
// Where a split-Q8_0 shared expert's three dense launches before the window keep what they hand on, in the caller's workspace
// buffers gu ([P + T][2 ff] floats, P = T topk pairs) and part ([P + T][n] floats). The f32 gate|up rows lie where the operators
// put them, behind the pairs' rows of gu: the window's own records of h (hq_words words a block of 32) end below, and T
// topk + T rows hold them whatever topk is. The q8_1 rows of h and the down rows share part.
struct WinShared {
    size_t gu;       // floats from gu: [T][2 ff]
    size_t hq;       // floats from part: [T][ff / 32] q8_1 blocks of 36 bytes
    size_t down;     // floats from part: [T][n], on a multiple of 256 bytes
    size_t gu_end, part_end;   // floats of gu and of part up to where these end
};
FNX_HOST_DEVICE inline WinShared win_shared(int T, int topk, int n, int ff) {
    WinShared w;
    w.gu = (size_t) T * topk * 2 * ff;
    w.hq = 0;
    w.down = ((size_t) T * (ff / 32) * 36 + 255) / 256 * 64;
    w.gu_end = w.gu + (size_t) T * 2 * ff;
    w.part_end = w.down + (size_t) T * n;
    return w;
}
// the most units a wave can hold a trip for rows of SBR sub-blocks (the registers of a block of sixteen waves)
FNX_HOST_DEVICE inline int win_rmax(int sbr) { return sbr / 8; }

}  // namespace fnx
