// Host-side check of the verify window's work (win_work in csrc/moe_window_plan.h) for the types that take blocks in fours only where a row gets
// more of them (`least`), and as the window works it out on the device (fours without eights): over grids, rows, widths and picks the blocks are
// walked as the kernel walks them, and `least` changes nothing but which of the two cuts it is.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <vector>

#include "moe_window_plan.h"

using namespace fnx;

static long checked = 0;
static void require(bool ok, const char* what, int nb, int Tl, int ff, int topk, int shared, int least) {
    ++checked;
    if (ok) return;
    std::printf("FAILED %s: blocks %d rows %d ff %d topk %d shared %d least %d\n", what, nb, Tl, ff, topk, shared, least);
    std::exit(1);
}

int main() {
    const int nexp = 100;
    long held = 0, fours = 0;
    for (int nb : {256, 304, 320, 512})
        for (int Tl = 1; Tl <= 16 && WN_WAVES * Tl <= nb; ++Tl)
            for (int ff : {256, 512, 1024})
                for (int topk = 1; topk <= 16; ++topk)
                    for (int shared = 0; shared < 2; ++shared)
                        for (int least : {0, 1, 2})
                            for (bool eights : {true, false}) {
#define REQ(c, what) require(c, what, nb, Tl, ff, topk, shared, least)
                                const WinWork p = win_work(nb, Tl, nexp, topk, shared != 0, ff, least, eights), all = win_work(nb, Tl, nexp, topk, shared != 0, ff, 0, eights);
                                const WinPlan e = win_plan(nb, Tl, nexp, topk, shared != 0, ff);
                                const bool grown = all.G != e.G && 8 * (all.G - e.G) > least * e.G;
                                held += all.G != e.G && !grown;
                                fours += p.G % 8 == 4;
                                if (grown) REQ(std::memcmp(&p, &all, sizeof p) == 0, "the deal of the other types");
                                else REQ(p.G == e.G && p.R == e.R && p.dwaves == e.dwaves && p.upb == e.upb && p.rpb == e.rpb && p.upb * p.G == ff, "the even cut");
                                REQ(p.G >= WN_WAVES && p.G * Tl <= nb && p.rpb * p.G >= nexp, "blocks and router rows");
                                std::vector<int> item(p.routed + p.shared, 0), unit(ff, 0);
                                int with = 0;
                                for (int g = 0; g < p.G; ++g) {
                                    const int s0 = win_shared_first(p, g), I0 = win_routed_first(p, g);
                                    int n = 0;
                                    for (int s = s0; s < s0 + p.spb; ++s)
                                        if (s >= 0 && s < p.shared) ++item[p.routed + s], ++n;
                                    for (int i = I0; i < I0 + p.ipb + (g < p.more); ++i, ++n) {
                                        REQ(i >= 0 && i < p.routed, "a routed item");
                                        ++item[i];
                                    }
                                    with += n > 0;
                                    for (int w = 0; w < p.dwaves; ++w) {
                                        const int at = g * p.upb + w * p.R, u0 = at < ff - p.R ? at : ff - p.R;
                                        if (at >= ff) continue;
                                        REQ(u0 >= 0, "a unit inside the matrix");
                                        for (int r = 0; r < p.R; ++r) ++unit[u0 + r];
                                    }
                                }
                                for (int v : item) REQ(v == 1, "every item once");
                                for (int v : unit) REQ(v >= 1, "every unit");
                                REQ(with == p.nbi, "the h hand-over's count");
                                const bool even = p.dwaves * p.R == p.upb && p.upb * p.G == ff;
                                REQ(p.dwaves >= 1 && p.dwaves <= WN_WAVES && p.R <= win_rmax(ff / 32) && (even || p.dwaves > WN_WAVES / 2), "units a wave");
#undef REQ
                            }
    // 256 blocks, 10 picks, width 1,024: 36 blocks a row of seven, 40 of six, 80 of three (in eights; in fours 84), 28 of nine
    require(win_work(256, 7, 512, 10, true, 1024, 0).G == 36 && win_work(256, 7, 512, 10, true, 1024, 1).G == 32, "seven rows", 256, 7, 1024, 10, 1, 1);
    require(win_work(256, 6, 512, 10, true, 1024, 1).G == 40 && win_work(256, 6, 512, 10, true, 1024, 2).G == 32, "six rows", 256, 6, 1024, 10, 1, 2);
    require(win_work(256, 3, 512, 10, true, 1024, 1).G == 80 && win_work(256, 3, 512, 10, true, 1024, 2).G == 64, "three rows", 256, 3, 1024, 10, 1, 2);
    require(win_work(256, 3, 512, 10, true, 1024, 0, false).G == 84 && win_work(256, 9, 512, 10, true, 1024, 2).G == 28, "three rows in fours, nine", 256, 3, 1024, 10, 1, 0);
    if (!held || !fours) return std::printf("FAILED: no growth too small, or no blocks in fours\n"), 1;
    std::printf("ok %ld\n", checked);
    return 0;
}
