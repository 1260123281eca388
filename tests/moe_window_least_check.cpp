// Host-side check of the verify window's work for the types that take blocks in fours only where a row gets more of them (win_work's `least` in
// csrc/moe_window_plan.h): over grids, rows, widths and picks it is the deal of the other types or, where the growth is too small, the cut in a
// power of two, whose blocks are walked here as the kernel walks them.
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
    long held = 0;
    for (int nb : {256, 304, 320, 512})
        for (int Tl = 1; Tl <= 16 && WN_WAVES * Tl <= nb; ++Tl)
            for (int ff : {256, 512, 1024})
                for (int topk = 1; topk <= 16; ++topk)
                    for (int shared = 0; shared < 2; ++shared)
                        for (int least : {0, 1, 2}) {
#define REQ(c, what) require(c, what, nb, Tl, ff, topk, shared, least)
                            const WinWork p = win_work(nb, Tl, nexp, topk, shared != 0, ff, least), all = win_work(nb, Tl, nexp, topk, shared != 0, ff);
                            const WinPlan e = win_plan(nb, Tl, nexp, topk, shared != 0, ff);
                            if (all.G == e.G || 8 * (all.G - e.G) > least * e.G) {
                                REQ(std::memcmp(&p, &all, sizeof p) == 0, "the deal of the other types");
                                continue;
                            }
                            ++held;
                            REQ(p.G == e.G && (p.G & (p.G - 1)) == 0 && p.G * Tl <= nb, "a power of two of blocks a row");
                            REQ(p.R == e.R && p.dwaves == e.dwaves && p.upb == e.upb && p.rpb == e.rpb && p.upb * p.G == ff && p.rpb * p.G >= nexp, "units and router rows");
                            std::vector<int> item(p.routed + p.shared, 0);
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
                            }
                            for (int v : item) REQ(v == 1, "every item once");
                            REQ(with == p.nbi, "the h hand-over's count");
#undef REQ
                        }
    // 256 blocks, 10 picks, width 1,024: 36 blocks a row of seven, 40 of six, 80 of three (in eights), 28 of nine
    require(win_work(256, 7, 512, 10, true, 1024, 0).G == 36 && win_work(256, 7, 512, 10, true, 1024, 1).G == 32, "seven rows", 256, 7, 1024, 10, 1, 1);
    require(win_work(256, 6, 512, 10, true, 1024, 1).G == 40 && win_work(256, 6, 512, 10, true, 1024, 2).G == 32, "six rows", 256, 6, 1024, 10, 1, 2);
    require(win_work(256, 3, 512, 10, true, 1024, 1).G == 80 && win_work(256, 3, 512, 10, true, 1024, 2).G == 64, "three rows", 256, 3, 1024, 10, 1, 2);
    require(win_work(256, 9, 512, 10, true, 1024, 2).G == 28, "nine rows", 256, 9, 1024, 10, 1, 2);
    if (!held) return std::printf("FAILED: no growth too small\n"), 1;
    std::printf("ok %ld\n", checked);
    return 0;
}
