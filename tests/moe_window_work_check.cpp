// Host-side check of the verify window's work as its kernel deals it (win_work in csrc/moe_window_plan.h): for every grid size, row count,
// expert width, pick count and expert count the window accepts, walk the blocks as the kernel does and check that every router
// row and every item is taken exactly once, every unit of the down matrices by a wave that stays inside them, that a wave never holds
// more units than its registers allow, and that the h hand-over's count equals the number of blocks that arrive on it. No GPU:
// a count that no block brings up would be a wait that only its time limit ends.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "moe_window_plan.h"

using namespace fnx;

static long checked = 0;
static void require(bool ok, const char* what, int nb, int Tl, int ff, int topk, int nexp, int shared) {
    ++checked;
    if (ok) return;
    std::printf("FAILED %s: blocks %d rows %d ff %d topk %d nexp %d shared %d\n", what, nb, Tl, ff, topk, nexp, shared);
    std::exit(1);
}

int main() {
    const int grids[] = {256, 304, 320, 512}, widths[] = {256, 512, 1024}, experts[] = {1, 8, 60, 64, 100, 512, 1000, 1024};
    long wide = 0;
    for (int nb : grids)
        for (int Tl = 1; Tl <= 16 && WN_WAVES * Tl <= nb; ++Tl)
            for (int ff : widths)
                for (int topk = 1; topk <= 16; ++topk)
                    for (int nexp : experts)
                        for (int shared = 0; shared < 2; ++shared) {
#define REQ(c, what) require(c, what, nb, Tl, ff, topk, nexp, shared)
                            const WinWork p = win_work(nb, Tl, nexp, topk, shared != 0, ff);
                            wide += (p.G & (p.G - 1)) != 0;
                            REQ(p.G >= WN_WAVES && p.G * Tl <= nb, "blocks a row (sixteen at least: they make the rows that do not count)");
                            REQ(p.routed == ff / 32 * topk && p.shared == shared * (ff / 32), "items a row");
                            REQ(p.spb <= 2, "the shared expert's items go ahead of the first block made (two sweeps later)");
                            std::vector<int> item(ff / 32 * (topk + 1), 0), row(nexp, 0), unit(ff, 0);
                            int with_items = 0;
                            for (int g = 0; g < p.G; ++g) {
                                const int s0 = win_shared_first(p, g), left = p.shared - s0 < p.spb ? p.shared - s0 : p.spb, nsh = left > 0 ? left : 0;
                                const int I0 = win_routed_first(p, g), nsweep = nsh + p.ipb + (g < p.more);
                                with_items += nsweep > 0;
                                int j = 0, k = 0;
                                for (int q = 0; q < nsweep; ++q) {
                                    const int I = I0 + q - nsh;
                                    if (q <= nsh) {
                                        j = q < nsh ? s0 + q : I / topk;
                                        k = q < nsh ? 0 : 1 + I - j * topk;
                                    } else if (++k > topk) {   // (the kernel steps through the routed ones)
                                        k = 1;
                                        ++j;
                                    }
                                    REQ(j >= 0 && j < ff / 32 && k >= 0 && k <= topk && (k == 0) == (q < nsh), "an item's block of 32 and matrix");
                                    ++item[j * (topk + 1) + k];
                                }
                                for (int w = 0; w < WN_WAVES; ++w)
                                    for (int r = g * p.rpb + w; r < nexp && r < (g + 1) * p.rpb; r += WN_WAVES) ++row[r];
                                for (int w = 0; w < p.dwaves; ++w) {
                                    const int at = g * p.upb + w * p.R, u0 = at < ff - p.R ? at : ff - p.R;
                                    if (at >= ff) continue;
                                    REQ(u0 >= 0, "a unit inside the matrix");
                                    for (int r = 0; r < p.R; ++r) ++unit[u0 + r];
                                }
                            }
                            for (int i = 0; i < (int) item.size(); ++i) REQ(item[i] == (i % (topk + 1) ? 1 : shared), "every item once");
                            REQ(with_items == p.nbi && p.nbi >= 1 && p.nbi <= p.G, "the h hand-over's count");
                            for (int v : row) REQ(v == 1, "every router row once");
                            REQ(p.R >= 1 && p.R <= win_rmax(ff / 32) && (p.R & (p.R - 1)) == 0 && p.dwaves >= 1 && p.dwaves <= WN_WAVES && p.dwaves * p.R >= p.upb, "units a wave");
                            const bool even = p.dwaves * p.R == p.upb && p.upb * p.G == ff;
                            REQ(even || p.dwaves > WN_WAVES / 2, "waves that share trips have an even cut");
                            for (int v : unit) REQ(even ? v == 1 : v >= 1, "every unit");
#undef REQ
                        }
    if (!wide) return std::printf("FAILED: no cut over all blocks\n"), 1;
    std::printf("ok %ld\n", checked);
    return 0;
}
