// A greedy decode round that the host only enqueues (session.cpp:530-679 drives the same steps from the host and waits
// for each; the reference captures its windows in graphs, engine_common.cu:993-1021, but accepts on the host):
//   verify the window -> accept -> commit -> draft from the rows kept -> prompt lookup -> the next window.
// What one step leaves for the next lives in device words (fnx_round.state), so a round's launches take no argument that
// changes from round to round: rounds can be enqueued back to back, or captured once in a graph and replayed.
//
// A window always has FNX_MAXT rows; state[FNX_RS_ROWS] says how many of them count. The others hold token 0: they
// append their K and V like any row (their cache cells are overwritten by the next window, as a rejected draft's are)
// but ask no queries and are not routed, so they pull no expert's weights, and acceptance never reaches them.
#pragma once

#include "../../include/fnx_mi355x.h"

namespace fnx {

// after the verify (session.cpp:565-573, 616-640): n = 1 + the drafts that equal the row before's pick; the picks of the
// rows kept join the context; the positions move on by n. One wave.
// A round whose next window would not fit the caches (max_ctx) or the context buffer raises FNX_RS_STOP and changes
// nothing; every later round then finds the same state and repeats the same work. So does the first round of a badly
// placed session (a position below zero, or a window that does not fit to begin with: the verify before this computed
// over the cells that exist and is not kept).
__global__ void k_round_commit(const int* __restrict__ rows, const int* __restrict__ best, int* __restrict__ state, int* __restrict__ ctx,
                               int ctx_cap, int max_ctx, int* __restrict__ log, int log_cap) {
    const int i = threadIdx.x;
    const int R = min(max(state[FNX_RS_ROWS], 1), FNX_MAXT), n_ctx = state[FNX_RS_NCTX], pos = state[FNX_RS_POS], rounds = state[FNX_RS_ROUNDS];
    const int stop = state[FNX_RS_STOP];
    const bool ok = i + 1 < R && rows[i + 1] == best[i];
    const int n = 1 + (int) __builtin_ctzll(~__ballot(ok));
    const int pick = i < n ? best[i] : 0;
    if (stop || pos < 0 || pos + n + FNX_MAXT > max_ctx || n_ctx + n + FNX_MAXT > ctx_cap) {
        if (i == 0) state[FNX_RS_STOP] = 1;
        return;
    }
    if (i < n) ctx[n_ctx + i] = pick;
    if (i == 0) {
        state[FNX_RS_NCTX] = n_ctx + n;
        state[FNX_RS_POS] = pos + n;
        state[FNX_RS_POS_PREV] = pos;
        state[FNX_RS_ACCEPTED] = n;
        state[FNX_RS_ROUNDS] = rounds + 1;
        if (log && rounds < log_cap) {
            log[2 * rounds] = R - 1;
            log[2 * rounds + 1] = n;
        }
    }
}

// The MTP chain (session.cpp:666-678) has no launches of its own but its steps': it begins in the lookup's, and a step's pick is
// kept by the step's argmax, the last one's making the next window too. A launch that does no more than move a word takes 4.5 us
// between others (eight rounds with a chain of three drafts: 6,929 -> 6,860 us for the four launches less a round).
//
// It starts when the lookup found nothing: its first draft is the draft layer's pick for the last row kept, its source that
// row of the draft layer's output. The steps' positions are written in any case (a step that does not count still appends
// its row to the draft layer's cache, in cells that the next round's pass over the rows kept writes again before
// anything reads them).
struct ChainBegin {
    int *state, *scratch;
    const float* hidden;             // the draft layer's output rows
    float* src;                      // the row kept last goes here
    int n;                           // values a row, 4,096 at most
};
// after step j (1 .. K - 1): its pick is draft j + 1; the last step hands the K drafts to the next window
struct ChainKeep {
    int *state, *scratch;
    const int* ctx;
    int* rows;                       // the next window, made after the last step
    int j, K;
};

// the next window without speculation (session.cpp:530-560): the last token of the context alone. One wave. (With it
// the window is that token, then the drafts: with a single draft a round the lookup's launch makes it, of what it found or else the
// draft layer's pick for the last row kept; with a chain the chain's last step, of what the lookup found or else the chain's drafts.)
__global__ void k_round_window(const int* __restrict__ ctx, int* __restrict__ state, int* __restrict__ rows) {
    const int i = threadIdx.x;
    if (state[FNX_RS_STOP]) return;
    if (i < FNX_MAXT) rows[i] = i == 0 ? ctx[state[FNX_RS_NCTX] - 1] : 0;
    if (i == 0) state[FNX_RS_ROWS] = 1;
}

}  // namespace fnx
