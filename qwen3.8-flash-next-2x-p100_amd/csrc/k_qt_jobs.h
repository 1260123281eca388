// Jobs over the other expert types (k_qtypes.h), operator by operator.
#pragma once

#include "k_qtypes.h"

namespace fnx {

struct QtArgs {
    const uint8_t* wbase;
    size_t w_stride;
    const uint8_t* const* ep;
    size_t row_bytes;
    int nrows, ncols;
    const fnx_job* jobs;
    const int* njobs;
    int njobs_max;
    const uint8_t* y;
    float* out;
    int out_stride;
};
template <uint32_t TYPE>
__global__ void __launch_bounds__(256) k_qt_jobs(const QtArgs a) {
    const int ji = blockIdx.y;
    if (ji >= (a.njobs ? min(*a.njobs, a.njobs_max) : a.njobs_max)) return;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= a.nrows) return;
    const fnx_job* jb = a.jobs + ji;
    const uint8_t* we = (a.ep ? a.ep[jb->w] : a.wbase + (size_t) jb->w * a.w_stride) + (size_t) row * a.row_bytes;
    const int sbr = a.ncols / 32, n = min(max(jb->n, 0), FNX_MAXT);
    const uint8_t* y = a.y ? a.y : g_moe_hq;   // moe_down: the pairs' q8_1 rows in the library's buffer
    for (int t = 0; t < n; ++t) {
        float acc = 0.f;
        for (int kb = lane; kb < sbr; kb += 64) {
            const QtSub s = qt_decode<TYPE>(we, kb);
            acc += qt_term<TYPE>(s, y + ((size_t) jb->y[t] * sbr + kb) * FNX_Q8_1_BLOCK);
        }
        acc = group_sum<64>(acc);
        if (lane == 0) a.out[(size_t) jb->out[t] * a.out_stride + row] = acc;
    }
}

}  // namespace fnx
