// The one-launch verify window (k_moe_window.h) over the expert types other than IQ3_S: a translation unit of its own, since
// it is a kernel per type and expert width.
#include "k_moe_window.h"

namespace fnx {

template <uint32_t TYPE>
static void launch_type(const WindowArgs& a, int blocks, hipStream_t s) {
    if (a.ff == 256) k_moe_window<8, false, 2, WinQt<TYPE>><<<blocks, WN_THREADS, 0, s>>>(a);
    else if (a.ff == 512) k_moe_window<16, false, 2, WinQt<TYPE>><<<blocks, WN_THREADS, 0, s>>>(a);
    else k_moe_window<32, false, 2, WinQt<TYPE>><<<blocks, WN_THREADS, 0, s>>>(a);
}
// type: one of window_takes_type()'s; ff 256, 512 or 1024
void window_launch_type(uint32_t type, const WindowArgs& a, int blocks, hipStream_t s) {
    switch (type) {
        case QT_Q4_0: return launch_type<QT_Q4_0>(a, blocks, s);
        case QT_Q5_1: return launch_type<QT_Q5_1>(a, blocks, s);
        case QT_Q8_0: return launch_type<QT_Q8_0>(a, blocks, s);
        case QT_IQ4_NL: return launch_type<QT_IQ4_NL>(a, blocks, s);
        case QT_IQ4_XS: return launch_type<QT_IQ4_XS>(a, blocks, s);
        case QT_Q4_K: return launch_type<QT_Q4_K>(a, blocks, s);
        default: return launch_type<QT_Q5_K>(a, blocks, s);
    }
}

}  // namespace fnx
