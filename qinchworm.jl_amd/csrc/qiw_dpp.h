// qiw_dpp.h -- multiply-adds whose factor is broadcast from one lane of each row of 16.
#pragma once
#include <hip/hip_runtime.h>

// c[0 .. 3] += (elements N .. N + 3 of the 16 in a) * y, and for two and one.  The wait states
// between a vector write of a and a DPP read of it stand in the block.  Its accumulators are written
// before the last read of a and y: early clobbers, so that none shares their registers.
template <int N, int R>
__device__ __forceinline__ void fmac_bcast(double *c, double a, double y) {
    if constexpr (R >= 4) {
        asm("s_nop 1\n"
            "v_fmac_f64_dpp %0, %4, %5 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n"
            "v_fmac_f64_dpp %1, %4, %5 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n"
            "v_fmac_f64_dpp %2, %4, %5 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n"
            "v_fmac_f64_dpp %3, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
            : "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3])
            : "v"(a), "v"(y), "n"(N), "n"(N + 1), "n"(N + 2), "n"(N + 3));
    } else if constexpr (R == 2) {
        asm("s_nop 1\n"
            "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n"
            "v_fmac_f64_dpp %1, %2, %3 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n"
            : "+&v"(c[0]), "+&v"(c[1])
            : "v"(a), "v"(y), "n"(N), "n"(N + 1));
    } else {
        asm("s_nop 1\n"
            "v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n"
            : "+v"(c[0])
            : "v"(a), "v"(y), "n"(N));
    }
}
