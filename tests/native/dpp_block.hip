// Accumulators that hold the same value as a factor that is not needed afterwards: the compiler
// then has a reason to give them one register (tests/test_dpp_block.py).
#include "qiw_dpp.h"

template <int R>
__global__ void k_same_as_y(double *out, const double *in) {
    const double a = in[threadIdx.x], y = in[threadIdx.x + 64];
    double c[4] = {y, y, y, y};
    fmac_bcast<0, R>(c, a, y);
    for (int i = 0; i < R; ++i) out[threadIdx.x + 64 * i] = c[i];
}
template <int R>
__global__ void k_same_as_a(double *out, const double *in) {
    const double a = in[threadIdx.x], y = in[threadIdx.x + 64];
    double c[4] = {a, a, a, a};
    fmac_bcast<4, R>(c, a, y);
    for (int i = 0; i < R; ++i) out[threadIdx.x + 64 * i] = c[i];
}
#define BOTH(R)                                                  \
    template __global__ void k_same_as_y<R>(double *, const double *); \
    template __global__ void k_same_as_a<R>(double *, const double *);
BOTH(4)
BOTH(2)
BOTH(1)
