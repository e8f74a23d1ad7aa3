// Entry points of mmq_x8.h, launched by rein_matmul_ws.
#include "mmq_x8.h"

extern "C" __global__ __launch_bounds__(256) void rein_x8_quantize(const float* __restrict__ x, unsigned char* __restrict__ img,
                                                                   BlockQ8* __restrict__ xq, unsigned int in_dim, unsigned int p_rows)
{
    rein_x8_quantize_body(x, img, xq, in_dim, p_rows);
}

extern "C" __global__ __launch_bounds__(256) void rein_x8_sum(const float* __restrict__ parts, float* __restrict__ y, unsigned int out_dim,
                                                              unsigned int p_rows, unsigned int n_grp, unsigned int n_whole, unsigned int split)
{
    rein_xh_sum_body(parts, y, out_dim, p_rows, n_grp, n_whole, split);
}

#define REIN_DEFINE_X8(name, FMT)                                                                                               \
    extern "C" __global__ __launch_bounds__(256) REIN_MMQ_OCC void name(                                                        \
        const unsigned char* __restrict__ w, const unsigned char* __restrict__ img, float* __restrict__ y, float* __restrict__ parts, \
        unsigned int in_dim, unsigned int out_dim, unsigned int p_rows, unsigned int n_grp, unsigned int n_whole, unsigned int split) \
    {                                                                                                                           \
        rein_xh_dense<X8Tile<FMT>>(w, img, y, parts, in_dim, out_dim, p_rows, n_grp, n_whole, split);                                \
    }
REIN_DEFINE_X8(rein_x8_q8_0, REIN_Q8_0)
REIN_DEFINE_X8(rein_x8_q4_0, REIN_Q4_0)
REIN_DEFINE_X8(rein_x8_iq4xs, REIN_IQ4_XS)
REIN_DEFINE_X8(rein_x8_iq3s, REIN_IQ3_S)
