// Entry points of mmq_exact16.h, launched by rein_matmul_ws.
#include "mmq_exact16.h"

extern "C" __global__ __launch_bounds__(256) void rein_xh_quantize(const float* __restrict__ x, unsigned char* __restrict__ img,
                                                                   BlockQ8* __restrict__ xq, unsigned int in_dim, unsigned int p_rows,
                                                                   unsigned int with_xsum)
{
    rein_xh_quantize_body(x, img, xq, in_dim, p_rows, with_xsum);
}

extern "C" __global__ __launch_bounds__(256) void rein_xh_sum(const float* __restrict__ parts, float* __restrict__ y, unsigned int out_dim,
                                                              unsigned int p_rows, unsigned int n_grp, unsigned int n_whole, unsigned int split)
{
    rein_xh_sum_body(parts, y, out_dim, p_rows, n_grp, n_whole, split);
}

#define REIN_DEFINE_XH(name, FMT)                                                                                               \
    extern "C" __global__ __launch_bounds__(256) REIN_MMQ_OCC void name(                                                        \
        const unsigned char* __restrict__ w, const unsigned char* __restrict__ img, float* __restrict__ y, float* __restrict__ parts, \
        unsigned int in_dim, unsigned int out_dim, unsigned int p_rows, unsigned int n_grp, unsigned int n_whole, unsigned int split) \
    {                                                                                                                           \
        rein_xh_dense<XhTile<FMT>>(w, img, y, parts, in_dim, out_dim, p_rows, n_grp, n_whole, split);                                        \
    }
REIN_DEFINE_XH(rein_xh_q4k, REIN_Q4_K)
REIN_DEFINE_XH(rein_xh_q5k, REIN_Q5_K)
REIN_DEFINE_XH(rein_xh_q6k, REIN_Q6_K)
