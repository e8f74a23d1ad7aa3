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

// rein_xf_*: groups of one and two token tiles, three workgroups per CU
extern "C" __global__ __launch_bounds__(256) void rein_xf_quantize(const float* __restrict__ x, unsigned char* __restrict__ img,
                                                                   BlockQ8* __restrict__ xq, unsigned int in_dim, unsigned int p_rows,
                                                                   unsigned int with_xsum)
{
    rein_xh_quantize_body(x, img, xq, in_dim, p_rows, with_xsum);
}

extern "C" __global__ __launch_bounds__(256) void rein_xf_sum(const float* __restrict__ parts, float* __restrict__ y, unsigned int out_dim,
                                                              unsigned int p_rows, unsigned int n_grp, unsigned int n_whole, unsigned int split)
{
    rein_xh_sum_body(parts, y, out_dim, p_rows, n_grp, n_whole, split);
}

#define REIN_DEFINE_XH(name, FMT, MOST, WAVES)                                                                                  \
    extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES))) void name(                         \
        const unsigned char* __restrict__ w, const unsigned char* __restrict__ img, float* __restrict__ y, float* __restrict__ parts, \
        unsigned int in_dim, unsigned int out_dim, unsigned int p_rows, unsigned int n_grp, unsigned int n_whole, unsigned int split) \
    {                                                                                                                           \
        rein_xh_dense<XhTile<FMT, MOST>>(w, img, y, parts, in_dim, out_dim, p_rows, n_grp, n_whole, split);                      \
    }
REIN_DEFINE_XH(rein_xh_q4k, REIN_Q4_K, 4, 2)
REIN_DEFINE_XH(rein_xh_q5k, REIN_Q5_K, 4, 2)
REIN_DEFINE_XH(rein_xh_q6k, REIN_Q6_K, 4, 2)
REIN_DEFINE_XH(rein_xf_q4k, REIN_Q4_K, 2, 3)
REIN_DEFINE_XH(rein_xf_q5k, REIN_Q5_K, 2, 3)
REIN_DEFINE_XH(rein_xf_q6k, REIN_Q6_K, 2, 3)
