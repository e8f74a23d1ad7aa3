// Entry points of moe_wide.h, launched by rein_moe_ffn.
#include "moe_wide.h"

#define REIN_DEFINE_XG_GATHER(name, X8)                                                                                       \
    extern "C" __global__ __launch_bounds__(256) void name(                                                                     \
        const BlockQ8* __restrict__ xq, const int* __restrict__ perm, const int* __restrict__ place, const int* __restrict__ n_sorted, \
        unsigned char* __restrict__ img, unsigned int in_dim, unsigned int n_used, unsigned int n_entries, unsigned int n_tt,   \
        unsigned int with_xsum)                                                                                                 \
    {                                                                                                                           \
        rein_xg_gather<X8>(xq, perm, place, n_sorted, img, in_dim, n_used, n_entries, n_tt, with_xsum);                         \
    }
REIN_DEFINE_XG_GATHER(rein_moe_gather_xh, false)
REIN_DEFINE_XG_GATHER(rein_moe_gather_x8, true)

#define REIN_DEFINE_XG(tag, TILE, WAVES)                                                                                        \
    extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES))) void rein_mmq_##tag##_swiglu(      \
        const unsigned char* __restrict__ gate, const unsigned char* __restrict__ up, unsigned int bytes_per_expert,            \
        const ReinMoeUnit* __restrict__ units, unsigned int per_xcd, const unsigned char* __restrict__ img,                     \
        unsigned char* __restrict__ out, unsigned int in_dim, unsigned int out_dim, unsigned int n_tt, unsigned int out_kind)                      \
    {                                                                                                                           \
        rein_xg_swiglu<TILE>(gate, up, bytes_per_expert, units, per_xcd, img, out, in_dim, out_dim, n_tt, out_kind); \
    }                                                                                                                           \
    extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES))) void rein_mmq_##tag##_rows(        \
        const unsigned char* __restrict__ slab, unsigned int bytes_per_expert, const ReinMoeUnit* __restrict__ units,           \
        unsigned int per_xcd, const unsigned char* __restrict__ img, float* __restrict__ y, unsigned int in_dim, unsigned int out_dim, unsigned int n_tt)  \
    {                                                                                                                           \
        rein_xg_rows<TILE>(slab, bytes_per_expert, units, per_xcd, img, y, in_dim, out_dim, n_tt);             \
    }
typedef XhTile<REIN_Q4_K, 2> XgQ4; typedef XhTile<REIN_Q5_K, 2> XgQ5; typedef XhTile<REIN_Q6_K, 2> XgQ6;
REIN_DEFINE_XG(q4k_xg2, XgQ4, 3)
REIN_DEFINE_XG(q5k_xg2, XgQ5, 3)
REIN_DEFINE_XG(q6k_xg2, XgQ6, 3)
REIN_DEFINE_XG(q8_0_xg4, X8Tile<REIN_Q8_0>, 2)
