// Several decode matvecs that share their activation rows (one, or the two to four of a speculative-decode
// verify step), in one launch: rein_mv_multi_r<R>_b<B>.
//
// The reference's decode step launches the Q, K and V projections one after the other on the same
// quantized activations, and likewise the gate and up projections of a dense FFN
// (src/runtime/qwen35.rs:2670-2672, 2702-2703, 3612-3614, 3662-3663); on this machine every launch of
// that size costs one to two microseconds of gap and ramp that no kernel can win back.  Here the
// wavefronts of one launch are dealt over up to four matrices: wavefront i belongs to the first
// matrix whose cumulative row-group count exceeds i and runs that matrix's row group exactly as the
// single-matrix kernel rein_mv_<fmt>_r<R>_b<B> does (the same function, the same sums in the same
// order: the outputs are the bits of those kernels).  The matrices may differ in format and in their
// number of rows; they share in_dim and the activation rows.
//
// At two to four activation rows those kernels are bound by the activations: every wavefront reads them from memory again, 40-byte
// records at a 40-byte stride, and with few wavefronts per CU the chain of its trips is what is left.  rein_mvl_multi_r<R>_b<B> (two
// to four rows) and rein_mvql_multi_t4_m (three and four, two matrices of an FFN's size) deal whole workgroups instead, each staging the
// activation rows in LDS and running its matrix as rein_mvl_<fmt> and rein_mvql_<fmt>_t4 would on its workgroups alone: the same
// functions again, so the same bits.  One launch in place of two or three also means that the activations are staged once per CU and
// that the tail of one matrix is covered by the next (us at 4 rows, before / after: Q, K, V 4096 -> 4096 + 2 x 1024 in Q5_K with Q6_K
// 11.6 / 8.9, 1.7 TB/s; gate, up 4096 -> 2 x 14336 in Q5_K 24.0 / 20.6, 4.0 TB/s, 5120 -> 2 x 17408 in Q8_0 41.9 / 31.4, 6.0 TB/s).
#include "matvec_lds.h"
#include "matvec_quad.h"
#include "matvec_repacked.h"

#define REIN_MULTI_MAX 4

struct ReinMultiMat {
    const uint8_t* w;
    float*         y;
    unsigned       out_dim;
    int            fmt;          // REIN_* format id of rein_formats.h
    unsigned       end;          // row groups (workgroups) of this matrix and of those before it
    unsigned       slices;       // rein_mvql_multi_t4_m: of the contraction, and << 16 the trips of weights in flight
};
struct ReinMultiArgs {
    ReinMultiMat m[REIN_MULTI_MAX];
};

template <int R, int B, int POL>
__device__ __forceinline__ void rein_matvec_multi_body(const ReinMultiArgs& a, const BlockQ8* __restrict__ xq,
                                                       unsigned in_dim, unsigned n_mat, unsigned n_rows)
{
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned wid = blockIdx.x * (blockDim.x >> 6) + wave;
    unsigned base = 0, end = a.m[0].end, out_dim = a.m[0].out_dim;
    const uint8_t* w = a.m[0].w;
    float* y = a.m[0].y;
    int fmt = a.m[0].fmt;
#pragma unroll
    for (int i = 1; i < REIN_MULTI_MAX; i++)
        if ((unsigned)i < n_mat && wid >= a.m[i - 1].end) {
            base = a.m[i - 1].end; end = a.m[i].end; out_dim = a.m[i].out_dim;
            w = a.m[i].w; y = a.m[i].y; fmt = a.m[i].fmt;
        }
    if (wid >= end) return;
    const unsigned g = wid - base;
    // one row group per wavefront: first = g, and a step that ends the walk after it
    const unsigned step = 0x40000000u;
    switch (fmt) {
    case REIN_Q4_K:   rein_matvec_span<REIN_Q4_K, R, B, 1, POL>(w, xq, y, in_dim, out_dim, n_rows, g, step); break;
    case REIN_Q6_K:   rein_matvec_span<REIN_Q6_K, R, B, 1, POL>(w, xq, y, in_dim, out_dim, n_rows, g, step); break;
    case REIN_Q5_K:   rein_matvec_span<REIN_Q5_K, R, B, 1, POL>(w, xq, y, in_dim, out_dim, n_rows, g, step); break;
    case REIN_Q8_0:   rein_matvec_span<REIN_Q8_0, R, B, 1, POL>(w, xq, y, in_dim, out_dim, n_rows, g, step); break;
    case REIN_Q4_0:   rein_matvec_span<REIN_Q4_0, R, B, 1, POL>(w, xq, y, in_dim, out_dim, n_rows, g, step); break;
    case REIN_IQ4_XS: rein_matvec_span<REIN_IQ4_XS, R, B, 1, POL>(w, xq, y, in_dim, out_dim, n_rows, g, step); break;
    case REIN_IQ3_S:  rein_matvec_span<REIN_IQ3_S, R, B, 1, POL>(w, xq, y, in_dim, out_dim, n_rows, g, step); break;
    default: break;
    }
}

// name(table, xq[n_rows][in_dim / 32], in_dim, n_mat, n_rows): n_rows <= B; y of matrix i is [n_rows][out_dim i]
// (name_m and name_p: the same with the other loads of the weights, rein_formats.h)
#define REIN_DEFINE_MATVEC_MULTI(name, R, B)                                                                 \
    REIN_DEFINE_MATVEC_MULTI_LD(name, R, B, REIN_LD_STREAM)                                                  \
    REIN_DEFINE_MATVEC_MULTI_LD(name##_m, R, B, REIN_LD_MIX)                                                 \
    REIN_DEFINE_MATVEC_MULTI_LD(name##_p, R, B, REIN_LD_PLAIN)
#define REIN_DEFINE_MATVEC_MULTI_LD(name, R, B, POL)                                                         \
    extern "C" __global__ __launch_bounds__(256) void name(ReinMultiArgs a, const BlockQ8* __restrict__ xq,   \
                                                           unsigned int in_dim, unsigned int n_mat,           \
                                                           unsigned int n_rows)                               \
    {                                                                                                        \
        rein_matvec_multi_body<R, B, POL>(a, xq, in_dim, n_mat, n_rows);                                          \
    }

REIN_DEFINE_MATVEC_MULTI(rein_mv_multi_r1_b1, 1, 1)
REIN_DEFINE_MATVEC_MULTI(rein_mv_multi_r2_b1, 2, 1)
REIN_DEFINE_MATVEC_MULTI(rein_mv_multi_r4_b1, 4, 1)
REIN_DEFINE_MATVEC_MULTI(rein_mv_multi_r1_b2, 1, 2)
REIN_DEFINE_MATVEC_MULTI(rein_mv_multi_r2_b2, 2, 2)
REIN_DEFINE_MATVEC_MULTI(rein_mv_multi_r4_b2, 4, 2)
REIN_DEFINE_MATVEC_MULTI(rein_mv_multi_r1_b4, 1, 4)
REIN_DEFINE_MATVEC_MULTI(rein_mv_multi_r2_b4, 2, 4)
REIN_DEFINE_MATVEC_MULTI(rein_mv_multi_r4_b4, 4, 4)

// run(format as a constant, matrix, workgroup, workgroups of the matrix)
template <int V> struct ReinFmtId { static constexpr int value = V; };
template <class Run>
__device__ __forceinline__ void rein_multi_blocks(const ReinMultiArgs& a, unsigned n_mat, const Run& run)
{
    unsigned base = 0;
    ReinMultiMat m = a.m[0];
#pragma unroll
    for (int i = 1; i < REIN_MULTI_MAX; i++)
        if ((unsigned)i < n_mat && blockIdx.x >= a.m[i - 1].end) {
            base = a.m[i - 1].end;
            m = a.m[i];
        }
    const unsigned block = blockIdx.x - base, n_block = m.end - base;
    switch (m.fmt) {
    case REIN_Q4_K:   run(ReinFmtId<REIN_Q4_K>(), m, block, n_block); break;
    case REIN_Q6_K:   run(ReinFmtId<REIN_Q6_K>(), m, block, n_block); break;
    case REIN_Q5_K:   run(ReinFmtId<REIN_Q5_K>(), m, block, n_block); break;
    case REIN_Q8_0:   run(ReinFmtId<REIN_Q8_0>(), m, block, n_block); break;
    case REIN_Q4_0:   run(ReinFmtId<REIN_Q4_0>(), m, block, n_block); break;
    case REIN_IQ4_XS: run(ReinFmtId<REIN_IQ4_XS>(), m, block, n_block); break;
    case REIN_IQ3_S:  run(ReinFmtId<REIN_IQ3_S>(), m, block, n_block); break;
    default: break;
    }
}
#define REIN_DEFINE_MATVEC_LDS_MULTI(name, R, B)                                                                                  \
    REIN_DEFINE_MATVEC_LDS_MULTI_LD(name, R, B, REIN_LD_STREAM)                                                                   \
    REIN_DEFINE_MATVEC_LDS_MULTI_LD(name##_m, R, B, REIN_LD_MIX)                                                                  \
    REIN_DEFINE_MATVEC_LDS_MULTI_LD(name##_p, R, B, REIN_LD_PLAIN)
#define REIN_DEFINE_MATVEC_LDS_MULTI_LD(name, R, B, POL)                                                                          \
    extern "C" __global__ __launch_bounds__(1024) void name(ReinMultiArgs a, const BlockQ8* __restrict__ xq, unsigned int in_dim, \
                                                            unsigned int n_mat, unsigned int n_rows)                              \
    {                                                                                                                             \
        rein_multi_blocks(a, n_mat, [&](auto fmt, const ReinMultiMat& m, unsigned block, unsigned n_block) {                      \
            rein_matvec_lds_body<decltype(fmt)::value, R, B, POL>(m.w, xq, m.y, in_dim, m.out_dim, n_rows, block, n_block);       \
        });                                                                                                                       \
    }
#define REIN_DEFINE_MATVEC_QUAD_LDS_MULTI_LD(name, POL)                                                                           \
    extern "C" __global__ __launch_bounds__(1024) void name(ReinMultiArgs a, const BlockQ8* __restrict__ xq, unsigned int in_dim, \
                                                            unsigned int n_mat, unsigned int n_rows)                              \
    {                                                                                                                             \
        rein_multi_blocks(a, n_mat, [&](auto fmt, const ReinMultiMat& m, unsigned block, unsigned n_block) {                      \
            rein_matvec_quad_lds_body<decltype(fmt)::value, 1, POL>(m.w, xq, m.y, in_dim, m.out_dim, n_rows, in_dim >> 5,         \
                                                                    m.slices & 0xFFFFu, m.slices >> 16, block, n_block);          \
        });                                                                                                                       \
    }

REIN_DEFINE_MATVEC_LDS_MULTI(rein_mvl_multi_r1_b2, 1, 2)
REIN_DEFINE_MATVEC_LDS_MULTI(rein_mvl_multi_r2_b2, 2, 2)
REIN_DEFINE_MATVEC_LDS_MULTI(rein_mvl_multi_r1_b4, 1, 4)
REIN_DEFINE_MATVEC_LDS_MULTI(rein_mvl_multi_r2_b4, 2, 4)
REIN_DEFINE_MATVEC_QUAD_LDS_MULTI_LD(rein_mvql_multi_t4_m, REIN_LD_MIX)
