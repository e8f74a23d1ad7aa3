// The routed experts' FFN for a small batch of tokens: gate + up + SwiGLU + quantize, and down, each reading every expert that
// the router touched ONCE for all of its tokens.
//
// Between the decode launches (moe_matvec.hip), which read an expert once per routing entry, and the grouped GEMM
// (mmq_gemm.h), whose 32-token tiles cost their full matrix work however few tokens an expert got: at 48 tokens x top-8
// of 128 experts an expert has three entries on average, the tiles took 133 us for 384 MB of experts (2.9 TB/s), and what they
// waited on was their own instructions.  Here a workgroup of four wavefronts owns an expert and a run of its rows.  It finds
// the expert's entries by scanning the router's ids (a few KB: no sort, no gather), stages their activations in LDS, up to
// eight at a time, and streams its rows past them: a lane owns 64 weights (FmtPair) of each of two rows -- gate and up of one column, or two
// rows of down -- so that a fetch from LDS serves both, dot4 against every entry, one unpack for all of them.  The first
// weights are requested before the scan: they depend on the expert alone.  G lanes share a row (16, or 4 for contractions
// that are not a multiple of 1024 values: 768 is three trips of 4 lanes without an idle one).
//
// grid = (runs of rows, n_expert), block = 64 * kGuWaves / kDownWaves; dynamic LDS = 8 * kParts * 16 * n_pad bytes, n_pad = in_dim / 64 in
// whole trips of G.  Contractions are a multiple of 64; ids [n_entries], at most 65535, as the router wrote them, entry e = token
// e / n_used; at most kMaxEntries of one expert (the router picks an expert at most once per token).  An expert without
// entries ends at once.
//
// Measured (us, gate + up / down of 128 experts top-8, 2048 x 768, Q4_K / Q6_K, against the tiles' 74 / 57 at any of these counts):
// 24 tokens 43 / 37, 48 tokens 53 / 44, 96 tokens 74 / 59; the whole FFN at 16 / 32 / 48 / 64 / 96 tokens 77 / 93 / 106 / 121 / 150 against
// 87 / 142 / 149 / 150 / 152.  What bounds it: at one entry per expert the chain of requests of short-lived workgroups (3.5-4.5 TB/s),
// from about four the dot4 and scale instructions, 13 per sub-block and entry.  Tried without gain: 8 or 16 wavefronts to a
// workgroup (31.7 against 24.7 us for gate + up at 8 tokens), two trips in flight per wavefront instead of
// one (38.3 against 32.7 then), runs of 32 or 128 columns.
#include "matvec_pair.h"
#include "q8_block.h"

namespace rein_few {

constexpr unsigned kBatch = 8;              // entries whose activations are in LDS at a time
constexpr unsigned kMaxEntries = 1024;
constexpr unsigned kGuCols = 64, kGuWaves = 4, kDownRows = 128, kDownWaves = 2;      // of a workgroup

// A staged entry: parts of n_pad 16-byte words, one word per pair of sub-blocks (padded with zeros to whole trips of G lanes): the quants
// 0-15 and 16-31 of the first sub-block, of the second, then {d, d, xsum, xsum}; Q6_K has {-32 * sum} of the four 16-quant halves there
// (the accumulators of its dots start from them) and {d, d} in a part of its own.
template <int FMT> constexpr unsigned kParts = FMT == REIN_Q6_K ? 6 : 5;

template <int FMT>
__device__ __forceinline__ void stage(uint4* x, unsigned n_pad, unsigned sb, const BlockQ8& v)
{
    const unsigned u = sb >> 1, o = sb & 1u;
    x[2 * o * n_pad + u] = make_uint4(v.qs[0], v.qs[1], v.qs[2], v.qs[3]);
    x[(2 * o + 1) * n_pad + u] = make_uint4(v.qs[4], v.qs[5], v.qs[6], v.qs[7]);
    if constexpr (FMT == REIN_Q6_K) {
        int q[8];
#pragma unroll
        for (int k = 0; k < 8; k++) q[k] = v.qs[k];
        const XSums xs = rein_xsums(q);
        reinterpret_cast<int2*>(&x[4 * n_pad + u])[o] = make_int2(-32 * xs.lo, -32 * xs.hi);
        reinterpret_cast<float*>(&x[5 * n_pad])[2 * u + o] = v.d;
    } else {
        float* h = reinterpret_cast<float*>(&x[4 * n_pad + u]);
        h[o] = v.d;
        h[2 + o] = v.xsum;
    }
}

template <int G> __device__ __forceinline__ float group_sum(float v)
{
    if constexpr (G == 16) return rein_row16_sum(v);
    v += rein_dpp_f32<0xB1>(0.0f, v);
    v += rein_dpp_f32<0x4E>(0.0f, v);
    if constexpr (G == 8) v += rein_dpp_f32<0x141>(0.0f, v);
    return v;
}

// A wavefront's rows: `rows(pass, lr, ra, rb)` says which row of wa and of wb the lane group lr works on in a pass.
// done(pass, lr, b, sum_a, sum_b) gets the sums of entry b, each on a lane of its own: lane b % G of the group.
template <int FMT, int G> struct Stream {
    using Planes = PairPlanes<FMT>;
    using Pair = FmtPair<FMT>[2];
    Pair cur;
    template <class Rows>
    static __device__ __forceinline__ void request(const Planes& wa, const Planes& wb, unsigned n_unit, unsigned pass, unsigned t,
                                                   const Rows& rows, Pair& v)
    {
        const unsigned lane = threadIdx.x & 63u, u = min((lane & (G - 1u)) + G * t, n_unit - 1);
        unsigned ra, rb;
        rows(pass, lane / G, ra, rb);
        v[0].load(wa, wa.at(ra, u), wa.super(ra, u));
        v[1].load(wb, wb.at(rb, u), wb.super(rb, u));
    }
    template <int B>
    static __device__ __forceinline__ void multiply(const Pair& v, const uint4* lds, unsigned at, unsigned n_pad, float (&acc)[2][B])
    {
        constexpr bool q6 = FMT == REIN_Q6_K, mins = !q6 && FMT != REIN_Q8_0;
        int w[2][2][8], sc[2][2][2];
        float s0[2][2], s1[2][2];
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int o = 0; o < 2; o++) {
                SubW sw;
                const auto raw = v[r].get(o);
                Fmt<FMT>::unpack(raw, sw);
#pragma unroll
                for (int k = 0; k < 8; k++) w[r][o][k] = sw.w[k];
                s0[r][o] = sw.s0;
                s1[r][o] = sw.s1;
                if constexpr (q6) {
                    sc[r][o][0] = (int)(int8_t)(raw.sm & 0xFFu);
                    sc[r][o][1] = (int)(int8_t)(raw.sm >> 8);
                    s0[r][o] = rein_h2f(raw.d);
                }
            }
        const uint4* x = lds + at;
#pragma unroll
        for (int b = 0; b < B; b++, x += kParts<FMT> * n_pad) {
            const uint4 hd = x[4 * n_pad];
            float2 d2;
            if constexpr (q6) d2 = reinterpret_cast<const float2*>(&x[5 * n_pad - at])[at];
            else d2 = make_float2(__builtin_bit_cast(float, hd.x), __builtin_bit_cast(float, hd.y));
#pragma unroll
            for (int o = 0; o < 2; o++) {
                const uint4 x0 = x[2 * o * n_pad], x1 = x[(2 * o + 1) * n_pad];
                const int q[8] = {(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w, (int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w};
                const float dx = o ? d2.y : d2.x;
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    int i0 = q6 ? (int)(o ? hd.z : hd.x) : 0, i1 = q6 ? (int)(o ? hd.w : hd.y) : 0;
#pragma unroll
                    for (int k = 0; k < 4; k++) i0 = rein_dot4(w[r][o][k], q[k], i0);
#pragma unroll
                    for (int k = 4; k < 8; k++) {
                        if constexpr (q6) i1 = rein_dot4(w[r][o][k], q[k], i1);
                        else i0 = rein_dot4(w[r][o][k], q[k], i0);
                    }
                    // (Q6_K: two scaled dots of 16, each below 2^23, added as whole numbers)
                    if constexpr (q6) i0 = __mul24(i0, sc[r][o][0]) + __mul24(i1, sc[r][o][1]);
                    acc[r][b] = fmaf(s0[r][o] * dx, (float)i0, acc[r][b]);
                    if constexpr (mins) acc[r][b] = fmaf(-s1[r][o], __builtin_bit_cast(float, o ? hd.w : hd.z), acc[r][b]);
                }
            }
        }
    }
    template <int B, class Rows, class Done>
    __device__ __forceinline__ void run(const Planes& wa, const Planes& wb, const uint4* lds, unsigned n_unit, unsigned n_pad, unsigned n_pass,
                                        const Rows& rows, const Done& done)
    {
        const unsigned lane = threadIdx.x & 63u, l = lane & (G - 1u), lr = lane / G;
        const unsigned trips = n_pad / G;
        float acc[2][B];
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int b = 0; b < B; b++) acc[r][b] = 0.0f;
        unsigned pass = 0, t = 0;
        // one trip on `now` while the next one's weights come into `next`
        const auto step = [&](Pair& now, Pair& next) {
            const bool last = t + 1 == trips;
            const unsigned pass2 = last ? pass + 1 : pass, t2 = last ? 0 : t + 1;
            request(wa, wb, n_unit, min(pass2, n_pass - 1), t2, rows, next);
            multiply<B>(now, lds, l + G * t, n_pad, acc);
            if (last) {
                constexpr int kEach = (B + G - 1) / G;
                float sa[kEach] = {}, sb[kEach] = {};
#pragma unroll
                for (int b = 0; b < B; b++) {
                    const float va = group_sum<G>(acc[0][b]), vb = group_sum<G>(acc[1][b]);
                    sa[b / G] = l == (unsigned)b % G ? va : sa[b / G];
                    sb[b / G] = l == (unsigned)b % G ? vb : sb[b / G];
                    acc[0][b] = acc[1][b] = 0.0f;
                }
#pragma unroll
                for (int i = 0; i < kEach; i++)
                    if (l + i * G < (unsigned)B) done(pass, lr, l + i * G, sa[i], sb[i]);
            }
            pass = pass2;
            t = t2;
        };
        Pair nxt;
        for (;;) {
            step(cur, nxt);
            if (pass == n_pass) break;
            step(nxt, cur);
            if (pass == n_pass) break;
        }
    }
    // the loops are compiled for 1, 2, 3, 4, 6 and 8 entries: what lies in LDS behind the nb-th is computed and dropped
    template <class Rows, class Done>
    __device__ __forceinline__ void run_some(unsigned nb, const Planes& wa, const Planes& wb, const uint4* lds, unsigned n_unit, unsigned n_pad,
                                             unsigned n_pass, const Rows& rows, const Done& done)
    {
        if (nb > 6) run<8>(wa, wb, lds, n_unit, n_pad, n_pass, rows, done);
        else if (nb > 4) run<6>(wa, wb, lds, n_unit, n_pad, n_pass, rows, done);
        else if (nb == 4) run<4>(wa, wb, lds, n_unit, n_pad, n_pass, rows, done);
        else if (nb == 3) run<3>(wa, wb, lds, n_unit, n_pad, n_pass, rows, done);
        else if (nb == 2) run<2>(wa, wb, lds, n_unit, n_pad, n_pass, rows, done);
        else run<1>(wa, wb, lds, n_unit, n_pad, n_pass, rows, done);
    }
};

// the entries of expert e, in any order (each entry's result does not depend on it)
__device__ __forceinline__ unsigned find_entries(const int* __restrict__ ids, unsigned n_entries, unsigned e, uint16_t* list, unsigned* count)
{
    if (threadIdx.x == 0) *count = 0;
    __syncthreads();
    for (unsigned i = threadIdx.x; i < n_entries; i += blockDim.x)
        if (ids[i] == (int)e) {
            const unsigned at = atomicAdd(count, 1u);
            if (at < kMaxEntries) list[at] = (uint16_t)i;
        }
    __syncthreads();
    return min(*count, kMaxEntries);
}

template <int FMT, int G>
__device__ __forceinline__ void gate_up(const uint8_t* __restrict__ gate_slab, const uint8_t* __restrict__ up_slab, unsigned bytes_per_expert,
                                        const int* __restrict__ ids, const BlockQ8* __restrict__ xq, BlockQ8* __restrict__ xq_out,
                                        unsigned in_dim, unsigned out_dim, unsigned n_used, unsigned n_entries)
{
    extern __shared__ uint4 rein_few_lds[];
    __shared__ uint16_t list[kMaxEntries];
    __shared__ unsigned count;
    __shared__ float vals[kBatch][kGuCols + 4];
    const unsigned e = blockIdx.y, c0 = blockIdx.x * kGuCols;
    const unsigned n_sub = in_dim >> 5, n_unit = n_sub >> 1, n_pad = (n_unit + G - 1) / G * G, wave = threadIdx.x >> 6;
    constexpr unsigned kRows = 64 / G, kStep = kGuWaves * kRows;                   // columns of a wavefront, of the workgroup, per pass
    const unsigned n_pass = min(kGuCols / kStep, (out_dim - c0 + kStep - 1) / kStep);
    const PairPlanes<FMT> wg(gate_slab + (size_t)e * bytes_per_expert, n_sub, out_dim), wu(up_slab + (size_t)e * bytes_per_expert, n_sub, out_dim);
    const auto rows = [&](unsigned pass, unsigned lr, unsigned& ra, unsigned& rb) {
        ra = rb = min(c0 + pass * kStep + wave * kRows + lr, out_dim - 1);
    };
    Stream<FMT, G> s;
    s.request(wg, wu, n_unit, 0, 0, rows, s.cur);
    const unsigned m = find_entries(ids, n_entries, e, list, &count);
    for (unsigned at = 0; at < m; at += kBatch) {
        const unsigned nb = min(kBatch, m - at);
        if (at) s.request(wg, wu, n_unit, 0, 0, rows, s.cur);
        if (n_pad > n_unit && at == 0)
            for (unsigned i = threadIdx.x; i < kBatch * kParts<FMT> * n_pad; i += blockDim.x) rein_few_lds[i] = make_uint4(0, 0, 0, 0);
        if (n_pad > n_unit && at == 0) __syncthreads();
        for (unsigned i = threadIdx.x; i < nb * n_sub; i += blockDim.x) {
            const unsigned b = i / n_sub, sb = i - b * n_sub;
            stage<FMT>(rein_few_lds + b * kParts<FMT> * n_pad, n_pad, sb, xq[(size_t)(list[at + b] / n_used) * n_sub + sb]);
        }
        __syncthreads();
        s.run_some(nb, wg, wu, rein_few_lds, n_unit, n_pad, n_pass, rows, [&](unsigned pass, unsigned lr, unsigned b, float g, float u) {
            vals[b][pass * kStep + wave * kRows + lr] = rein_silu_det(g) * u;
        });
        __syncthreads();
        const unsigned l = threadIdx.x & 15u;
        for (unsigned i = threadIdx.x >> 4; i < nb * (kGuCols / 32); i += blockDim.x >> 4) {
            const unsigned b = i / (kGuCols / 32), h = i % (kGuCols / 32);
            if (c0 + 32 * h < out_dim)
                rein_q8_store_sub(xq_out + (size_t)list[at + b] * (out_dim >> 5) + (c0 >> 5) + h, l, vals[b][32 * h + l], vals[b][32 * h + l + 16]);
        }
    }
}

template <int FMT, int G>
__device__ __forceinline__ void down(const uint8_t* __restrict__ slab, unsigned bytes_per_expert, const int* __restrict__ ids,
                                     const BlockQ8* __restrict__ xq, float* __restrict__ y, unsigned in_dim, unsigned out_dim, unsigned n_entries)
{
    extern __shared__ uint4 rein_few_lds[];
    __shared__ uint16_t list[kMaxEntries];
    __shared__ unsigned count;
    const unsigned e = blockIdx.y, r0 = blockIdx.x * kDownRows;
    const unsigned n_sub = in_dim >> 5, n_unit = n_sub >> 1, n_pad = (n_unit + G - 1) / G * G, wave = threadIdx.x >> 6;
    constexpr unsigned kRows = 64 / G, kStep = 2 * kDownWaves * kRows;                   // two rows per lane group
    const unsigned n_pass = min(kDownRows / kStep, (out_dim - r0 + kStep - 1) / kStep);
    const PairPlanes<FMT> w(slab + (size_t)e * bytes_per_expert, n_sub, out_dim);
    const auto first = [&](unsigned pass, unsigned lr) { return r0 + pass * kStep + wave * 2 * kRows + lr; };
    const auto rows = [&](unsigned pass, unsigned lr, unsigned& ra, unsigned& rb) {
        ra = min(first(pass, lr), out_dim - 1);
        rb = min(first(pass, lr) + kRows, out_dim - 1);
    };
    Stream<FMT, G> s;
    s.request(w, w, n_unit, 0, 0, rows, s.cur);
    const unsigned m = find_entries(ids, n_entries, e, list, &count);
    for (unsigned at = 0; at < m; at += kBatch) {
        const unsigned nb = min(kBatch, m - at);
        if (at) {
            __syncthreads();
            s.request(w, w, n_unit, 0, 0, rows, s.cur);
        }
        if (n_pad > n_unit && at == 0)
            for (unsigned i = threadIdx.x; i < kBatch * kParts<FMT> * n_pad; i += blockDim.x) rein_few_lds[i] = make_uint4(0, 0, 0, 0);
        if (n_pad > n_unit && at == 0) __syncthreads();
        for (unsigned i = threadIdx.x; i < nb * n_sub; i += blockDim.x) {
            const unsigned b = i / n_sub, sb = i - b * n_sub;
            stage<FMT>(rein_few_lds + b * kParts<FMT> * n_pad, n_pad, sb, xq[(size_t)list[at + b] * n_sub + sb]);
        }
        __syncthreads();
        s.run_some(nb, w, w, rein_few_lds, n_unit, n_pad, n_pass, rows, [&](unsigned pass, unsigned lr, unsigned b, float va, float vb) {
            if (b >= nb) return;
            float* o = y + (size_t)list[at + b] * out_dim;
            const unsigned ra = first(pass, lr), rb = ra + kRows;
            if (ra < out_dim) o[ra] = va;
            if (rb < out_dim) o[rb] = vb;
        });
    }
}

}  // namespace rein_few

#define REIN_DEFINE_MOE_FEW(tag, FMT, G)                                                                                     \
    extern "C" __global__ __launch_bounds__(64 * rein_few::kGuWaves, 2) void rein_moe_few_gate_up_##tag##_g##G(              \
        const unsigned char* __restrict__ gate_slab, const unsigned char* __restrict__ up_slab, const int* __restrict__ ids, \
        const BlockQ8* __restrict__ xq, BlockQ8* __restrict__ xq_out, unsigned int bytes_per_expert, unsigned int in_dim,    \
        unsigned int out_dim, unsigned int n_used, unsigned int n_entries)                                                   \
    {                                                                                                                        \
        rein_few::gate_up<FMT, G>(gate_slab, up_slab, bytes_per_expert, ids, xq, xq_out, in_dim, out_dim, n_used, n_entries); \
    }                                                                                                                        \
    extern "C" __global__ __launch_bounds__(64 * rein_few::kDownWaves, 2) void rein_moe_few_down_##tag##_g##G(               \
        const unsigned char* __restrict__ slab, const int* __restrict__ ids, const BlockQ8* __restrict__ xq,                 \
        float* __restrict__ y, unsigned int bytes_per_expert, unsigned int in_dim, unsigned int out_dim,                     \
        unsigned int n_entries)                                                                                              \
    {                                                                                                                        \
        rein_few::down<FMT, G>(slab, bytes_per_expert, ids, xq, y, in_dim, out_dim, n_entries);                              \
    }
#define REIN_DEFINE_MOE_FEW_G(tag, FMT) REIN_DEFINE_MOE_FEW(tag, FMT, 16) REIN_DEFINE_MOE_FEW(tag, FMT, 8) REIN_DEFINE_MOE_FEW(tag, FMT, 4)
REIN_DEFINE_MOE_FEW_G(q4k, REIN_Q4_K)
REIN_DEFINE_MOE_FEW_G(q5k, REIN_Q5_K)
REIN_DEFINE_MOE_FEW_G(q6k, REIN_Q6_K)
REIN_DEFINE_MOE_FEW_G(q8_0, REIN_Q8_0)
REIN_DEFINE_MOE_FEW_G(q5_1, REIN_Q5_1)
