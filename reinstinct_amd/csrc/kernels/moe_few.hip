// The routed experts' FFN for a small batch of tokens: gate + up + SwiGLU + quantize, and down, each reading every expert that
// the router touched ONCE for all of its tokens.
//
// Between the decode launches (moe_matvec.hip), which read an expert once per routing entry, and the grouped GEMM
// (mmq_gemm.h), whose 32-token tiles cost their full matrix work however few tokens an expert got: at 48 tokens x top-8
// of 128 experts an expert has three entries on average, the tiles took 133 us for 384 MB of experts (2.9 TB/s), and what they
// waited on was their own instructions.  Here a workgroup of four wavefronts owns an expert and a run of its rows.  It finds
// the expert's entries by scanning the router's ids (a few KB: no sort, no gather), stages their activations in LDS, up to
// eight at a time, and streams its rows past them: a lane owns 64 weights (FmtPair) of each of two rows -- gate and up of one column, or two
// rows of down -- so that a fetch from LDS serves both, one unpack for all entries.  One or two entries go on dot4; three to eight on
// v_mfma_i32_4x4x4_16b_i8, four rows of a unit (two sub-blocks) to a quad of lanes against four entries, where the dots of four cost what
// one and a half do on dot4 and an operand of the activations is read once for four rows: each wavefront turns its weights through an LDS
// image of 76 words, from the order in which memory is read fastest into the instruction's.  The first weights are requested before the
// scan: they depend on the expert alone.  G lanes share a row (16, or 4 for contractions
// that are not a multiple of 1024 values: 768 is three trips of 4 lanes without an idle one).
//
// grid = (runs of rows, n_expert), block = 64 * kGuWaves / kDownWaves; dynamic LDS = 8 entries of entry_stride(n_pad) 16-byte words, n_pad =
// in_dim / 64 in whole trips of G.  Contractions are a multiple of 64; ids [n_entries], at most 65535, as the router wrote them, entry e = token
// e / n_used; at most kMaxEntries of one expert (the router picks an expert at most once per token).  An expert without
// entries ends at once.
//
// What bounds it (48 tokens of 128 experts top-8, 2048 x 768, Q4_K / Q6_K): not memory -- with every load from the cache the dot4 form took
// 45 / 39 us of 52 / 45 -- but the vector instructions of unpack, dots and scales and the returns of 32-byte pieces to registers.  Hence the
// matrix instruction, three wavefronts to a SIMD for Q4_K (168 registers; Q5_K and Q6_K would spill: 106 -> 118 us on dot4).  Whole FFN at 16 / 32 /
// 48 / 64 / 80 tokens, dot4 for every count / this: 75.5 / 74.3, 92.3 / 89.7, 103.9 / 96.7, 119.2 / 108.2, 131.2 / 117.1 us; 44 tokens of 32
// experts top-4, 4096 x 1536, 134.3 / 120.0; Q5_K at 60 tokens 122.5 / 111.8; Q8_0 at 48 134.4 / 130.8; the tiles of the pipeline 149-152 at any
// of the counts of the first shape.  Tried without gain: 8 or 16 wavefronts to a workgroup, two trips in flight per wavefront
// instead of one, runs of 32 or 128 columns, one sub-block at a time for fewer registers, the ids before the weights (-0.8 us), weights
// requested in the matrix instruction's order (quads of lanes on four rows: 78.8 / 101.1 at 16 / 48 tokens).
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

// 16-byte words between staged entries: 2 modulo 8, so that the four entries that a quad of lanes reads lie in different banks
template <int FMT> __device__ __forceinline__ unsigned entry_stride(unsigned n_pad) { return ((kParts<FMT> * n_pad + 5u) & ~7u) + 2u; }

// Over the units of a row, on lanes l = unit (dot4) or on quads of lanes 4 unit + c (the 4x4x4 form): both add the units that differ
// in bit 3, then 2, 1, 0, so an entry's result does not depend on the form that its batch took.
template <int G> __device__ __forceinline__ float group_sum(float v)
{
    if constexpr (G == 16) v += rein_dpp_f32<0x128>(0.0f, v);           // row_ror 8
    if constexpr (G == 16) v += rein_dpp_f32<0x124>(0.0f, v);           // row_ror 4
    if constexpr (G == 8) v += rein_row_xor4(v);
    v += rein_dpp_f32<0x4E>(0.0f, v);
    v += rein_dpp_f32<0xB1>(0.0f, v);
    return v;
}
// a + the same register 32 (16) lanes away, in the lower half (even rows of 16 lanes); b's in the others
__device__ __forceinline__ float sum_far32(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ float sum_far16(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ float sum_quads(float v)
{
    v += rein_dpp_f32<0x128>(0.0f, v);
    v += rein_dpp_f32<0x124>(0.0f, v);
    return v;
}
// four sums over the G quads of a lane group at once; held() says which of them a lane ends with, stores() the lane of each that is first
template <int G> __device__ __forceinline__ float group_sum4(const float (&v)[4])
{
    const unsigned lane = threadIdx.x & 63u;
    if constexpr (G == 16) {
        return sum_quads(sum_far16(sum_far32(v[0], v[2]), sum_far32(v[1], v[3])));
    } else if constexpr (G == 8) {
        const float a = sum_quads(sum_far16(v[0], v[1])), b = sum_quads(sum_far16(v[2], v[3]));
        return lane & 8u ? b : a;
    } else {
        const float a = sum_quads(v[0]), b = sum_quads(v[1]), c = sum_quads(v[2]), d = sum_quads(v[3]);
        const float ab = lane & 4u ? b : a, cd = lane & 4u ? d : c;
        return lane & 8u ? cd : ab;
    }
}
template <int G> __device__ __forceinline__ unsigned held()
{
    const unsigned lane = threadIdx.x & 63u;
    return G == 16 ? lane >> 4 : G == 8 ? ((lane >> 4) & 1u) + ((lane >> 2) & 2u) : (lane >> 2) & 3u;
}
template <int G> __device__ __forceinline__ bool stores() { return G == 16 ? !(threadIdx.x & 12u) : G == 8 ? !(threadIdx.x & 4u) : true; }

template <int R> __device__ __forceinline__ float quad_lane(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), R * 0x55, 0xF, 0xF, true));
}
template <int R> __device__ __forceinline__ int quad_lane(int v) { return __builtin_amdgcn_mov_dpp(v, R * 0x55, 0xF, 0xF, true); }

typedef int v4i __attribute__((ext_vector_type(4)));

// A pair of sub-blocks as 16-byte words, and a wavefront's image of 64 of them: written in the order of memory (lane = row, unit), read in
// the order of the 4x4x4 instruction (lane = unit, row).  Entry e lies at e + 4 (e / 16): sixteen lanes touch every bank once both ways.
template <int FMT> constexpr unsigned kWords = FMT == REIN_Q8_0 ? 5 : FMT == REIN_Q6_K ? 4 : 3;
constexpr unsigned kImage = 76;
template <int FMT> __device__ __forceinline__ void pack(const FmtPair<FMT>& v, uint4 (&o)[kWords<FMT>])
{
    o[0] = v.q0;
    o[1] = v.q1;
    if constexpr (FMT == REIN_Q8_0) { o[2] = v.h0; o[3] = v.h1; o[4] = make_uint4(v.sm, 0, 0, 0); }
    else if constexpr (FMT == REIN_Q6_K) { o[2] = make_uint4(v.h0.x, v.h0.y, v.h1.x, v.h1.y); o[3] = make_uint4(v.sm, v.dd, 0, 0); }
    else if constexpr (FMT == REIN_Q5_1) o[2] = make_uint4(v.qh.x, v.qh.y, v.dm.x, v.dm.y);
    else if constexpr (FMT == REIN_Q5_K) o[2] = make_uint4(v.sm, v.dd, v.qh.x, v.qh.y);
    else o[2] = make_uint4(v.sm, v.dd, 0, 0);
}
template <int FMT> __device__ __forceinline__ void unpack_words(FmtPair<FMT>& v, const uint4 (&o)[kWords<FMT>])
{
    v.q0 = o[0];
    v.q1 = o[1];
    if constexpr (FMT == REIN_Q8_0) { v.h0 = o[2]; v.h1 = o[3]; v.sm = o[4].x; }
    else if constexpr (FMT == REIN_Q6_K) { v.h0.x = o[2].x; v.h0.y = o[2].y; v.h1.x = o[2].z; v.h1.y = o[2].w; v.sm = o[3].x; v.dd = o[3].y; }
    else if constexpr (FMT == REIN_Q5_1) { v.qh.x = o[2].x; v.qh.y = o[2].y; v.dm.x = o[2].z; v.dm.y = o[2].w; }
    else { v.sm = o[2].x; v.dd = o[2].y; if constexpr (FMT == REIN_Q5_K) { v.qh.x = o[2].z; v.qh.y = o[2].w; } }
}

// A wavefront's rows: `rows(pass, lr, ra, rb)` says which row of wa and of wb the lane group lr works on in a pass.
// done(pass, lr, b, sum_a, sum_b) gets the sums of entry b, each on a lane of its own: lane b % G of the group.
template <int FMT, int G> struct Stream {
    static constexpr bool q6 = FMT == REIN_Q6_K, mins = !q6 && FMT != REIN_Q8_0;
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
        for (int b = 0; b < B; b++, x += entry_stride<FMT>(n_pad)) {
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
    struct Sub { int w[8]; float s0, s1; int sc[2]; };
    static __device__ __forceinline__ void unpack(const FmtPair<FMT>& v, int o, Sub& s)
    {
        SubW sw;
        const auto raw = v.get(o);
        Fmt<FMT>::unpack(raw, sw);
#pragma unroll
        for (int k = 0; k < 8; k++) s.w[k] = sw.w[k];
        s.s0 = sw.s0;
        s.s1 = sw.s1;
        if constexpr (q6) {
            s.sc[0] = (int)(int8_t)(raw.sm & 0xFFu);
            s.sc[1] = (int)(int8_t)(raw.sm >> 8);
            s.s0 = rein_h2f(raw.d);
        }
    }
    // what a lane reads of an entry for sub-block o of its unit
    struct X { int q[8]; float dx, xsum; int fold[2]; };
    static __device__ __forceinline__ void read(const uint4* x, unsigned u, unsigned n_pad, int o, X& v)
    {
        const uint4 x0 = x[2 * o * n_pad + u], x1 = x[(2 * o + 1) * n_pad + u], hd = x[4 * n_pad + u];
        v.q[0] = x0.x; v.q[1] = x0.y; v.q[2] = x0.z; v.q[3] = x0.w;
        v.q[4] = x1.x; v.q[5] = x1.y; v.q[6] = x1.z; v.q[7] = x1.w;
        if constexpr (q6) {
            v.fold[0] = o ? hd.z : hd.x;
            v.fold[1] = o ? hd.w : hd.y;
            const float2 d = reinterpret_cast<const float2*>(&x[5 * n_pad])[u];
            v.dx = o ? d.y : d.x;
        } else {
            v.dx = __builtin_bit_cast(float, o ? hd.y : hd.x);
            v.xsum = __builtin_bit_cast(float, o ? hd.w : hd.z);
        }
    }
    template <int R> static __device__ __forceinline__ void scale(const Sub& s, const X& e, const v4i& d0, const v4i& d1, float& acc)
    {
        int i = d0[R];
        if constexpr (q6) i = __mul24(i, quad_lane<R>(s.sc[0])) + __mul24(d1[R], quad_lane<R>(s.sc[1]));
        acc = fmaf(quad_lane<R>(s.s0) * e.dx, (float)i, acc);
        if constexpr (mins) acc = fmaf(-quad_lane<R>(s.s1), e.xsum, acc);
    }
    // NQ groups of four entries: lane 4 (G h + g) + c has the unit g of row 4 h + c, and of each group entry c with those four rows
    template <int NQ>
    static __device__ __forceinline__ void fours(const Pair& v, const uint4* lds, unsigned stride, unsigned u, unsigned n_pad, float (&acc)[2][NQ][4])
    {
#pragma unroll
        for (int o = 0; o < 2; o++) {
            Sub s[2];
            unpack(v[0], o, s[0]);
            unpack(v[1], o, s[1]);
#pragma unroll
            for (int n = 0; n < NQ; n++) {
                X e;
                read(lds + (4 * n + (threadIdx.x & 3u)) * stride, u, n_pad, o, e);
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    v4i d0 = {0, 0, 0, 0}, d1 = {0, 0, 0, 0};
                    if constexpr (q6) {
                        d0 = v4i{e.fold[0], e.fold[0], e.fold[0], e.fold[0]};
                        d1 = v4i{e.fold[1], e.fold[1], e.fold[1], e.fold[1]};
                    }
#pragma unroll
                    for (int k = 0; k < 4; k++) d0 = __builtin_amdgcn_mfma_i32_4x4x4i8(s[r].w[k], e.q[k], d0, 0, 0, 0);
#pragma unroll
                    for (int k = 4; k < 8; k++) {
                        if constexpr (q6) d1 = __builtin_amdgcn_mfma_i32_4x4x4i8(s[r].w[k], e.q[k], d1, 0, 0, 0);
                        else d0 = __builtin_amdgcn_mfma_i32_4x4x4i8(s[r].w[k], e.q[k], d0, 0, 0, 0);
                    }
                    scale<0>(s[r], e, d0, d1, acc[r][n][0]);
                    scale<1>(s[r], e, d0, d1, acc[r][n][1]);
                    scale<2>(s[r], e, d0, d1, acc[r][n][2]);
                    scale<3>(s[r], e, d0, d1, acc[r][n][3]);
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
    // three to eight entries on the 4x4x4 instruction, whose 4 NQ columns cost the same whatever they hold
    template <int NQ, class Rows, class Done>
    __device__ __forceinline__ void run_fours(const Planes& wa, const Planes& wb, const uint4* lds, uint4* image, unsigned n_unit, unsigned n_pad,
                                              unsigned n_pass, const Rows& rows, const Done& done)
    {
        const unsigned lane = threadIdx.x & 63u, c = lane & 3u, g = (lane >> 2) % G, h4 = (lane >> 2) / G * 4u;
        const unsigned trips = n_pad / G, stride = entry_stride<FMT>(n_pad);
        const unsigned e = (h4 + c) * G + g;
        uint4* const put = image + lane + 4u * (lane >> 4);
        const uint4* const get = image + e + 4u * (e >> 4);
        float acc[2][NQ][4] = {};
        unsigned pass = 0, t = 0;
        const auto step = [&](Pair& now, Pair& next) {
            const bool last = t + 1 == trips;
            const unsigned pass2 = last ? pass + 1 : pass, t2 = last ? 0 : t + 1;
            request(wa, wb, n_unit, min(pass2, n_pass - 1), t2, rows, next);
            Pair mine;
#pragma unroll
            for (int r = 0; r < 2; r++) {
                uint4 o[kWords<FMT>];
                pack<FMT>(now[r], o);
#pragma unroll
                for (unsigned k = 0; k < kWords<FMT>; k++) {
                    *put = o[k];
                    __builtin_amdgcn_wave_barrier();
                    o[k] = *get;
                    __builtin_amdgcn_wave_barrier();
                }
                unpack_words<FMT>(mine[r], o);
            }
            fours<NQ>(mine, lds, stride, g + G * t, n_pad, acc);
            if (last) {
#pragma unroll
                for (int n = 0; n < NQ; n++) {
                    const float a = group_sum4<G>(acc[0][n]), b = group_sum4<G>(acc[1][n]);
                    if (stores<G>()) done(pass, h4 + held<G>(), 4 * n + c, a, b);
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[0][n][i] = acc[1][n][i] = 0.0f;
                }
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
    // what lies in LDS behind the nb-th entry is computed and dropped
    template <class Rows, class Done>
    __device__ __forceinline__ void run_some(unsigned nb, const Planes& wa, const Planes& wb, const uint4* lds, uint4* images, unsigned n_unit,
                                             unsigned n_pad, unsigned n_pass, const Rows& rows, const Done& done)
    {
        uint4* image = images + (threadIdx.x >> 6) * kImage;
        if (nb > 4) run_fours<2>(wa, wb, lds, image, n_unit, n_pad, n_pass, rows, done);
        else if (nb > 2) run_fours<1>(wa, wb, lds, image, n_unit, n_pad, n_pass, rows, done);
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
    __shared__ uint4 images[kGuWaves * kImage];
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
            for (unsigned i = threadIdx.x; i < kBatch * entry_stride<FMT>(n_pad); i += blockDim.x) rein_few_lds[i] = make_uint4(0, 0, 0, 0);
        if (n_pad > n_unit && at == 0) __syncthreads();
        for (unsigned i = threadIdx.x; i < nb * n_sub; i += blockDim.x) {
            const unsigned b = i / n_sub, sb = i - b * n_sub;
            stage<FMT>(rein_few_lds + b * entry_stride<FMT>(n_pad), n_pad, sb, xq[(size_t)(list[at + b] / n_used) * n_sub + sb]);
        }
        __syncthreads();
        s.run_some(nb, wg, wu, rein_few_lds, images, n_unit, n_pad, n_pass, rows, [&](unsigned pass, unsigned lr, unsigned b, float g, float u) {
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
    __shared__ uint4 images[kDownWaves * kImage];
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
            for (unsigned i = threadIdx.x; i < kBatch * entry_stride<FMT>(n_pad); i += blockDim.x) rein_few_lds[i] = make_uint4(0, 0, 0, 0);
        if (n_pad > n_unit && at == 0) __syncthreads();
        for (unsigned i = threadIdx.x; i < nb * n_sub; i += blockDim.x) {
            const unsigned b = i / n_sub, sb = i - b * n_sub;
            stage<FMT>(rein_few_lds + b * entry_stride<FMT>(n_pad), n_pad, sb, xq[(size_t)list[at + b] * n_sub + sb]);
        }
        __syncthreads();
        s.run_some(nb, w, w, rein_few_lds, images, n_unit, n_pad, n_pass, rows, [&](unsigned pass, unsigned lr, unsigned b, float va, float vb) {
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
    extern "C" __global__ __launch_bounds__(64 * rein_few::kGuWaves, (FMT == REIN_Q4_K ? 3 : 2)) void rein_moe_few_gate_up_##tag##_g##G(              \
        const unsigned char* __restrict__ gate_slab, const unsigned char* __restrict__ up_slab, const int* __restrict__ ids, \
        const BlockQ8* __restrict__ xq, BlockQ8* __restrict__ xq_out, unsigned int bytes_per_expert, unsigned int in_dim,    \
        unsigned int out_dim, unsigned int n_used, unsigned int n_entries)                                                   \
    {                                                                                                                        \
        rein_few::gate_up<FMT, G>(gate_slab, up_slab, bytes_per_expert, ids, xq, xq_out, in_dim, out_dim, n_used, n_entries); \
    }                                                                                                                        \
    extern "C" __global__ __launch_bounds__(64 * rein_few::kDownWaves, (FMT == REIN_Q4_K ? 3 : 2)) void rein_moe_few_down_##tag##_g##G(               \
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
