// The matvec over on-disk (GGUF) blocks as the library launches it, rein_mvd_<fmt>: the output projection of a model whose
// embedding is tied (src/runtime/qwen35.rs:2209-2229).  Same product as the reference-named kernels of
// matvec_ondisk.hip, which take any launch geometry and no LDS; what differs is who reads which bytes.
//
// There a lane owns a 32-weight sub-block, and a sub-block's fields are spread over its 256-weight block: in Q6_K the 2-bit
// plane's bytes are read by four lanes each, the nibbles by two, four bytes at a time because the blocks are 2-byte aligned.
// The launch was bound by those load instructions (Q6_K 2048 -> 151936, 255 MB: 80 us = 3.2 TB/s).  Here a lane owns the 64 weights
// that share bytes -- part p of a block:
//   Q6_K   16 columns of one half: ql[64n + 16h ..+16], ql[64n + 32 + 16h ..+16], qh[32n + 16h ..+16] (n = p / 2, h = p % 2)
//          -> 16 weights, exactly one scale group, of each of the half's four sub-blocks
//   Q4_K   qs[32p ..+32] -> sub-blocks 2p (low nibbles) and 2p + 1 (high);  Q5_K also all of qh (bits 2p, 2p + 1)
//   Q8_0   two blocks, 68 bytes
// so every byte is read once, in 16-byte loads whatever the alignment.  Sixteen lanes (one DPP row, which also does the
// reduction) walk a row, four blocks a trip; a wavefront works on four rows, which suits the short contractions these
// matrices have: 2048 weights are two trips without an idle lane, where 64 lanes to a row left half of them idle.
// The activations are staged in LDS once per workgroup (a lane needs pieces of four of their blocks per trip), with a pad per 256
// values that spreads the blocks of a trip over the banks; the next trip's weights, or the next row group's first,
// are requested before the present ones are used.
#include "rein_formats.h"

typedef uint32_t rein_u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t rein_u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t rein_u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// What a workgroup keeps of the activations: quants in blocks of 256 + kPad bytes, dx per sub-block, and the sums a format
// needs: xsum per sub-block (fp32), or the integer sums of 16 quants, one array per half (Q6_K).
template <int FMT> struct DiskX {
    static constexpr unsigned kPad = FMT == REIN_Q6_K ? 32 : 16;
    static constexpr bool kSums16 = FMT == REIN_Q6_K, kXsum = FMT == REIN_Q4_K || FMT == REIN_Q5_K;
    const uint8_t* q;
    const float* dx;
    const float* xsum;        // or int sums: [2][n_pad]
    unsigned n_pad;
    __device__ DiskX(uint8_t* lds, unsigned n_sub)
    {
        n_pad = (n_sub + 7u) & ~7u;
        q = lds;
        dx = reinterpret_cast<const float*>(lds + (n_pad >> 3) * (256 + kPad));
        xsum = dx + n_pad;
    }
    __device__ __forceinline__ const uint4* at(unsigned blk, unsigned byte) const
    {
        return reinterpret_cast<const uint4*>(q + blk * (256 + kPad) + byte);
    }
    __device__ __forceinline__ void stage(uint8_t* lds, const BlockQ8* __restrict__ xq, unsigned n_sub) const
    {
        float* d = const_cast<float*>(dx);
        float* s = const_cast<float*>(xsum);
        for (unsigned sb = threadIdx.x; sb < n_sub; sb += blockDim.x) {
            const BlockQ8 b = xq[sb];
            uint4* o = reinterpret_cast<uint4*>(lds + (sb >> 3) * (256 + kPad) + (sb & 7u) * 32);
            o[0] = make_uint4(b.qs[0], b.qs[1], b.qs[2], b.qs[3]);
            o[1] = make_uint4(b.qs[4], b.qs[5], b.qs[6], b.qs[7]);
            d[sb] = b.d;
            if (kXsum) s[sb] = b.xsum;
            if (kSums16) {
                int lo = 0, hi = 0;
#pragma unroll
                for (int j = 0; j < 4; j++) { lo = rein_dot4(b.qs[j], 0x01010101, lo); hi = rein_dot4(b.qs[4 + j], 0x01010101, hi); }
                reinterpret_cast<int*>(s)[sb] = lo;
                reinterpret_cast<int*>(s)[n_pad + sb] = hi;
            }
        }
    }
};

__device__ __forceinline__ int rein_dot16(const uint4& a, const uint32_t w[4])
{
    int i = rein_dot4((int)w[0], (int)a.x, 0);
    i = rein_dot4((int)w[1], (int)a.y, i);
    i = rein_dot4((int)w[2], (int)a.z, i);
    return rein_dot4((int)w[3], (int)a.w, i);
}

// Part p of block blk of a row: raw words, and its contribution to the row's sum
template <int FMT> struct DiskPart;

template <> struct DiskPart<REIN_Q6_K> {
    static constexpr unsigned kBlock = 210;
    rein_u32x4_a2 l0, l1, hi;
    rein_u32x2_a2 sc;
    uint16_t d;
    __device__ __forceinline__ void load(const uint8_t* row, unsigned blk, unsigned p)
    {
        const uint8_t* b = row + blk * kBlock;
        const unsigned n = p >> 1, h = p & 1u;
        l0 = *reinterpret_cast<const rein_u32x4_a2*>(b + 64 * n + 16 * h);
        l1 = *reinterpret_cast<const rein_u32x4_a2*>(b + 64 * n + 32 + 16 * h);
        hi = *reinterpret_cast<const rein_u32x4_a2*>(b + 128 + 32 * n + 16 * h);
        sc = *reinterpret_cast<const rein_u32x2_a2*>(b + 192 + 8 * n);
        d = *reinterpret_cast<const uint16_t*>(b + 208);
    }
    struct X { uint4 q[4]; float4 dx; int4 s; };
    static __device__ __forceinline__ X fetch(const DiskX<REIN_Q6_K>& x, unsigned blk, unsigned p)
    {
        X v;
        const unsigned n = p >> 1, h = p & 1u, sb = blk * 8 + 4 * n;
#pragma unroll
        for (int g = 0; g < 4; g++) v.q[g] = *x.at(blk, 128 * n + 32 * g + 16 * h);
        v.dx = *reinterpret_cast<const float4*>(x.dx + sb);
        v.s = *reinterpret_cast<const int4*>(reinterpret_cast<const int*>(x.xsum) + h * x.n_pad + sb);
        return v;
    }
    // d * sum over the four sub-blocks of dx * (sc * (dot - 32 * sum of the quants)); the product of whole numbers is below 2^24
    __device__ __forceinline__ float term(const X& x, unsigned p) const
    {
        const float dx[4] = {x.dx.x, x.dx.y, x.dx.z, x.dx.w};
        const int s[4] = {x.s.x, x.s.y, x.s.z, x.s.w};
        const unsigned sh = 8u * (p & 1u);
        const uint32_t sc01 = sc.x >> sh, sc23 = sc.y >> sh;
        float t = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const rein_u32x4_a2& l = g & 1 ? l1 : l0;
            uint32_t w[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t lo = (g & 2 ? l[k] >> 4 : l[k]) & 0x0F0F0F0Fu;
                const uint32_t h2 = g == 0 ? hi[k] << 4 : g == 1 ? hi[k] << 2 : g == 2 ? hi[k] : hi[k] >> 2;
                w[k] = (h2 & 0x30303030u) | lo;
            }
            const int dot = rein_dot16(x.q[g], w) - 32 * s[g];
            const int scale = (int)(int8_t)((g & 2 ? sc23 : sc01) >> (g & 1 ? 16 : 0));
            t = fmaf((float)__mul24(dot, scale), dx[g], t);
        }
        return t * rein_h2f(d);
    }
};

// (scale, min) of sub-blocks 2p and 2p + 1 from the 12 packed bytes s0, s1, s2 (q4_k.rs:40-48), in bytes 0 and 1
__device__ __forceinline__ void rein_scales_pair(unsigned p, uint32_t s0, uint32_t s1, uint32_t s2, uint32_t& sc, uint32_t& mn)
{
    const unsigned sh = 16u * (p & 1u);
    const uint32_t a = s0 >> sh, b = s1 >> sh, c = s2 >> sh;
    if (p < 2u) {
        sc = a & 0x3F3Fu;
        mn = b & 0x3F3Fu;
    } else {
        sc = (c & 0x0F0Fu) | ((a >> 2) & 0x3030u);
        mn = ((c >> 4) & 0x0F0Fu) | ((b >> 2) & 0x3030u);
    }
}

template <int FMT> struct DiskPartK {           // Q4_K, Q5_K
    static constexpr bool kFive = FMT == REIN_Q5_K;
    static constexpr unsigned kBlock = kFive ? 176 : 144;
    uint4 head, a, b, ha, hb;
    __device__ __forceinline__ void load(const uint8_t* row, unsigned blk, unsigned p)
    {
        const uint4* u = reinterpret_cast<const uint4*>(row + blk * kBlock);
        head = u[0];
        if (kFive) { ha = u[1]; hb = u[2]; }
        const uint4* q = u + (kFive ? 3 : 1) + 2 * p;
        a = q[0];
        b = q[1];
    }
    struct X { uint4 q[4]; float2 dx, xs; };
    static __device__ __forceinline__ X fetch(const DiskX<FMT>& x, unsigned blk, unsigned p)
    {
        X v;
        const unsigned sb = blk * 8 + 2 * p;
#pragma unroll
        for (int k = 0; k < 4; k++) v.q[k] = x.at(blk, 64 * p)[k];
        v.dx = *reinterpret_cast<const float2*>(x.dx + sb);
        v.xs = *reinterpret_cast<const float2*>(x.xsum + sb);
        return v;
    }
    __device__ __forceinline__ float term(const X& x, unsigned p) const
    {
        const uint32_t q[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        const uint32_t h[8] = {ha.x, ha.y, ha.z, ha.w, hb.x, hb.y, hb.z, hb.w};
        int dot[2] = {0, 0};
#pragma unroll
        for (int k = 0; k < 8; k++) {
            uint32_t lo = q[k] & 0x0F0F0F0Fu, hi = (q[k] >> 4) & 0x0F0F0F0Fu;
            if (kFive) {
                const uint32_t v = h[k] >> (2 * p);
                lo |= (v << 4) & 0x10101010u;
                hi |= (v << 3) & 0x10101010u;
            }
            const uint4& x0 = x.q[k >> 2];
            const uint4& x1 = x.q[2 + (k >> 2)];
            dot[0] = rein_dot4((int)lo, (int)(k % 4 == 0 ? x0.x : k % 4 == 1 ? x0.y : k % 4 == 2 ? x0.z : x0.w), dot[0]);
            dot[1] = rein_dot4((int)hi, (int)(k % 4 == 0 ? x1.x : k % 4 == 1 ? x1.y : k % 4 == 2 ? x1.z : x1.w), dot[1]);
        }
        uint32_t sc, mn;
        rein_scales_pair(p, head.y, head.z, head.w, sc, mn);
        const float d = rein_h2f((uint16_t)(head.x & 0xFFFFu)), dmin = rein_h2f((uint16_t)(head.x >> 16));
        // whole-number products are below 2^24: 32 * 31 * 127 * 63 < 2^23
        const float t = fmaf((float)__mul24(dot[1], (int)(sc >> 8)), x.dx.y, (float)__mul24(dot[0], (int)(sc & 0xFFu)) * x.dx.x);
        const float m = fmaf((float)(mn >> 8), x.xs.y, (float)(mn & 0xFFu) * x.xs.x);
        return d * t - dmin * m;
    }
};
template <> struct DiskPart<REIN_Q4_K> : DiskPartK<REIN_Q4_K> {};
template <> struct DiskPart<REIN_Q5_K> : DiskPartK<REIN_Q5_K> {};

template <> struct DiskPart<REIN_Q8_0> {        // two 34-byte blocks; rows are an even number of them, so 4-byte aligned
    static constexpr unsigned kBlock = 272;     // of eight
    rein_u32x4_a4 v[4];
    uint32_t last;
    __device__ __forceinline__ void load(const uint8_t* row, unsigned blk, unsigned p)
    {
        const uint8_t* b = row + blk * kBlock + p * 68;
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = *reinterpret_cast<const rein_u32x4_a4*>(b + 16 * k);
        last = *reinterpret_cast<const uint32_t*>(b + 64);
    }
    struct X { uint4 q[4]; float2 dx; };
    static __device__ __forceinline__ X fetch(const DiskX<REIN_Q8_0>& x, unsigned blk, unsigned p)
    {
        X r;
#pragma unroll
        for (int k = 0; k < 4; k++) r.q[k] = x.at(blk, 64 * p)[k];
        r.dx = *reinterpret_cast<const float2*>(x.dx + blk * 8 + 2 * p);
        return r;
    }
    __device__ __forceinline__ float term(const X& x, unsigned) const
    {
        uint32_t w[17];
#pragma unroll
        for (int k = 0; k < 16; k++) w[k] = v[k >> 2][k & 3];
        w[16] = last;
        uint32_t q0[8];                          // the first block's quants start at byte 2
#pragma unroll
        for (int k = 0; k < 8; k++) q0[k] = __builtin_amdgcn_alignbyte(w[k + 1], w[k], 2);
        const int i0 = rein_dot16(x.q[0], q0) + rein_dot16(x.q[1], q0 + 4);
        const int i1 = rein_dot16(x.q[2], w + 9) + rein_dot16(x.q[3], w + 13);
        const float d0 = rein_h2f((uint16_t)(w[0] & 0xFFFFu)), d1 = rein_h2f((uint16_t)(w[8] >> 16));
        return fmaf((float)i1, d1 * x.dx.y, (float)i0 * (d0 * x.dx.x));
    }
};

// LDS: DiskX of the row, (n_pad / 8) * (256 + kPad) + n_pad * 4 * (1 + sums) bytes.  A workgroup per 512 (Q6_K, Q8_0) or
// 1024 (Q4_K, Q5_K) strides over the rows; two rows per 16 lanes (half the LDS reads, more registers) and more or all
// workgroups at once are 5-20 % slower.  us before -> now (TB/s of weights), three matrices in turn:
//   2048 -> 151936   Q6_K 80.2 -> 45.5 (5.6)   Q4_K 48.0 -> 30.5 (5.7)   Q5_K 60.0 -> 37.3 (5.7)   Q8_0 81.7 -> 54.4 (6.1)
//   5120 -> 151936   Q6_K 235 -> 107 (6.0)     Q4_K 124 -> 72.2 (6.1)    Q5_K 158 -> 89.7 (6.0)    Q8_0 202 -> 139 (5.9)
// which is the rate at which this part reads: what bounds it now is HBM.  Up to 2048 rows, where the kernels of matvec_ondisk.hip have a
// workgroup per CU, rein_matvec_ondisk_xq8 keeps those for Q8_0 and for most contractions of Q6_K.
template <int FMT>
__device__ __forceinline__ void rein_matvec_disk(const uint8_t* __restrict__ w, const BlockQ8* __restrict__ xq, float* __restrict__ y,
                                                 unsigned in_dim, unsigned out_dim)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t rein_lds_disk[];
    using P = DiskPart<FMT>;
    const unsigned n_sub = in_dim >> 5, n_unit = n_sub >> 1;                 // parts of a row (n_sub is even)
    const size_t row_bytes = FMT == REIN_Q8_0 ? (size_t)n_sub * 34 : (size_t)(n_sub >> 3) * P::kBlock;
    const unsigned lane = threadIdx.x & 63u, wpb = blockDim.x >> 6, l = lane & 15u;
    const unsigned trips = (n_unit + 15u) >> 4;
    const unsigned n_groups = (out_dim + 3) / 4, rmax = out_dim - 1;
    const DiskX<FMT> x(rein_lds_disk, n_sub);

    unsigned g = blockIdx.x * wpb + (threadIdx.x >> 6), t = 0;
    P cur, nxt;
    // always a valid row and part: past the end the last ones are read again, which keeps the loads out of a branch
    const auto request = [&](unsigned gg, unsigned tt, P& v) {
        const unsigned u = min(l + 16u * tt, n_unit - 1), row = min(min(gg, n_groups - 1) * 4u + (lane >> 4), rmax);
        v.load(w + row * row_bytes, u >> 2, u & 3u);
    };
    request(g, 0, cur);
    x.stage(rein_lds_disk, xq, n_sub);
    __syncthreads();
    float acc = 0.0f;
    while (g < n_groups) {
        const bool last = t + 1 == trips;
        const unsigned g2 = last ? g + gridDim.x * wpb : g, t2 = last ? 0 : t + 1;
        request(g2, t2, nxt);
        const unsigned u = l + 16u * t, uc = min(u, n_unit - 1);
        const float c = cur.term(P::fetch(x, uc >> 2, uc & 3u), uc & 3u);
        acc += u < n_unit ? c : 0.0f;
        if (last) {
            const float s = rein_row16_sum(acc);
            const unsigned row = g * 4u + (lane >> 4);
            if (l == 0 && row < out_dim) y[row] = s;
            acc = 0.0f;
        }
        cur = nxt;
        g = g2;
        t = t2;
    }
}

#define REIN_DEFINE_MATVEC_DISK(name, FMT)                                                                               \
    extern "C" __global__ __launch_bounds__(256) void name(const unsigned char* __restrict__ w, const BlockQ8* __restrict__ xq, \
                                                           float* __restrict__ y, unsigned int in_dim, unsigned int out_dim)    \
    {                                                                                                                    \
        rein_matvec_disk<FMT>(w, xq, y, in_dim, out_dim);                                                                \
    }
REIN_DEFINE_MATVEC_DISK(rein_mvd_q4k, REIN_Q4_K)
REIN_DEFINE_MATVEC_DISK(rein_mvd_q5k, REIN_Q5_K)
REIN_DEFINE_MATVEC_DISK(rein_mvd_q6k, REIN_Q6_K)
REIN_DEFINE_MATVEC_DISK(rein_mvd_q8_0, REIN_Q8_0)
