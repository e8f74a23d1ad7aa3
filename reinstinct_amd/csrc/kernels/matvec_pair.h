// Two consecutive sub-blocks of a repacked row as one lane reads them: 64 weights, the words of both sub-blocks of a plane
// side by side.  Needs an even number of sub-blocks per row and a slab below 4 GiB (offsets are 32-bit, so that a load is a
// scalar base plus one register).
//
// The loads are ordinary ones, not the streaming loads of rein_formats.h: a group of lanes reads a few hundred
// bytes of a row at a time, the rest of a cache line follows a trip later or belongs to the next row's lanes, and a line that
// was marked for early eviction is then fetched again (a 16-lane matvec of Q4_K 5120 -> 34816 on these pairs: 25.4 us with streaming
// loads, 20.4 without).
#pragma once

#include "rein_formats.h"

typedef uint32_t rein_u32_a2 __attribute__((aligned(2)));
struct __attribute__((packed, aligned(4))) ReinU32x2A4 { uint32_t x, y; };

// Where a slab's planes begin (uniform), and a row's entries in them
template <int FMT> struct PairPlanes {
    const uint8_t *p0, *p1, *p2, *p3;
    unsigned nsp, n_super;
    __device__ PairPlanes(const uint8_t* w, unsigned n_sub, unsigned out_dim)
    {
        nsp = rein_nsp(n_sub);
        n_super = n_sub >> 3;
        constexpr unsigned e0 = 16, e1 = FMT == REIN_Q8_0 ? 16 : FMT == REIN_Q6_K ? 8 : FMT == REIN_Q4_K ? 2 : 4, e2 = FMT == REIN_Q5_1 ? 4 : 2;
        const size_t n = (size_t)out_dim * nsp;
        p0 = w;
        p1 = w + n * e0;
        p2 = p1 + n * e1;
        p3 = FMT == REIN_Q4_K ? p2 : p2 + n * e2;           // superblock entries
    }
    // byte offset / 16 of a pair in the first plane; of its superblock, in entries
    __device__ __forceinline__ unsigned at(unsigned row, unsigned u) const { return row * nsp + 2u * u; }
    __device__ __forceinline__ unsigned super(unsigned row, unsigned u) const { return row * n_super + (u >> 2); }
};

template <class T> __device__ __forceinline__ T rein_at(const uint8_t* p, unsigned byte) { return *reinterpret_cast<const T*>(p + byte); }

template <int FMT> struct FmtPair {
    static constexpr bool kFive = FMT == REIN_Q5_K || FMT == REIN_Q5_1;
    uint4 q0, q1;
    uint4 h0, h1;                 // Q8_0: quants 16-31; Q6_K: x, y are its 2-bit words
    ReinU32x2A4 qh;               // fifth bits
    ReinU32x2A4 dm;               // Q5_1: fp16 d, m of both
    uint32_t sm, dd;              // scale bytes or fp16 d of both; superblock scales
    __device__ __forceinline__ void load(const PairPlanes<FMT>& f, unsigned i, unsigned s)
    {
        q0 = rein_at<uint4>(f.p0, i * 16);
        q1 = rein_at<uint4>(f.p0, i * 16 + 16);
        if constexpr (FMT == REIN_Q8_0) {
            h0 = rein_at<uint4>(f.p1, i * 16);
            h1 = rein_at<uint4>(f.p1, i * 16 + 16);
        }
        if constexpr (FMT == REIN_Q6_K) {
            const uint2 a = rein_at<uint2>(f.p1, i * 8), b = rein_at<uint2>(f.p1, i * 8 + 8);
            h0.x = a.x; h0.y = a.y; h1.x = b.x; h1.y = b.y;
        }
        if constexpr (kFive) qh = rein_at<ReinU32x2A4>(f.p1, i * 4);
        if constexpr (FMT == REIN_Q5_1) dm = rein_at<ReinU32x2A4>(f.p2, i * 4);
        else sm = rein_at<rein_u32_a2>(FMT == REIN_Q4_K ? f.p1 : f.p2, i * 2);
        if constexpr (FMT == REIN_Q4_K || FMT == REIN_Q5_K) dd = rein_at<uint32_t>(f.p3, s * 4);
        if constexpr (FMT == REIN_Q6_K) dd = rein_at<uint16_t>(f.p3, s * 2);
    }
    // sub-block o of the pair as the words of the format's own unpack
    __device__ __forceinline__ typename Fmt<FMT>::Raw get(int o) const
    {
        typename Fmt<FMT>::Raw r;
        const uint16_t two = (uint16_t)(o ? sm >> 16 : sm & 0xFFFFu);
        if constexpr (FMT == REIN_Q8_0) {
            r.lo = o ? q1 : q0;
            r.hi = o ? h1 : h0;
            r.d = two;
        } else {
            r.q = o ? q1 : q0;
            if constexpr (FMT == REIN_Q6_K) { r.h2 = o ? make_uint2(h1.x, h1.y) : make_uint2(h0.x, h0.y); r.sm = two; r.d = (uint16_t)dd; }
            if constexpr (FMT == REIN_Q4_K || FMT == REIN_Q5_K) { r.sm = two; r.dd = dd; }
            if constexpr (kFive) r.qh = o ? qh.y : qh.x;
            if constexpr (FMT == REIN_Q5_1) r.dm = o ? dm.y : dm.x;
        }
        return r;
    }
};
