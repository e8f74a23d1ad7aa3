// Host-side mirror of the reference's src/quant layout contract: repacked_len,
// repacked_n_sub_padded and repack_for_matvec for the six formats.  Load-time
// code (runs once per weight, host to host): a row of on-disk blocks at a time, eight bytes of
// a plane per step.  Rows are split over threads.
#include <algorithm>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

#include "../../../include/rein.h"
#include "hip_api.h"
#include "iq3s_grid.h"
#include "repack.h"

namespace {

struct Geometry {
    int    block;        // weights per on-disk block
    int    bytes;        // bytes per on-disk block
    size_t per_sub;      // bytes per sub-block over all per-sub-block planes
    size_t per_super;    // bytes per 256-weight superblock plane entry
};

bool geometry(int fmt, Geometry* g)
{
    switch (fmt) {
    case REIN_TYPE_Q4_0:   *g = {32, 18, 16 + 2, 0}; return true;       // src/quant/q4_0.rs:22-23,66-69
    case REIN_TYPE_Q8_0:   *g = {32, 34, 32 + 2, 0}; return true;       // src/quant/q8_0.rs:8-9,74-77
    case REIN_TYPE_Q4_K:   *g = {256, 144, 16 + 2, 4}; return true;     // src/quant/q4_k.rs:17-18,98-102
    case REIN_TYPE_Q5_K:   *g = {256, 176, 16 + 4 + 2, 4}; return true; // src/quant/q5_k.rs:21-22,100-104
    case REIN_TYPE_Q6_K:   *g = {256, 210, 16 + 8 + 2, 2}; return true; // src/quant/q6_k.rs:18-19,89-93
    case REIN_TYPE_IQ4_XS: *g = {256, 136, 16 + 2, 0}; return true;     // src/quant/iq4_xs.rs:23-24,85-88
    case REIN_TYPE_Q5_1:   *g = {32, 24, 16 + 4 + 4, 0}; return true;   // src/quant/q5_1.rs:25-26,76-81
    case REIN_TYPE_IQ3_S:  *g = {256, 110, 16 + 2, 0}; return true;     // src/quant/iq3_s.rs:24-25,178-184
    default: return false;
    }
}

inline uint16_t load16(const uint8_t* p) { return (uint16_t)(p[0] | (p[1] << 8)); }
inline void store16(uint8_t* p, uint16_t v) { p[0] = (uint8_t)v; p[1] = (uint8_t)(v >> 8); }

// IEEE half <-> float with the reference's rounding behaviour
// (src/quant/half.rs:9-40, 51-84: RNE for normal results, truncation for
// subnormal results).
float half_to_float(uint16_t h)
{
    const uint32_t sign = (uint32_t)(h >> 15) << 31;
    int      e = (h >> 10) & 31;
    uint32_t m = h & 1023u;
    uint32_t bits;
    if (e == 31) {
        bits = sign | 0x7F800000u | (m << 13);
    } else if (e != 0) {
        bits = sign | ((uint32_t)(e + 112) << 23) | (m << 13);
    } else if (m == 0) {
        bits = sign;
    } else {
        e = 113;
        while (!(m & 1024u)) { m <<= 1; e--; }
        bits = sign | ((uint32_t)e << 23) | ((m & 1023u) << 13);
    }
    float f;
    std::memcpy(&f, &bits, 4);
    return f;
}

uint16_t float_to_half(float f)
{
    uint32_t b;
    std::memcpy(&b, &f, 4);
    const uint16_t sign = (uint16_t)((b >> 16) & 0x8000u);
    const int      e = (int)((b >> 23) & 255u) - 127;
    const uint32_t m = b & 0x7FFFFFu;
    if (e == 128) return (uint16_t)(sign | 0x7C00u | (m ? 0x200u : 0u));
    if (e > 15) return (uint16_t)(sign | 0x7C00u);
    if (e < -24) return sign;
    if (e < -14) return (uint16_t)(sign | (uint16_t)((m | 0x800000u) >> (unsigned)(-1 - e)));
    uint16_t h = (uint16_t)(sign | (uint16_t)((e + 15) << 10) | (uint16_t)(m >> 13));
    const uint32_t rest = m & 0x1FFFu;
    if (rest > 0x1000u || (rest == 0x1000u && (h & 1u))) h = (uint16_t)(h + 1u);
    return h;
}

// nibbles 8 + l of the four weights of a codebook entry, one to a byte
struct Iq3sNibbles {
    uint32_t at[512];
    constexpr Iq3sNibbles() : at()
    {
        for (unsigned e = 0; e < 512; e++)
            for (unsigned j = 0; j < 4; j++) at[e] |= (uint32_t)((rein::iq3s_magnitude(e, j) + 15) / 2) << (8 * j);
    }
    constexpr uint32_t operator[](unsigned e) const { return at[e]; }
};
constexpr Iq3sNibbles kIq3sNibbles;
// bits 0-3 -> 0xFF in bytes 0-3
inline uint32_t spread4(uint32_t v) { return (((v & 15u) * 0x00204081u) & 0x01010101u) * 0xFFu; }

// ---- eight bytes at a time.  Every nibble plane byte j of a sub-block is weight j in the low half and weight 16 + j in
// the high half (q4_k.rs:158-165), so it comes from two runs of source bytes by a mask and a shift.
constexpr uint64_t kLow = 0x0F0F0F0F0F0F0F0Full, kHigh = ~kLow;
inline uint64_t load64(const uint8_t* p) { uint64_t v; std::memcpy(&v, p, 8); return v; }
inline uint32_t load32(const uint8_t* p) { uint32_t v; std::memcpy(&v, p, 4); return v; }
inline void store64(uint8_t* p, uint64_t v) { std::memcpy(p, &v, 8); }
inline void store32(uint8_t* p, uint32_t v) { std::memcpy(p, &v, 4); }
// low nibbles (high nibbles) of 32 bytes -> one 16-byte plane entry
inline void low_entry(const uint8_t* q, uint8_t* o)
{
    for (int j = 0; j < 16; j += 8) store64(o + j, (load64(q + j) & kLow) | ((load64(q + 16 + j) & kLow) << 4));
}
inline void high_entry(const uint8_t* q, uint8_t* o)
{
    for (int j = 0; j < 16; j += 8) store64(o + j, ((load64(q + j) >> 4) & kLow) | (load64(q + 16 + j) & kHigh));
}
// bit 0 of four bytes -> four bits, two bits of four bytes -> one byte: the partial products of the
// multiplication do not overlap
inline uint32_t gather1(uint32_t v) { return ((v & 0x01010101u) * 0x01020408u) >> 24 & 15u; }
inline uint32_t gather2(uint32_t v) { return ((v & 0x03030303u) * 0x01041040u) >> 24; }
static_assert(0x01041040u == ((1u << 24) | (1u << 18) | (1u << 12) | (1u << 6)), "byte i of the word moves to bit 24 + 2 i");

// (scale, min) pairs of the eight sub-blocks from the 12 packed bytes (q4_k.rs:40-48), interleaved
inline void scales_k4(const uint8_t* q, uint8_t* o)
{
    const uint32_t a = load32(q), b = load32(q + 4), c = load32(q + 8);
    const uint32_t sc[2] = {a & 0x3F3F3F3Fu, (c & 0x0F0F0F0Fu) | ((a >> 2) & 0x30303030u)};
    const uint32_t mn[2] = {b & 0x3F3F3F3Fu, ((c >> 4) & 0x0F0F0F0Fu) | ((b >> 2) & 0x30303030u)};
    for (int h = 0; h < 2; h++)
        for (int i = 0; i < 4; i++) {
            o[8 * h + 2 * i]     = (uint8_t)(sc[h] >> (8 * i));
            o[8 * h + 2 * i + 1] = (uint8_t)(mn[h] >> (8 * i));
        }
}

// One output row's place in the planes of a slab: byte offsets of its first entry, in plane order (at most four planes
// of one entry per sub-block, then one entry per superblock).
struct Layout {
    size_t n_sub, nsp, n_super, n_rows;
    size_t entry[4];                   // bytes per sub-block of each plane (0: no such plane)
    size_t super;                      // bytes per superblock
};

Layout layout_of(int fmt, const Geometry& g, size_t in_dim, size_t out_dim)
{
    Layout l = {in_dim / 32, rein_repacked_n_sub_padded(in_dim), in_dim / 256, out_dim, {16, 0, 0, 0}, g.per_super};
    switch (fmt) {
    case REIN_TYPE_Q8_0: l.entry[1] = 16; l.entry[2] = 2; break;      // quants 16-31; fp16 d
    case REIN_TYPE_Q5_K: l.entry[1] = 4; l.entry[2] = 2; break;       // fifth bits; scale, min
    case REIN_TYPE_Q5_1: l.entry[1] = 4; l.entry[2] = 4; break;       // fifth bits; fp16 d, m
    case REIN_TYPE_Q6_K: l.entry[1] = 8; l.entry[2] = 2; break;       // bits 4-5; two int8 scales
    default:             l.entry[1] = 2; break;                       // scale, min (Q4_K) or fp16 scale
    }
    return l;
}

// One row: `b` its on-disk blocks; p[i] its first entry of plane i, ps its first superblock entry.
template <int FMT>
void repack_row(const uint8_t* b, size_t n_sub, uint8_t* const p[4], uint8_t* ps)
{
    uint8_t *nib = p[0], *p1 = p[1], *p2 = p[2];
    if constexpr (FMT == REIN_TYPE_Q4_0) {             // q4_0.rs:86-104: nibble bytes verbatim, fp16 d split out
        for (size_t i = 0; i < n_sub; i++, b += 18) {
            std::memcpy(nib + i * 16, b + 2, 16);
            std::memcpy(p1 + i * 2, b, 2);
        }
    } else if constexpr (FMT == REIN_TYPE_Q8_0) {      // q8_0.rs:93-119: quants 0-15 | quants 16-31 | fp16 d
        for (size_t i = 0; i < n_sub; i++, b += 34) {
            std::memcpy(nib + i * 16, b + 2, 16);
            std::memcpy(p1 + i * 16, b + 18, 16);
            std::memcpy(p2 + i * 2, b, 2);
        }
    } else if constexpr (FMT == REIN_TYPE_Q5_1) {      // q5_1.rs:82-104: nibbles verbatim, qh in dot-group order, raw fp16 d | m
        for (size_t i = 0; i < n_sub; i++, b += 24) {
            std::memcpy(nib + i * 16, b + 8, 16);
            // on disk bit k is weight k; in the plane byte j holds weights 4j.. and 16 + 4j..
            const uint32_t bits = load32(b + 4);
            uint32_t qh = 0;
            for (int j = 0; j < 4; j++) qh |= (((bits >> (4 * j)) & 15u) | (((bits >> (16 + 4 * j)) & 15u) << 4)) << (8 * j);
            store32(p1 + i * 4, qh);
            std::memcpy(p2 + i * 4, b, 4);
        }
    } else {
        for (size_t sb = 0; sb < n_sub; sb += 8) {
            uint8_t* n0 = nib + sb * 16;
            if constexpr (FMT == REIN_TYPE_IQ4_XS) {   // iq4_xs.rs:106-136: nibbles verbatim, fp16(d*(ls-32))
                std::memcpy(n0, b + 8, 128);
                const float d = half_to_float(load16(b));
                const unsigned high = load16(b + 2);
                for (int s = 0; s < 8; s++) {
                    const int ls = ((b[4 + s / 2] >> (4 * (s & 1))) & 15) | (((high >> (2 * s)) & 3) << 4);
                    store16(p1 + (sb + s) * 2, float_to_half(d * (float)(ls - 32)));
                }
                b += 136;
            } else if constexpr (FMT == REIN_TYPE_IQ3_S) {   // iq3_s.rs:186-207: signed odd values -> nibble (v + 15) / 2, fp16(d * (1 + 2*scale))
                const float d = half_to_float(load16(b));
                for (int s = 0; s < 8; s++) {
                    const uint8_t* index = b + 2 + 8 * s;                // eight grid indices, low 8 bits
                    const unsigned high = b[66 + s];                     // their 9th bits
                    const uint32_t sign = load32(b + 74 + 4 * s);        // one bit per weight
                    uint32_t half[2][4];                                 // nibbles of weights 0-15, 16-31, four to a word
                    for (int q = 0; q < 8; q++) {
                        const uint32_t mag = kIq3sNibbles[index[q] | (((high >> q) & 1u) << 8)];
                        // (15 - mag) / 2 for a negative weight is 7 - l, and (15 + mag) / 2 is 8 + l: the complement of 8 + l in four bits
                        half[q / 4][q % 4] = mag ^ (0x0F0F0F0Fu & spread4(sign >> (4 * q)));
                    }
                    for (int j = 0; j < 4; j++) store32(n0 + s * 16 + 4 * j, half[0][j] | (half[1][j] << 4));
                    const int scale = (b[106 + s / 2] >> (4 * (s & 1))) & 15;
                    store16(p1 + (sb + s) * 2, float_to_half(d * (1.0f + 2.0f * (float)scale)));
                }
                b += 110;
            } else if constexpr (FMT == REIN_TYPE_Q4_K || FMT == REIN_TYPE_Q5_K) {   // q4_k.rs:126-176, q5_k.rs:97-151
                constexpr bool q5 = FMT == REIN_TYPE_Q5_K;
                const uint8_t* qs = b + (q5 ? 48 : 16);
                for (int s = 0; s < 8; s += 2, qs += 32) {
                    low_entry(qs, n0 + s * 16);
                    high_entry(qs, n0 + s * 16 + 16);
                }
                if constexpr (q5) {                    // byte j: fifth bits of weights 4j.. and 16 + 4j.. (q5_k.rs:122-141)
                    for (int s = 0; s < 8; s++) {
                        uint32_t qh = 0;
                        for (int j = 0; j < 4; j++)
                            qh |= (gather1(load32(b + 16 + 4 * j) >> s) | (gather1(load32(b + 32 + 4 * j) >> s) << 4)) << (8 * j);
                        store32(p1 + (sb + s) * 4, qh);
                    }
                }
                scales_k4(b + 4, (q5 ? p2 : p1) + sb * 2);
                std::memcpy(ps + sb / 8 * 4, b, 4);
                b += q5 ? 176 : 144;
            } else {                                   // Q6_K (q6_k.rs:86-148)
                for (int chunk = 0; chunk < 2; chunk++) {
                    const uint8_t *ql = b + chunk * 64, *qh = b + 128 + chunk * 32;
                    uint8_t* o = n0 + chunk * 64;
                    low_entry(ql, o);
                    low_entry(ql + 32, o + 16);
                    high_entry(ql, o + 32);
                    high_entry(ql + 32, o + 48);
                    // byte g = the four 2-bit fields of dot group g (q6_k.rs:128-138)
                    for (int quad = 0; quad < 4; quad++) {
                        uint8_t* h2 = p1 + (sb + chunk * 4 + quad) * 8;
                        for (int j = 0; j < 4; j++) {
                            h2[2 * j]     = (uint8_t)gather2(load32(qh + 4 * j) >> (2 * quad));
                            h2[2 * j + 1] = (uint8_t)gather2(load32(qh + 16 + 4 * j) >> (2 * quad));
                        }
                    }
                }
                std::memcpy(p2 + sb * 2, b + 192, 16);
                std::memcpy(ps + sb / 8 * 2, b + 208, 2);
                b += 210;
            }
        }
    }
}

using RowFn = void (*)(const uint8_t*, size_t, uint8_t* const*, uint8_t*);
RowFn row_fn(int fmt)
{
    switch (fmt) {
    case REIN_TYPE_Q4_0:   return repack_row<REIN_TYPE_Q4_0>;
    case REIN_TYPE_Q8_0:   return repack_row<REIN_TYPE_Q8_0>;
    case REIN_TYPE_Q4_K:   return repack_row<REIN_TYPE_Q4_K>;
    case REIN_TYPE_Q5_K:   return repack_row<REIN_TYPE_Q5_K>;
    case REIN_TYPE_Q6_K:   return repack_row<REIN_TYPE_Q6_K>;
    case REIN_TYPE_IQ4_XS: return repack_row<REIN_TYPE_IQ4_XS>;
    case REIN_TYPE_Q5_1:   return repack_row<REIN_TYPE_Q5_1>;
    default:               return repack_row<REIN_TYPE_IQ3_S>;
    }
}

void repack_range(int fmt, const Layout& l, size_t row_bytes, uint8_t* dst, rein::RowSource source, const void* ctx, bool staged,
                  size_t row_begin, size_t row_end)
{
    const RowFn fn = row_fn(fmt);
    std::vector<uint8_t> staging(staged ? row_bytes : 0);
    for (size_t row = row_begin; row < row_end; row++) {
        uint8_t *p[4], *at = dst;
        for (int i = 0; i < 4; i++) {
            p[i] = at + row * l.nsp * l.entry[i];
            at += l.n_rows * l.nsp * l.entry[i];
        }
        fn(source(ctx, row, staging.data()), l.n_sub, p, at + row * l.n_super * l.super);
        for (int i = 0; i < 4 && l.nsp > l.n_sub; i++) std::memset(p[i] + l.n_sub * l.entry[i], 0, l.entry[i]);
    }
}

}  // namespace

// The output is the larger part of the traffic and, in a buffer that a loader has just allocated, is touched here for the
// first time: each thread writes its rows (and zeroes their padding) itself, so the kernel hands out and clears the pages
// of all threads at once.  A pass that zeroed the slab before the threads started was most of the call (Q4_K 5120 x 17408,
// 50 MB in and out, sixteen threads of the GPU host: 9.7 ms with it and a byte at a time, 1.1 ms now).  A thread is worth
// its start from about a million weights on.
void rein::repack_parallel(int fmt, size_t in_dim, size_t out_dim, uint8_t* dst, RowSource source, const void* ctx, bool staged)
{
    Geometry g;
    geometry(fmt, &g);
    const Layout l = layout_of(fmt, g, in_dim, out_dim);
    const size_t row_bytes = in_dim / (size_t)g.block * (size_t)g.bytes;
    size_t n_threads = std::min<size_t>(std::max(1u, std::thread::hardware_concurrency()), 16);
    n_threads = std::max<size_t>(1, std::min({n_threads, in_dim * out_dim >> 20, out_dim}));
    std::vector<std::thread> pool;
    const size_t step = (out_dim + n_threads - 1) / n_threads;
    size_t next = step;
    try {
        pool.reserve(n_threads);
        for (; next < out_dim; next += step)
            pool.emplace_back(repack_range, fmt, std::cref(l), row_bytes, dst, source, ctx, staged, next, std::min(out_dim, next + step));
    } catch (const std::exception&) {                // no more threads to be had: the calling one does the rows that are left
    }
    repack_range(fmt, l, row_bytes, dst, source, ctx, staged, 0, std::min(out_dim, step));
    if (next < out_dim) repack_range(fmt, l, row_bytes, dst, source, ctx, staged, next, out_dim);
    for (auto& th : pool) th.join();
}

extern "C" {

size_t rein_repacked_n_sub_padded(size_t in_dim)
{
    const size_t n = in_dim / 32;
    return (n != 0 && (n & (n - 1)) == 0) ? n + 1 : n;
}

size_t rein_repacked_len(int fmt, size_t in_dim, size_t out_dim)
{
    Geometry g;
    if (!geometry(fmt, &g)) return 0;
    return out_dim * rein_repacked_n_sub_padded(in_dim) * g.per_sub + out_dim * (in_dim / 256) * g.per_super;
}

int rein_block_size(int fmt)
{
    Geometry g;
    return geometry(fmt, &g) ? g.block : 0;
}

int rein_bytes_per_block(int fmt)
{
    Geometry g;
    return geometry(fmt, &g) ? g.bytes : 0;
}

int rein_repack_for_matvec(int fmt, const uint8_t* src, size_t in_dim, size_t out_dim, uint8_t* dst)
{
    Geometry g;
    if (!geometry(fmt, &g)) return rein::fail(REIN_E_BAD_FORMAT, "rein_repack_for_matvec: unknown format " + std::to_string(fmt));
    if (in_dim == 0 || in_dim % (size_t)g.block != 0)
        return rein::fail(REIN_E_BAD_SHAPE, "rein_repack_for_matvec: in_dim must be a non-zero multiple of " + std::to_string(g.block));
    if (!src || !dst) return rein::fail(REIN_E_BAD_POINTER, "rein_repack_for_matvec: null pointer");
    const struct { const uint8_t* src; size_t row_bytes; } rows = {src, in_dim / (size_t)g.block * (size_t)g.bytes};
    rein::repack_parallel(fmt, in_dim, out_dim, dst,
                          [](const void* ctx, size_t row, uint8_t*) {
                              const auto* r = static_cast<const decltype(rows)*>(ctx);
                              return r->src + row * r->row_bytes;
                          }, &rows, false);
    return 0;
}

}  // extern "C"
