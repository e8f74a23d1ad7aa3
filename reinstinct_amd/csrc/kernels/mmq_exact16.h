// Prefill GEMM for Q4_K, Q5_K and Q6_K on the fp16 matrix instruction with exact block dots.
//
// The int8 tile (mmq_gemm.h) leaves a conversion, a scale outer product and a multiply-add per output element and 32-weight
// sub-block on the vector ALU, and for Q6_K a second matrix instruction per sub-block with half of its operand zeroed plus an
// integer combine.  Here the integer scale of a sub-block goes into the weight operand and stays exact:
//   Q4_K  q * sc               4 + 6 bits, at most 945: one fp16 number
//   Q5_K  q * sc               5 + 6 bits, at most 1953: one
//   Q6_K  (q - 32) * sc / 4  = n * sc / 4  +  4 * (c - 2) * sc     n the nibble, c the two high bits, q = n + 16 c: both
//                              terms are integers of at most 11 bits times a power of two, so each is one fp16 number, and
//                              the two are two operands of the same accumulation
// and the activations are their int8 quants as fp16.  v_mfma_f32_32x32x16_f16 multiplies exactly and every partial sum is an
// integer (times 1/4) below 2^24, so the fp32 result IS the integer dot of the sub-block with its scale: no rounding, nothing
// to convert.  With the weights as rows of the tile (register = weight row, lane = token) the activation scale is one number
// per lane: per sub-block and element the vector ALU does s1 += dx * dot, per 256 weights acc += d * s1 -- the products and
// sums that the int8 tile makes in fp32, fewer of them.  The minimum term of Q4_K and Q5_K is the int8 tile's: bf16 instructions on
// the three-way bf16 split of xsum (24 bits) against the integer minimums, scaled by -dmin.
//
// A wavefront owns 32 weight rows x 32 NT tokens (the unpack of a weight is shared by NT tiles), a workgroup of four 128 rows x
// 32 NT tokens: NT two to four, two workgroups per CU (rein_xh_*), or one and two, three per CU (rein_xf_*: one tile leaves
// registers and LDS for the third, which fills the waits of the others' short steps; Q4_K 64 x 5120 -> 17408 45 -> 40 us).
//
// Bound: the same instructions alone, on every CU, take 65 ns (Q4_K) and 90 (Q6_K) per tile and sub-block and SIMD -- two / four matrix
// instructions, the 16 multiply-adds and a quarter of the unpack, the two units overlapping but for issue, the clock at 1.8-2.0 of
// 2.4 GHz under this load; the kernel takes 88 and 118.  Without its transfers it is 14 % faster (Q4_K 17 %), with the activations
// always from one place in cache 3-7 %: what is left is the way from L2 to LDS and the scalar issue around it.  Waits, barriers and
// the operand reads from LDS cost nothing measurable.  Whole calls of rein_matmul_ws against the launches of rein_mmq_xq8_ws (fp6 for
// Q4_K, else int8), both on one card, three inputs and the weights of several matrices in turn, us, Q4_K / Q5_K / Q6_K: 2048 x 5120 -> 17408 569 / 715 /
// 1066 -> 511 / 552 / 676; 512 x 5120 -> 17408 148 / 192 / 292 -> 138 / 150 / 183; 777 x 17408 -> 5120 Q6_K 492 -> 325; 45 x 17408 -> 5120 (one group of
// two tiles) Q5_K 44.5 -> 38.0.  Other cards are up to 7 % off (777 rows 328 to 343).  The figures beside single choices below have both sides from one
// card and one session each; they do not add up over sessions.
//
// Replaces, from nine rows, kernels/mmq_gemm_{q4k,q5k,q6k}_repacked.cpp of the reference behind rein_matmul_ws.
#pragma once

#include "mmq_fp6.h"

typedef _Float16 rein_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 rein_v8h __attribute__((ext_vector_type(8)));

// HBM -> LDS transfers of a dword / a 16-bit word per lane (which lands as a dword, zero-extended), scalar base + lane offset
__device__ __forceinline__ void rein_xh_dma_u32(unsigned voff, const void* sbase, unsigned lds_base)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_base) : "memory", "m0");
}
__device__ __forceinline__ void rein_xh_dma_u16(unsigned voff, const void* sbase, unsigned lds_base)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_ushort %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_base) : "memory", "m0");
}

// ---- operand slot order ---------------------------------------------------------------
// An instruction contracts 16 slots; lane half h holds slots 8h .. 8h+7 of both operands.  The two instructions kh = 0, 1 of
// a sub-block take word 2h + kh of its 16-byte nibble entry (low nibble of byte f: weight 4 (2h + kh) + f, high nibble 16 more),
// in the order in which the masks below produce them.
__host__ __device__ constexpr int rein_xh_slot_weight(int kh, int h, int e)
{
    constexpr int t[8] = {0, 2, 16, 18, 1, 3, 17, 19};
    return 4 * (2 * h + kh) + t[e];
}

// ---- activation image -----------------------------------------------------------------
//   records  [superblock][32-token tile] of 17408 bytes: [sub-block][kh][lane = 32 h + token][8 x fp16], then dx [sub-block][token] fp32
//   xsum     [superblock][32-token tile] of 2048 bytes: [op][lane][8 x bf16]: lane halves 0 / 1 of op 0 the first and second
//            bf16 of the 8 sub-blocks' xsum, half 0 of op 1 the third, half 1 zeros
#define REIN_XH_PAIR 4096u
#define REIN_XH_X    16384u
#define REIN_XH_REC  17408u
#define REIN_XH_DX   1024u
#define REIN_XH_XS   2048u
struct XhImage {
    uint8_t *rec, *xs;
    unsigned n_tt;
    __device__ __forceinline__ XhImage(uint8_t* img, unsigned in_dim, unsigned n_tt) : rec(img), xs(img + (size_t)(in_dim >> 8) * n_tt * REIN_XH_REC), n_tt(n_tt) {}
};

// A block of 32 values of row `tok` (zeros past p_rows, with d = 0) with the numbers that quantize_q8_f32 gives, by four lanes: lane q of
// the four holds values 4 q .. 4 q + 3 and those 16 further on, which are the two dwords of quants that it writes to xq and one 16-byte
// piece of the operand order.  The sum tree is halves of 16 (inside the lane), 8 and 4 (between lanes), 2 and 1.
struct XhBlock { float d, sum; int q[8]; };
__device__ __forceinline__ void rein_xh_quantize_values(XhBlock& b, const float (&v)[8])
{
#pragma clang fp contract(off)
    float t[4], amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(v[i]));
    amax = fmaxf(amax, rein_dpp_f32<0x4E>(amax, amax));                  // lane ^ 2
    amax = fmaxf(amax, rein_dpp_f32<0xB1>(amax, amax));                  // lane ^ 1
#pragma unroll
    for (int i = 0; i < 4; i++) t[i] = v[i] + v[i + 4];
#pragma unroll
    for (int i = 0; i < 4; i++) t[i] = t[i] + rein_dpp_f32<0x4E>(t[i], t[i]);
#pragma unroll
    for (int i = 0; i < 4; i++) t[i] = t[i] + rein_dpp_f32<0xB1>(t[i], t[i]);
    b.sum = (t[0] + t[2]) + (t[1] + t[3]);
    b.d   = amax > 0.0f ? amax / 127.0f : 1.0f;
    const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) b.q[i] = max(-127, min(127, (int)rintf(v[i] * inv)));
}
// values 4 q .. 4 q + 3 and 16 further on of block sb of a row
__device__ __forceinline__ void rein_xh_load_values(float (&v)[8], const float* __restrict__ row, unsigned sb, unsigned q, bool aligned)
{
    const float* p = row + sb * 32u + 4u * q;
    if (aligned) {
        const float4 lo = reinterpret_cast<const float4*>(p)[0], hi = reinterpret_cast<const float4*>(p)[4];
        v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
        v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) { v[i] = p[i]; v[4 + i] = p[16 + i]; }
    }
}
// a lane's dword of the first (k = 0) or second sixteen quants
__device__ __forceinline__ uint32_t rein_xh_word(const XhBlock& b, int k)
{
    return (b.q[4 * k] & 0xFF) | (b.q[4 * k + 1] & 0xFF) << 8 | (b.q[4 * k + 2] & 0xFF) << 16 | (uint32_t)b.q[4 * k + 3] << 24;
}
__device__ __forceinline__ void rein_xh_quantize_block(XhBlock& b, const float* __restrict__ x, BlockQ8* __restrict__ xq, unsigned in_dim, unsigned p_rows,
                                                       unsigned tok, unsigned sb, unsigned q)
{
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = 0.0f;
    if (tok < p_rows) rein_xh_load_values(v, x + (size_t)tok * in_dim, sb, q, ((size_t)x & 15u) == 0u);
    rein_xh_quantize_values(b, v);
    if (tok >= p_rows) b.d = 0.0f;
    if (tok < p_rows) {
        BlockQ8* const o = xq + (size_t)tok * (in_dim >> 5) + sb;
        if (q == 0u) { o->d = b.d; o->xsum = b.sum; }
#pragma unroll
        for (int k = 0; k < 2; k++) o->qs[4 * k + q] = rein_xh_word(b, k);
    }
}

// A block's piece of the image: sub-block sb of token j of a tile
__device__ __forceinline__ void rein_xh_store_block(const XhImage& img, const XhBlock& b, unsigned tile, unsigned sb, unsigned j, unsigned q)
{
    uint8_t* const rec = img.rec + ((size_t)(sb >> 3) * img.n_tt + tile) * REIN_XH_REC;
    if (q == 0u) reinterpret_cast<float*>(rec + REIN_XH_X)[(sb & 7u) * 32u + j] = b.d;
    const unsigned kh = q & 1u, h = q >> 1;          // words 2 h + kh
    rein_v8h o;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        constexpr int part[8] = {0, 0, 4, 4, 0, 0, 4, 4};
        o[e] = (_Float16)b.q[part[e] + (rein_xh_slot_weight(0, 0, e) & 3)];
    }
    *reinterpret_cast<rein_v8h*>(rec + (sb & 7u) * 2048u + kh * 1024u + (32u * h + j) * 16u) = o;
}
// The first to third bf16 of two sub-blocks' xsum as the word of operand `op` for lane half hh
__device__ __forceinline__ uint32_t rein_xh_xsum_word(float s0, float s1, unsigned op, unsigned hh)
{
    uint16_t a[3], b[3];
    rein_mmq_split_xsum(s0, a);
    rein_mmq_split_xsum(s1, b);
    const unsigned k = op ? 2u : hh;
    const uint32_t x0 = k == 2u ? a[2] : k ? a[1] : a[0], x1 = k == 2u ? b[2] : k ? b[1] : b[0];
    return op && hh ? 0u : x0 | x1 << 16;
}

// x [p_rows][in_dim] fp32 -> image, and the blocks themselves to xq [p_rows][in_dim / 32] (the caller of rein_matmul_ws may read
// them there).  blockIdx.x = eight tokens, blockIdx.y = superblock, 256 threads, four to a block of 32: a wavefront reads 512 bytes of
// four rows and writes runs of 64 bytes to the image and 160 to xq (eight rows of 256 bytes, or two of 1024: 2048 x 5120 17.2 -> 17.7 us).
// Bound by memory from a few hundred rows on: 4 bytes in, 3.4 out per value (777 x 17408: 54 + 46 MB); below, by the latency of a load and of
// what a thread does with it, which is why a block has four (a thread a block: 30 x 5120 4.0 us instead of 2.9).
struct XhQuantize { unsigned q, j, tok, sb; };
__device__ __forceinline__ XhQuantize rein_xh_quantize_who()             // j: the token in its tile
{
    const unsigned l = threadIdx.x & 63u, w = threadIdx.x >> 6, tok = blockIdx.x * 8u + (w >> 1) * 4u + (l >> 4);
    return XhQuantize{l & 3u, tok & 31u, tok, blockIdx.y * 8u + (w & 1u) * 4u + ((l >> 2) & 3u)};
}
__device__ __forceinline__ void rein_xh_quantize_body(const float* __restrict__ x, uint8_t* __restrict__ img, BlockQ8* __restrict__ xq, unsigned in_dim,
                                                      unsigned p_rows, unsigned with_xsum)
{
    __shared__ float xsum[8][9];
    const XhQuantize w = rein_xh_quantize_who();
    const XhImage image(img, in_dim, (p_rows + 31u) / 32u);
    const unsigned tt = w.tok >> 5;
    XhBlock b;
    rein_xh_quantize_block(b, x, xq, in_dim, p_rows, w.tok, w.sb, w.q);
    rein_xh_store_block(image, b, tt, w.sb, w.j, w.q);
    if (!with_xsum) return;                          // the image of a format without minimums has no xsum part
    if (w.q == 0u) xsum[w.sb & 7u][w.tok & 7u] = b.sum;
    __syncthreads();
    if (threadIdx.x < 32u) {                         // [op][lane half][token]
        const unsigned op = threadIdx.x >> 4, hh = (threadIdx.x >> 3) & 1u, j = (blockIdx.x * 8u + (threadIdx.x & 7u)) & 31u;
        uint32_t o3[4];
#pragma unroll
        for (int k = 0; k < 4; k++) o3[k] = rein_xh_xsum_word(xsum[2 * k][threadIdx.x & 7u], xsum[2 * k + 1][threadIdx.x & 7u], op, hh);
        uint8_t* dst = image.xs + ((size_t)blockIdx.y * image.n_tt + tt) * REIN_XH_XS;
        *reinterpret_cast<uint4*>(dst + op * 1024u + (32u * hh + j) * 16u) = make_uint4(o3[0], o3[1], o3[2], o3[3]);
    }
}

// Token tiles are dealt evenly over the n_grp groups of the launch (at least ceil(tiles / 4), at most one per tile): 25 tiles in
// seven groups are four of 4 and three of 3, not six of 4 and one of 1.
struct XhGroup { unsigned tile, n; };
__device__ __forceinline__ XhGroup rein_xh_group(unsigned p_rows, unsigned n_grp, unsigned g)
{
    const unsigned n_tt = (p_rows + 31u) >> 5, base = n_tt / n_grp, more = n_tt - base * n_grp;
    return XhGroup{g * base + min(g, more), base + (g < more ? 1u : 0u)};
}

// Partial tiles of unit (rb, group g) of the ones that are cut: ranges one after the other, the tiles of a range together, units in
// order from the first that is cut.
__device__ __forceinline__ size_t rein_xh_part(unsigned p_rows, unsigned n_grp, unsigned n_whole, unsigned rb, const XhGroup& g, unsigned split)
{
    const unsigned n_tt = (p_rows + 31u) >> 5, rb0 = n_whole / n_grp, tile0 = rein_xh_group(p_rows, n_grp, n_whole - rb0 * n_grp).tile;
    return ((size_t)(rb - rb0) * n_tt + g.tile - tile0) * split * 4096u;
}

// ---- weight operands ------------------------------------------------------------------
// A nibble or-ed into the mantissa of 1024 (low nibble) or 64 (high nibble, which sits four bits up) is 1024 + n or 64 + n;
// one packed fma with the scale takes the offset out again, exactly: (1024 + n) sc - 1024 sc.
// (v & mask) | base as one instruction, which takes one constant out of a scalar register and needs the other in a vector one
struct XhMasks {
    uint32_t lo, hi, two;                            // low nibbles, high nibbles, bits 8, 9 of both halves
    __device__ __forceinline__ XhMasks() : lo(0x000F000Fu), hi(0x00F000F0u), two(0x03000300u)
    {
        asm volatile("" : "+v"(lo), "+v"(hi), "+v"(two));
    }
};
__device__ __forceinline__ uint32_t rein_xh_or(uint32_t v, uint32_t mask, uint32_t base) { return (v & mask) | base; }
__device__ __forceinline__ rein_h2 rein_xh_fma(uint32_t v, rein_h2 sc, rein_h2 c) { return __builtin_elementwise_fma(__builtin_bit_cast(rein_h2, v), sc, c); }
// (as an operand of a packed instruction: its half of a register, no copy)
__device__ __forceinline__ rein_h2 rein_xh_both(_Float16 v) { return rein_h2{v, v}; }
__device__ __forceinline__ rein_v8h rein_xh_join(rein_h2 a, rein_h2 b, rein_h2 c, rein_h2 d)
{
    return rein_v8h{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

template <int FMT> struct XhWeights;

template <> struct XhWeights<REIN_Q4_K> {
    static constexpr int kOps = 1;                   // operands per instruction position
    static constexpr bool kHasMin = true;
    static constexpr float kUnit = 1.0f;             // what the operands were divided by
    // plane of extra bits: bytes per sub-block (0: none); plane of the superblocks' scales
    static constexpr unsigned kHiBytes = 0, kDBytes = 4;
    static __device__ __forceinline__ const char* hi(const Fmt<REIN_Q4_K>&) { return nullptr; }
    static __device__ __forceinline__ const char* d(const Fmt<REIN_Q4_K>& f) { return reinterpret_cast<const char*>(f.ddp); }
    static __device__ __forceinline__ float scale(uint32_t dd) { return rein_h2f((uint16_t)(dd & 0xFFFFu)); }
    static __device__ __forceinline__ float min_scale(uint32_t dd) { return -rein_h2f((uint16_t)(dd >> 16)); }
    // words 2h, 2h + 1 of a sub-block's nibbles and its (sc, m)
    static __device__ __forceinline__ void unpack(rein_v8h (&o)[2][kOps], uint2 w2, uint32_t, uint32_t sm, unsigned, const XhMasks& mk)
    {
        const rein_h2 sc = rein_xh_both((_Float16)(uint16_t)(sm & 0xFFu)), c = sc * rein_h2{(_Float16)-1024.0f, (_Float16)-64.0f};
        const rein_h2 c1024 = rein_xh_both(c[0]), c64 = rein_xh_both(c[1]);
#pragma unroll
        for (int kh = 0; kh < 2; kh++) {
            const uint32_t w = kh ? w2.y : w2.x, w8 = w >> 8;
            o[kh][0] = rein_xh_join(rein_xh_fma(rein_xh_or(w, mk.lo, 0x64006400u), sc, c1024), rein_xh_fma(rein_xh_or(w, mk.hi, 0x54005400u), sc, c64),
                                    rein_xh_fma(rein_xh_or(w8, mk.lo, 0x64006400u), sc, c1024), rein_xh_fma(rein_xh_or(w8, mk.hi, 0x54005400u), sc, c64));
        }
    }
};

template <> struct XhWeights<REIN_Q5_K> {
    static constexpr int kOps = 1;
    static constexpr bool kHasMin = true;
    static constexpr float kUnit = 1.0f;
    static constexpr unsigned kHiBytes = 4, kDBytes = 4;
    static __device__ __forceinline__ const char* hi(const Fmt<REIN_Q5_K>& f) { return reinterpret_cast<const char*>(f.qhp); }
    static __device__ __forceinline__ const char* d(const Fmt<REIN_Q5_K>& f) { return reinterpret_cast<const char*>(f.ddp); }
    static __device__ __forceinline__ float scale(uint32_t dd) { return rein_h2f((uint16_t)(dd & 0xFFFFu)); }
    static __device__ __forceinline__ float min_scale(uint32_t dd) { return -rein_h2f((uint16_t)(dd >> 16)); }
    // words 2h, 2h + 1 of a sub-block's nibbles, its fifth bits and (sc, m)
    static __device__ __forceinline__ void unpack(rein_v8h (&o)[2][kOps], uint2 w2, uint32_t qh, uint32_t sm, unsigned h, const XhMasks& mk)
    {
        const rein_h2 sc = rein_xh_both((_Float16)(uint16_t)(sm & 0xFFu)), c = sc * rein_h2{(_Float16)-1024.0f, (_Float16)-64.0f};
        const rein_h2 c1024 = rein_xh_both(c[0]), c64 = rein_xh_both(c[1]);
        const uint32_t q = qh >> (16u * h), q2 = q >> 2;      // bits f of byte kh: weights f of the low nibbles, bits 4 + f: of the high
#pragma unroll
        for (int kh = 0; kh < 2; kh++) {
            const uint32_t w = kh ? w2.y : w2.x, w8 = w >> 8;
            // byte kh with elements 0, 1 in the low half, elements 2, 3 in the high half
            const uint32_t p = __builtin_amdgcn_perm(q2, q, kh ? 0x0C050C01u : 0x0C040C00u), p4 = p << 4, p3 = p << 3;
            const uint32_t r0 = rein_xh_or(p4, 0x00100010u, rein_xh_or(w, mk.lo, 0x64006400u));
            const uint32_t r1 = rein_xh_or(p4, 0x01000100u, rein_xh_or(w, mk.hi, 0x54005400u));
            const uint32_t r2 = rein_xh_or(p3, 0x00100010u, rein_xh_or(w8, mk.lo, 0x64006400u));
            const uint32_t r3 = rein_xh_or(p3, 0x01000100u, rein_xh_or(w8, mk.hi, 0x54005400u));
            o[kh][0] = rein_xh_join(rein_xh_fma(r0, sc, c1024), rein_xh_fma(r1, sc, c64), rein_xh_fma(r2, sc, c1024), rein_xh_fma(r3, sc, c64));
        }
    }
};

template <> struct XhWeights<REIN_Q6_K> {
    static constexpr int kOps = 2;
    static constexpr bool kHasMin = false;
    static constexpr float kUnit = 4.0f;
    static constexpr unsigned kHiBytes = 8, kDBytes = 2;
    static __device__ __forceinline__ const char* hi(const Fmt<REIN_Q6_K>& f) { return reinterpret_cast<const char*>(f.h2p); }
    static __device__ __forceinline__ const char* d(const Fmt<REIN_Q6_K>& f) { return reinterpret_cast<const char*>(f.dp); }
    static __device__ __forceinline__ float scale(uint32_t dd) { return rein_h2f((uint16_t)dd); }
    static __device__ __forceinline__ float min_scale(uint32_t) { return 0.0f; }
    // Words 2h, 2h + 1 of a sub-block's nibbles, the word of two-bit fields that goes with them, both group scales.  Low nibbles
    // are weights 0..15 (first scale), high ones 16..31 (second).  Or-ed into the mantissas of 256 and 16 they are 256 + n / 4 and
    // 16 + n / 4, a two-bit field at bits 8, 9 of 16 is 16 + 4 c: one packed fma with the scale itself and an offset of it makes
    // n sc / 4 and 4 (c - 2) sc, and the offsets (256, 16, 24 times a scale of 8 bits) are exact.  The quarter is taken back at the
    // end.  (With scales multiplied by 1/4 and 4 first it is eight conversions and twelve products a sub-block instead of two and two:
    // 2048 x 5120 -> 17408 739 -> 719 us.)
    static __device__ __forceinline__ void unpack(rein_v8h (&o)[2][kOps], uint2 w2, uint32_t hw, uint32_t sm, unsigned, const XhMasks& mk)
    {
        const rein_h2 sc = {(_Float16)(short)(int8_t)(sm & 0xFFu), (_Float16)(short)(int8_t)((sm >> 8) & 0xFFu)};
        const rein_h2 cn = sc * rein_h2{(_Float16)-256.0f, (_Float16)-16.0f}, cg = sc * rein_h2{(_Float16)-24.0f, (_Float16)-24.0f};
        const rein_h2 a = rein_xh_both(sc[0]), b = rein_xh_both(sc[1]), ca = rein_xh_both(cn[0]), cb = rein_xh_both(cn[1]);
        const rein_h2 ga = rein_xh_both(cg[0]), gb = rein_xh_both(cg[1]);
        const uint32_t hw4 = hw >> 4;
#pragma unroll
        for (int kh = 0; kh < 2; kh++) {
            const uint32_t w = kh ? w2.y : w2.x, w8 = w >> 8;
            o[kh][0] = rein_xh_join(rein_xh_fma(rein_xh_or(w, mk.lo, 0x5C005C00u), a, ca), rein_xh_fma(rein_xh_or(w, mk.hi, 0x4C004C00u), b, cb),
                                    rein_xh_fma(rein_xh_or(w8, mk.lo, 0x5C005C00u), a, ca), rein_xh_fma(rein_xh_or(w8, mk.hi, 0x4C004C00u), b, cb));
            // byte 2 kh (weights of the low nibbles) / 2 kh + 1 (of the high ones): elements 0, 1 to bits 8..11, 2, 3 to bits 24..27
            const uint32_t pa = __builtin_amdgcn_perm(hw4, hw, kh ? 0x060C020Cu : 0x040C000Cu), pa2 = pa >> 2;
            const uint32_t pb = __builtin_amdgcn_perm(hw4, hw, kh ? 0x070C030Cu : 0x050C010Cu), pb2 = pb >> 2;
            o[kh][1] = rein_xh_join(rein_xh_fma(rein_xh_or(pa, mk.two, 0x4C004C00u), a, ga), rein_xh_fma(rein_xh_or(pb, mk.two, 0x4C004C00u), b, gb),
                                    rein_xh_fma(rein_xh_or(pa2, mk.two, 0x4C004C00u), a, ga), rein_xh_fma(rein_xh_or(pb2, mk.two, 0x4C004C00u), b, gb));
        }
    }
};

// Sums tied to this point of the program: instruction selection otherwise moves them past the scheduling fences
__device__ __forceinline__ void rein_xh_pin(float (&s)[16])
{
    asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(s[4]), "+v"(s[5]), "+v"(s[6]), "+v"(s[7]));
    asm volatile("" : "+v"(s[8]), "+v"(s[9]), "+v"(s[10]), "+v"(s[11]), "+v"(s[12]), "+v"(s[13]), "+v"(s[14]), "+v"(s[15]));
}

// ---- the tile -------------------------------------------------------------------------
// LDS of one workgroup:
//   acts  2 x MOST x 4096  records of two consecutive sub-block pairs
//   dx    2 x MOST x 1024  activation scales of two superblocks
//   ring  4 x 2 x 2048     per wavefront: two slots of 4 sub-blocks x 32 rows x 16 B
//   small 4 x              per wavefront: extra bits of a superblock [row][sub-block] in granules of 16 bytes, rotated; (sc, m) or both
//                          group scales of two superblocks, 48 bytes a row; the scale words of four [row][superblock] in a dword each
//   xs    MOST x 2048      xsum operands of a superblock (formats with minimums)
// MOST: tiles of the launch's largest group, 4 (80 KB: two workgroups to a CU) or (rein_xf_*) 2 (52 KB: three).
template <int FMT, unsigned MOST> struct XhLds {
    static constexpr unsigned kAct = MOST * REIN_XH_PAIR, kDx = 2u * kAct, kRing = kDx + 2u * MOST * REIN_XH_DX, kSmall = kRing + 4u * 4096u;
    static constexpr unsigned kSm = 256u * XhWeights<FMT>::kHiBytes, kD = kSm + 1536u, kWave = kD + 512u, kXs = kSmall + 4u * kWave;
    static constexpr unsigned kBytes = kXs + (XhWeights<FMT>::kHasMin ? MOST * REIN_XH_XS : 0u);
    static_assert(kBytes <= (MOST == 2u ? 54272u : 81920u), "LDS for three workgroups to a CU, or two");
};

// Superblocks [c0, c1) of the wavefront's 32 rows from row_base on and the NT token tiles from `tile` on, into acc.  One barrier per sub-block
// pair: at its top everything in flight has landed (it was issued a whole pair earlier: 8 NT or 16 NT matrix instructions per
// wavefront), behind it the next pair's transfers go out.
template <int FMT, int NT, unsigned MOST>
__device__ __forceinline__ void rein_xh_acc(const uint8_t* __restrict__ w, const uint8_t* __restrict__ img, unsigned in_dim, unsigned out_dim,
                                            unsigned n_tt, unsigned row_base, unsigned tile, unsigned c0, unsigned c1, unsigned char* const raw, float (&acc)[NT][16])
{
    using W = XhWeights<FMT>;
    typedef __attribute__((address_space(3))) const void* lptr_t;
    using L = XhLds<FMT, MOST>;
    const unsigned lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 31u, h = lane >> 5;
    const unsigned n_sub = in_dim >> 5;
    const Fmt<FMT> fmt(w, n_sub, out_dim);
    const unsigned first = min(row_base, out_dim - 1u);
    // rows past the matrix read its last one; offsets from the wavefront's first row
    const unsigned row = min(row_base + j, out_dim - 1u) - first;
    // Transfers of a step go out one by one between the matrix instructions of three and four tiles; with one or two tiles there are
    // too few instructions for that, and they go out at the step's top (spread: Q4_K 60 x 5120 -> 5120 19.9 -> 20.9 us).
    constexpr bool kSpread = NT > 2;
    // Small planes come in long pieces: a transfer occupies a CU's address path for 16 cycles if its 64 lanes are one run, for 23 if they are
    // 16 runs, for 64 if they are 32, however few bytes those are.  A row's superblock of extra bits is four granules (Q6_K) or two
    // (Q5_K), rotated so that the reads of one granule of every row meet every bank.  With one and two tiles, where a weight is used least:
    //   (sc, m)      of two superblocks, three granules from the dword boundary below them on (rows start at two bytes where the slab pads
    //                them): two transfers of 64 granules, the middle third in both.  What that reads behind a row's end is the next row or,
    //                behind the last, up to 32 bytes of the plane of scale words; a matrix that has fewer of those takes its scales word by word.
    //   scale words  of four superblocks, a lane each.
    // (a superblock at a time and by 16-bit words in padded rows: 45 x 17408 -> 5120 Q5_K 35.5 -> 33.8 us, 512 tokens of 128 experts of 2048 x 768,
    // gate + up 105 -> 100).  With three and four tiles the scales of a superblock are one transfer (padded: four) and its scale words another: the
    // branches that the longer pieces need cost more between the matrix instructions (777 x 17408 -> 5120 Q6_K 318 -> 326 us).
    auto row_at = [&](unsigned n) { return min(row_base + n, out_dim - 1u) - first; };
    const unsigned odd = ((first + row) * fmt.nsp * 2u) & 2u;            // of this lane's row
    unsigned hi_off[2] = {0u, 0u}, sm_off[4];
    if constexpr (W::kHiBytes == 8) {
#pragma unroll
        for (unsigned k = 0; k < 2; k++) {
            const unsigned n = 16u * k + (lane >> 2);
            hi_off[k] = row_at(n) * fmt.nsp * 8u + (((lane & 3u) - (n >> 1)) & 3u) * 16u;
        }
    } else if constexpr (W::kHiBytes == 4) {
        hi_off[0] = row_at(lane >> 1) * fmt.nsp * 4u + ((lane ^ (lane >> 3)) & 1u) * 16u;
    }
    const bool padded = (fmt.nsp & 1u) != 0u;
#pragma unroll
    for (unsigned k = 0; k < (kSpread ? 4u : 2u); k++) {
        if constexpr (kSpread) {                     // (unpadded: the upper lanes fetch the rows again)
            sm_off[k] = padded ? (row_at(8u * k + (lane >> 3)) * fmt.nsp + (lane & 7u)) * 2u : row * fmt.nsp * 2u;
        } else {
            const unsigned i = 32u * k + lane, n = i / 3u, r = row_at(n);
            sm_off[k] = r * fmt.nsp * 2u - (((first + r) * fmt.nsp * 2u) & 2u) + (i - 3u * n) * 16u + 2u;      // from two bytes below the plane's place
        }
    }
    const unsigned sm_step = kSpread && padded ? 4u : 2u;


    const uint4* const ring = reinterpret_cast<const uint4*>(raw + L::kRing + wave * 4096u);
    const unsigned char* const small = raw + L::kSmall + wave * L::kWave;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lptr_t)raw);
    MmqWSrc<FMT> wsrc;
    wsrc.init(*reinterpret_cast<const MmqWLds<FMT>*>(ring), fmt, row_base, out_dim, lane);
    const XhImage image(const_cast<uint8_t*>(img), in_dim, n_tt);

    // src: a pair's record of the first tile.  It runs along with the pairs: addresses worked out of the pair's number for each transfer
    // cost as much scalar issue as the transfers do (777 x 17408 -> 5120 Q6_K 328 -> 320 us).
    auto issue_act = [&](const uint8_t* src, unsigned buf, unsigned t) {
        const unsigned at = wave * 1024u;
        rein_lds_dma16_s(lane * 16u, src + t * REIN_XH_REC + at, lds0 + buf * L::kAct + t * REIN_XH_PAIR + at);
    };
    auto issue_dx = [&](unsigned c) {
        if (NT == 4 || wave < (unsigned)NT) rein_lds_dma16_s(lane * 16u, img + ((size_t)c * n_tt + tile + wave) * REIN_XH_REC + REIN_XH_X, lds0 + L::kDx + ((c & 1u) * MOST + wave) * REIN_XH_DX);
    };
    auto issue_xs = [&](unsigned c) {
        if constexpr (W::kHasMin) {
            const uint8_t* src = image.xs + ((size_t)c * n_tt + tile) * REIN_XH_XS;
#pragma unroll
            for (unsigned k = 0; k < 2; k++) {
                const unsigned off = (k * 4u + wave) * 1024u;
                if (k * 4u + wave < 2u * NT) rein_lds_dma16_s(lane * 16u, src + off, lds0 + L::kXs + off);
            }
        }
    };
    const unsigned small_at = lds0 + L::kSmall + wave * L::kWave;
    auto issue_hi = [&](unsigned c) {
        if constexpr (W::kHiBytes != 0) {
            const char* hp = W::hi(fmt) + ((size_t)first * fmt.nsp + c * 8u) * W::kHiBytes;
            rein_lds_dma16_s(hi_off[0], hp, small_at);
            if constexpr (W::kHiBytes == 8) rein_lds_dma16_s(hi_off[1], hp, small_at + 1024u);
        }
    };
    auto issue_sm = [&](unsigned c) {                // of c (and c + 1)
        const char* sp = reinterpret_cast<const char*>(fmt.smp) + ((size_t)first * fmt.nsp + c * 8u) * 2u;
        if constexpr (kSpread) {
            if (padded) {
#pragma unroll
                for (unsigned k = 0; k < 4; k++) rein_xh_dma_u16(sm_off[k], sp, small_at + L::kSm + k * 256u);
            } else {
                rein_lds_dma16_s(sm_off[0], sp, small_at + L::kSm);
            }
        } else if (out_dim * fmt.n_super >= 16u) {
#pragma unroll
            for (unsigned k = 0; k < 2; k++) rein_lds_dma16_s(sm_off[k], sp - 2, small_at + L::kSm + k * 512u);
        } else if (lane < 32u) {
            uint16_t* const to = reinterpret_cast<uint16_t*>(raw + L::kSmall + wave * L::kWave + L::kSm + j * 48u + odd);
            for (unsigned k = 0; k < 16u && c * 8u + k < n_sub; k++) to[k] = fmt.smp[(size_t)(first + row) * fmt.nsp + c * 8u + k];
        }
    };
    // Scale words: of one superblock (in two places, odd and even) where a step has room for a transfer of 32 runs; of four, a lane each, with
    // one and two tiles
    constexpr unsigned kD4 = kSpread ? 1u : 4u;
    const unsigned d_off = row * fmt.n_super * W::kDBytes;
    auto issue_d = [&](unsigned c) {
        const char* dp = W::d(fmt) + ((size_t)first * fmt.n_super + c) * W::kDBytes;
#pragma unroll
        for (unsigned k = 0; k < (kSpread ? 1u : 2u); k++) {
            const unsigned off = kSpread ? d_off : (row_at(16u * k + (lane >> 2)) * fmt.n_super + min(lane & 3u, fmt.n_super - 1u - c)) * W::kDBytes;
            const unsigned to = small_at + L::kD + (kSpread ? c & 1u : k) * 256u;
            if constexpr (W::kDBytes == 4) rein_xh_dma_u32(off, dp, to);
            else rein_xh_dma_u16(off, dp, to);
        }
    };
    // Dots are multiplied by their dx one stage after their instructions went out, two where a stage has two instructions and registers
    // are left: nothing waits for the matrix unit then (Q4_K 2048 x 5120 -> 17408 540 -> 530 us).
    constexpr int kLag = W::kOps == 1 && NT > 2 ? 2 : 1, kBuf = kLag + 1;
    rein_v16f dot[kBuf], z16;
    float s1[NT][16];
    float dx[kBuf];
#pragma unroll
    for (int v = 0; v < 16; v++) z16[v] = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[t][v] = s1[t][v] = 0.0f;
#pragma unroll
    for (int b = 0; b < kBuf; b++) { dot[b] = z16; dx[b] = 0.0f; }

    const size_t src_next = (size_t)n_tt * REIN_XH_REC - 3u * REIN_XH_PAIR;
    const uint8_t* src = img + ((size_t)c0 * n_tt + tile) * REIN_XH_REC;
    __syncthreads();                                 // the LDS may still be read by the caller's previous tile
#pragma unroll
    for (unsigned t = 0; t < (unsigned)NT; t++) issue_act(src, 0u, t);
    issue_dx(c0);
    if (kSpread) issue_d(c0);
    issue_hi(c0);
    issue_sm(c0);
    rein_mmq_wload<FMT>(wsrc, 0u, fmt, c0 * 8u, n_sub);
    const unsigned rot = j >> 1;
    const XhMasks mk;

    for (unsigned c = c0; c < c1; c++) {
        uint32_t mpk[4];                             // the superblock's minimums as bf16
#pragma unroll
        for (unsigned u = 0; u < 4; u++) {
            const unsigned pair = c * 4u + u;
            const bool more = c + 1u < c1;
            if (u < 3u) src += REIN_XH_PAIR;
            else if (more) src += src_next;          // (past the last pair: it again, read by nobody)
            REIN_WAIT_VMCNT(0);
            __syncthreads();
            const unsigned char* const sms = small + L::kSm + (kSpread ? (8u * j + 2u * u) * sm_step : j * 48u + odd + ((c - c0) & 1u) * 16u + 4u * u);
            const uint32_t sm2[2] = {*reinterpret_cast<const uint16_t*>(sms), *reinterpret_cast<const uint16_t*>(sms + sm_step)};
            uint32_t hi2[2] = {0u, 0u};
            if constexpr (W::kHiBytes == 8) {
                const uint4 g = *reinterpret_cast<const uint4*>(small + j * 64u + ((u + rot) & 3u) * 16u);
                hi2[0] = h ? g.y : g.x; hi2[1] = h ? g.w : g.z;
            } else if constexpr (W::kHiBytes == 4) {
                const uint2 g = *reinterpret_cast<const uint2*>(small + j * 32u + (((u >> 1) ^ (j >> 2)) & 1u) * 16u + (u & 1u) * 8u);
                hi2[0] = g.x; hi2[1] = g.y;
            }
            const unsigned buf = (pair & 1u) ^ 1u;
            auto issue_other = [&]() {
                if (u == 0u) {
                    rein_mmq_wload<FMT>(wsrc, 1u, fmt, c * 8u + 4u, n_sub);
                    if (!kSpread && ((c - c0) & 3u) == 0u) issue_d(c);   // read at the end of this superblock and the next three
                }
                if (u == 1u) {
                    issue_xs(c);                     // read at the superblock's end; the barrier of u = 0 freed it
                    if (!kSpread && more) issue_dx(c + 1u);
                }
                if (u == 2u && more) rein_mmq_wload<FMT>(wsrc, 0u, fmt, c * 8u + 8u, n_sub);
                if (u == 3u && more) {
                    if constexpr (!kSpread) __builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0): the reads above have left the buffer
                    if constexpr (kSpread) {         // (any earlier step: 777 x 17408 -> 5120 Q6_K 325 -> 333 us)
                        issue_dx(c + 1u);
                        issue_d(c + 1u);
                    }
                    issue_hi(c + 1u);
                    if (kSpread || ((c - c0) & 1u)) issue_sm(c + 1u);
                }
            };
            if constexpr (!kSpread) {
                if (u < 3u || more) {
#pragma unroll
                    for (unsigned t = 0; t < (unsigned)NT; t++) issue_act(src, buf, t);
                }
                issue_other();
            }
            const unsigned char* const act = raw + (pair & 1u) * L::kAct;
#pragma unroll
            for (unsigned q = 0; q < 2; q++) {
                const unsigned sb = 2u * u + q, s4 = sb & 3u;
                const uint2 w2 = reinterpret_cast<const uint2*>(ring + (u >> 1) * 128u + 4u * j + ((s4 + rot) & 3u))[h];
                rein_v8h a[2][W::kOps];
                const uint32_t sm = sm2[q];
                W::unpack(a, w2, hi2[q], sm, h, mk);
                if constexpr (W::kHasMin) {
                    const uint32_t m = rein_bf16_of_u8(sm >> 8);
                    if (q == 0u) mpk[u] = m; else mpk[u] |= m << 16;
                }
                const float* const dxp = reinterpret_cast<const float*>(raw + L::kDx + (c & 1u) * (MOST * REIN_XH_DX)) + sb * 32u + j;
                const unsigned char* const x = act + q * 2048u + lane * 16u;
                rein_v8h xa[2][2];
                xa[0][0] = *reinterpret_cast<const rein_v8h*>(x);
                xa[0][1] = *reinterpret_cast<const rein_v8h*>(x + 1024u);
                __builtin_amdgcn_sched_barrier(0);
                // While this wavefront has matrix instructions to issue it goes before the SIMD's other one, which then does its
                // unpack and waits under them: Q6_K 17408 -> 5120 at 777 rows 360 -> 351 us, 2048 rows 817 -> 786.
                __builtin_amdgcn_s_setprio(1);
                // Stage t: tile t's dots in the matrix unit, the multiply-adds of the tile before (the last tile of the
                // previous sub-block for t = 0) under them, the next tile's operand reads.  The fences keep the stages as
                // written: left alone, the scheduler starts all tiles at once and spills.
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const int i = (int)(sb * NT) + t, now = i % kBuf;
                    if (t + 1 < NT) {
                        xa[(t + 1) & 1][0] = *reinterpret_cast<const rein_v8h*>(x + (t + 1) * REIN_XH_PAIR);
                        xa[(t + 1) & 1][1] = *reinterpret_cast<const rein_v8h*>(x + (t + 1) * REIN_XH_PAIR + 1024u);
                    }
                    if constexpr (kSpread) {
                        if (q == 0u) issue_act(src, buf, (unsigned)t);
                        if (q == 1u && t == 0) issue_other();
                    }
                    dot[now] = z16;
#pragma unroll
                    for (int k = 0; k < W::kOps; k++) {
                        dot[now] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][k], xa[t & 1][0], dot[now], 0, 0, 0);
                        dot[now] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1][k], xa[t & 1][1], dot[now], 0, 0, 0);
                    }
                    dx[now] = dxp[t * (REIN_XH_DX / 4u)];
                    if (i >= kLag) {
                        const int tp = (i - kLag) % NT, old = (i - kLag) % kBuf;
                        const bool first = i - kLag < NT;                            // the sums' first term of this superblock
#pragma unroll
                        for (int v = 0; v < 16; v++) s1[tp][v] = first ? dx[old] * dot[old][v] : fmaf(dx[old], dot[old][v], s1[tp][v]);
                        rein_xh_pin(s1[tp]);
                    }
                    // the order in a stage: operand reads, then the matrix instructions with the multiply-adds behind them.  Left to
                    // itself the scheduler puts multiply-adds behind the first one of Q6_K, where they wait for the stage before
                    // (777 x 17408 -> 5120 335 -> 330 us).
                    if constexpr (W::kOps == 1 && NT > 2) {
                        __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);
                    }
                    if constexpr (W::kOps == 2) {
                        __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                        __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                __builtin_amdgcn_s_setprio(0);
            }
        }
#pragma unroll
        for (int i = 8 * NT - kLag; i < 8 * NT; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) s1[i % NT][v] = fmaf(dx[i % kBuf], dot[i % kBuf][v], s1[i % NT][v]);
        // acc += d s1 - dmin (m . xsum): register v is weight row 8 (v / 4) + 4 h + v % 4
        const unsigned char* const xb = raw + L::kXs + lane * 16u;
        float dv[16], nv[16];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint32_t* const dw = reinterpret_cast<const uint32_t*>(small + L::kD + (kSpread ? (c & 1u) * 256u : 0u) + (8 * g + 4u * h) * (4u * kD4)) + ((c - c0) & (kD4 - 1u));
#pragma unroll
            for (int v = 0; v < 4; v++) { dv[4 * g + v] = W::scale(dw[kD4 * v]); nv[4 * g + v] = W::min_scale(dw[kD4 * v]); }
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
#pragma unroll
            for (int v = 0; v < 16; v++) acc[t][v] = fmaf(dv[v], s1[t][v], acc[t][v]);
            if constexpr (W::kHasMin) {
                const rein_v8bf m = __builtin_bit_cast(rein_v8bf, make_uint4(mpk[0], mpk[1], mpk[2], mpk[3]));
                rein_v16f s2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m, *reinterpret_cast<const rein_v8bf*>(xb + t * 2048u), z16, 0, 0, 0);
                s2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m, *reinterpret_cast<const rein_v8bf*>(xb + t * 2048u + 1024u), s2, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; v++) acc[t][v] = fmaf(nv[v], s2[v], acc[t][v]);
            }
        }
    }
    if constexpr (W::kUnit != 1.0f) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[t][v] *= W::kUnit;
    }
    REIN_WAIT_VMCNT(0);
}

// kMost / kLeast: tiles of the largest and of the smallest group that the launch may have; kSlots: resident workgroups
template <int FMT, unsigned MOST> struct XhTile {
    static constexpr unsigned kMost = MOST, kLeast = MOST == 2u ? 1u : 2u, kSlots = MOST == 2u ? 768u : 512u;
    template <int NT>
    static __device__ __forceinline__ void run(const uint8_t* __restrict__ w, const uint8_t* __restrict__ img, unsigned in_dim, unsigned out_dim, unsigned n_tt,
                                               unsigned row_base, unsigned tile, unsigned c0, unsigned c1, unsigned char* const raw, float (&acc)[NT][16])
    {
        rein_xh_acc<FMT, NT, MOST>(w, img, in_dim, out_dim, n_tt, row_base, tile, c0, c1, raw, acc);
    }
};

// One piece of the launch: superblocks [c0, c1) of unit (rb, grp), to y or (part not null) to a partial tile
// [t][v / 4][thread] of float4.
template <class Tile, int NT>
__device__ __forceinline__ void rein_xh_piece(const uint8_t* __restrict__ w, const uint8_t* __restrict__ img, float* __restrict__ y, float* __restrict__ part,
                                              unsigned in_dim, unsigned out_dim, unsigned p_rows, unsigned rb, unsigned tile, unsigned c0, unsigned c1,
                                              unsigned char* raw)
{
    float acc[NT][16];
    const unsigned lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 31u, h = lane >> 5;
    Tile::template run<NT>(w, img, in_dim, out_dim, (p_rows + 31u) / 32u, rb * 128u + wave * 32u, tile, c0, c1, raw, acc);
    if (part) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                reinterpret_cast<float4*>(part)[(t * 4 + g) * 256 + threadIdx.x] = make_float4(acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]);
        return;
    }
    const bool wide = (out_dim & 3u) == 0u && ((size_t)y & 15u) == 0u;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const unsigned tok = (tile + t) * 32u + j;
        if (tok >= p_rows) continue;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const unsigned row = rb * 128u + wave * 32u + 8u * g + 4u * h;
            float* o = y + (size_t)tok * out_dim + row;
            if (wide) {
                if (row < out_dim) *reinterpret_cast<float4*>(o) = make_float4(acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]);
            } else {
#pragma unroll
                for (unsigned v = 0; v < 4; v++)
                    if (row + v < out_dim) o[v] = acc[t][4 * g + v];
            }
        }
    }
}

// Units u = (128-row block u / n_grp, token group u % n_grp).  The first n_whole (whole rounds of resident
// workgroups) are one workgroup each; the others are cut into `split` ranges of superblocks, a workgroup each, whose partial tiles
// rein_xh_sum_body adds in range order.  Workgroup i runs on XCD i % 8: neighbouring units and ranges go to one XCD, so the
// token groups of a row block meet its weights in one L2.  Grid: n_whole + 8 ceil((units - n_whole) split / 8).
__device__ __forceinline__ unsigned rein_xh_deal(unsigned i, unsigned n)
{
    const unsigned per = (n + 7u) >> 3, k = i >> 3;
    return k < per ? (i & 7u) * per + k : 0xFFFFFFFFu;
}
// Unit `v` of n_rb x n_grp in the order of the launch: bands of up to four token groups, in a band row block by row block.  An XCD's
// 64 resident workgroups are then 16 row blocks x 4 groups instead of 4 x 16: they share the activations sixteen ways in their L2, and what
// it fetches is halved (a group's activations are 272 bytes a value of the contraction, a row block's weights 72 to 136).  Whole calls of 2048 x 5120
// -> 17408 Q4_K 527 -> 511 us, Q5_K 568 -> 552, Q8_0 506 -> 490, Q6_K 678 -> 676; bands of eight are 2 and 1 % slower (Q4_K, Q8_0).  Band b has the groups b,
// b + n_band, ..., so that the longer groups, which come first, are in all of them.  Units that are cut keep their order, the ranges of
// one side by side: banded, or range by range, 777 x 17408 -> 5120 takes 345 to 360 us instead of 333.
__device__ __forceinline__ unsigned rein_xh_banded(unsigned v, unsigned n_rb, unsigned n_grp)
{
    const unsigned n_band = (n_grp + 3u) / 4u, base = n_grp / n_band, more = n_grp - base * n_band, wide = more * (base + 1u) * n_rb;
    unsigned w = base + 1u, b0 = 0u;
    if (v >= wide) { v -= wide; w = base; b0 = more; }
    const unsigned b = v / (w * n_rb), r = (v - b * w * n_rb) / w;
    return r * n_grp + b0 + b + (v - (b * n_rb + r) * w) * n_band;
}
template <class Tile>
__device__ __forceinline__ void rein_xh_dense(const uint8_t* __restrict__ w, const uint8_t* __restrict__ img, float* __restrict__ y, float* __restrict__ parts,
                                              unsigned in_dim, unsigned out_dim, unsigned p_rows, unsigned n_grp, unsigned n_whole, unsigned split)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char rein_xh_lds[];
    const unsigned n_unit = ((out_dim + 127u) / 128u) * n_grp, n_chunk = in_dim >> 8, rb_whole = n_whole / n_grp;
    unsigned u, c0 = 0u, c1 = n_chunk, k = 0u;
    if (blockIdx.x < n_whole) {
        u = blockIdx.x / Tile::kSlots * Tile::kSlots + rein_xh_deal(blockIdx.x % Tile::kSlots, Tile::kSlots);
        if (u < rb_whole * n_grp) u = rein_xh_banded(u, rb_whole, n_grp);
    } else {
        const unsigned n_seg = (n_unit - n_whole) * split, seg = rein_xh_deal(blockIdx.x - n_whole, n_seg);
        if (seg >= n_seg) return;
        const unsigned tu = seg / split;
        k = seg - tu * split;
        u = n_whole + tu;
        c0 = n_chunk * k / split; c1 = n_chunk * (k + 1u) / split;       // split <= n_chunk: no range is empty
    }
    if (u >= n_unit) return;
    u = __builtin_amdgcn_readfirstlane(u);           // (the divisions above left it in a vector register)
    const unsigned rb = u / n_grp;
    const XhGroup g = rein_xh_group(p_rows, n_grp, u - rb * n_grp);
    float* const part = u >= n_whole && split > 1u ? parts + rein_xh_part(p_rows, n_grp, n_whole, rb, g, split) + (size_t)k * g.n * 4096u : nullptr;
    if (g.n == 2u) { rein_xh_piece<Tile, 2>(w, img, y, part, in_dim, out_dim, p_rows, rb, g.tile, c0, c1, rein_xh_lds); return; }
    if constexpr (Tile::kMost == 4u) {
        if (g.n == 4u) rein_xh_piece<Tile, 4>(w, img, y, part, in_dim, out_dim, p_rows, rb, g.tile, c0, c1, rein_xh_lds);
        else if (g.n == 3u) rein_xh_piece<Tile, 3>(w, img, y, part, in_dim, out_dim, p_rows, rb, g.tile, c0, c1, rein_xh_lds);
    }
    if constexpr (Tile::kLeast == 1u) {
        if (g.n == 1u) rein_xh_piece<Tile, 1>(w, img, y, part, in_dim, out_dim, p_rows, rb, g.tile, c0, c1, rein_xh_lds);
    }
}

// y of the split units.  Grid (units - n_whole, 4 x the tiles of the largest group): blockIdx.y = 4 t + v / 4, 256 threads as in the GEMM.
__device__ __forceinline__ void rein_xh_sum_body(const float* __restrict__ parts, float* __restrict__ y, unsigned out_dim, unsigned p_rows, unsigned n_grp, unsigned n_whole, unsigned split)
{
    const unsigned u = n_whole + blockIdx.x, rb = u / n_grp;
    const XhGroup grp = rein_xh_group(p_rows, n_grp, u - rb * n_grp);
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, j = lane & 31u, h = lane >> 5, t = blockIdx.y >> 2, g = blockIdx.y & 3u;
    const unsigned tok = (grp.tile + t) * 32u + j, row = rb * 128u + wave * 32u + 8u * g + 4u * h;
    if (t >= grp.n || tok >= p_rows) return;
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const float4* src = reinterpret_cast<const float4*>(parts + rein_xh_part(p_rows, n_grp, n_whole, rb, grp, split)) + blockIdx.y * 256u + threadIdx.x;
#pragma unroll 4
    for (unsigned k = 0; k < split; k++) {
        const float4 p = src[(size_t)k * (grp.n * 1024u)];
        s[0] += p.x; s[1] += p.y; s[2] += p.z; s[3] += p.w;
    }
    float* o = y + (size_t)tok * out_dim + row;
    if ((out_dim & 3u) == 0u && ((size_t)y & 15u) == 0u) {
        if (row < out_dim) *reinterpret_cast<float4*>(o) = make_float4(s[0], s[1], s[2], s[3]);
        return;
    }
#pragma unroll
    for (unsigned v = 0; v < 4; v++)
        if (row + v < out_dim) o[v] = s[v];
}
