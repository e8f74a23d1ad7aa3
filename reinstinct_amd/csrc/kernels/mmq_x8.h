// Prefill GEMM for Q8_0, Q4_0, IQ4_XS and IQ3_S (an fp16 scale per 32 weights) on the int8 matrix instruction, 32 rows x up to 128
// tokens per wavefront.
//
// The arithmetic is that of the tile of mmq_gemm.h: per tile and sub-block one v_mfma_i32_32x32x32_i8 gives the exact dots, half a
// v_mfma_f32_32x32x1_2b the scales dx * d, and the vector ALU a subtract (the dots are accumulated on the bits of 1.5 * 2^23, so
// that they read as 12582912 + dot) and a multiply-add per element.  What is different is everything around it:
//   * a weight's unpack, its scale and its operand registers serve up to four token tiles (there: one or two);
//   * the activations come as an image in operand order, written once per call (rein_x8_quantize) and moved to LDS by the
//     transfer instructions: no registers, no regrouping, no second barrier;
//   * weights are the rows of the tile (lane = token), which makes units, partial tiles and output those of mmq_exact16.h;
//   * the matrix instructions of a tile issue between the vector instructions of the tile before, in an order that the
//     scheduler is given (two wavefronts per SIMD hide each other's latencies, but not a wavefront's own dependent runs).
//
// Bound: vector ALU beside the matrix unit; the same mix of instructions alone, on every CU, takes 67 ns per tile and sub-block and
// SIMD, the kernel without its transfers 73, with them 91-94: reads of L2 and LDS writes cost their share of issue and of the
// clock, which is at 2.1 of 2.4 GHz under this load.  GEMM kernel, us, the 64-token tile of mmq_gemm.h -> this: Q8_0
// 5120 -> 17408 at 2048 rows 620 -> 491-505, IQ4_XS at 512 rows 211 -> 134-140, Q4_0 4096 -> 6144 at 700 rows 103 -> 67, Q8_0
// 17408 -> 5120 at 200 rows 195 -> 74.  Eight wavefronts per workgroup (256 rows share the activations) 519, one order left to the
// scheduler 511, conversions instead of the biased dots 501-511 (2048 rows).
//
// Replaces, from nine rows, kernels/mmq_gemm_{q8_0,q4_0,iq4xs}_repacked.cpp of the reference behind rein_matmul_ws.
#pragma once

#include "mmq_exact16.h"

// ---- activation image: [sub-block pair][32-token tile] of 2304 bytes: [q: sub-block of the pair][lane = 32 h + token][quants
// 16 h .. 16 h + 15], then dx [q][32] fp32
#define REIN_X8_X   2048u
#define REIN_X8_REC 2304u

// a block's piece of a record, as rein_xh_store_block: lane q's words of the first and second sixteen quants
__device__ __forceinline__ void rein_x8_store_words(uint8_t* __restrict__ rec, float d, const int (&word)[2], unsigned half, unsigned j, unsigned q)
{
    if (q == 0u) reinterpret_cast<float*>(rec + REIN_X8_X)[half * 32u + j] = d;
#pragma unroll
    for (unsigned h = 0; h < 2; h++) *reinterpret_cast<int*>(rec + half * 1024u + (32u * h + j) * 16u + 4u * q) = word[h];
}
__device__ __forceinline__ void rein_x8_store_block(uint8_t* __restrict__ rec, const XhBlock& b, unsigned half, unsigned j, unsigned q)
{
    const int word[2] = {(int)rein_xh_word(b, 0), (int)rein_xh_word(b, 1)};
    rein_x8_store_words(rec, b.d, word, half, j, q);
}

// x -> image and blocks, as rein_xh_quantize_body.  Bound by memory: 4 bytes in, 2.4 out per value.
__device__ __forceinline__ void rein_x8_quantize_body(const float* __restrict__ x, uint8_t* __restrict__ img, BlockQ8* __restrict__ xq, unsigned in_dim,
                                                      unsigned p_rows)
{
    const XhQuantize w = rein_xh_quantize_who();
    const unsigned n_tt = (p_rows + 31u) / 32u;
    XhBlock b;
    rein_xh_quantize_block(b, x, xq, in_dim, p_rows, w.tok, w.sb, w.q);
    rein_x8_store_block(img + ((size_t)(w.sb >> 1) * n_tt + (w.tok >> 5)) * REIN_X8_REC, b, w.sb & 1u, w.j, w.q);
}

// LDS of one workgroup:
//   acts  2 x 8 x 2304               records of two consecutive steps (a step: two sub-block pairs), [pair of the step][tile]
//   ring  4 x 2 x planes x 2048      per wavefront: two slots of 4 sub-blocks x 32 rows x 16 B (Q8_0: of both planes)
//   scale 4 x 2 x 1024               per wavefront: fp16 scales of two superblocks: [row][8], or (padded rows) a dword each
template <int FMT> struct X8Lds {
    static constexpr unsigned kAct = 8u * REIN_X8_REC, kPlanes = FMT == REIN_Q8_0 ? 2u : 1u, kRing = 2u * kAct, kRingWave = 2u * kPlanes * 2048u;
    static constexpr unsigned kScale = kRing + 4u * kRingWave, kBytes = kScale + 4u * 2048u;
};

// (bits of the biased dots) -> dots, times the scales, onto elements [LO, HI) of a tile
template <int LO, int HI, int SO>
__device__ __forceinline__ void rein_x8_step(float (&acc)[16], const rein_v16i& dot, const rein_v32f& s, float bias)
{
#pragma unroll
    for (int v = LO; v < HI; v++) acc[v] = fmaf(__builtin_bit_cast(float, (int)dot[v]) - bias, s[SO + v], acc[v]);
}
// one matrix instruction, then N vector instructions, in this stretch of the program; nothing moves in or out
#define REIN_X8_STRETCH(N)                                       \
    do {                                                         \
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);         \
        __builtin_amdgcn_sched_group_barrier(0x2, N, 0);         \
        __builtin_amdgcn_sched_barrier(0);                       \
    } while (0)

// Superblocks [c0, c1) of the wavefront's 32 rows from row_base on and the NT token tiles from `tile` on, into acc.  One barrier per step of four
// sub-blocks: at its top everything that the step reads has landed (issued a whole step earlier: 4 NT matrix instructions of dots and
// NT of scales per wavefront), behind it the next step's transfers go out.  Padded rows of the slab (a power of two of sub-blocks)
// leave a row's scales at two-byte alignment: then they come by 16-bit words.
template <int FMT, int NT>
__device__ __forceinline__ void rein_x8_acc(const uint8_t* __restrict__ w, const uint8_t* __restrict__ img, unsigned in_dim, unsigned out_dim,
                                            unsigned n_tt, unsigned row_base, unsigned tile, unsigned c0, unsigned c1, unsigned char* const raw, float (&acc)[NT][16])
{
    using L = X8Lds<FMT>;
    using C = MmqChunk<FMT>;
    typedef __attribute__((address_space(3))) const void* lptr_t;
    const unsigned lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 31u, h = lane >> 5;
    const unsigned n_sub = in_dim >> 5;
    const Fmt<FMT> fmt(w, n_sub, out_dim);
    // rows past the matrix read its last one; offsets from the wavefront's first row
    const unsigned first = min(row_base, out_dim - 1u);
    auto row_at = [&](unsigned n) { return min(row_base + n, out_dim - 1u) - first; };
    const bool padded = (fmt.nsp & 1u) != 0u;
    unsigned w_off[2], sc_off[4];
#pragma unroll
    for (unsigned k = 0; k < 2; k++) {               // slot entry of (row n, sub-block s): 4 n + ((s + n / 2) & 3), as in MmqWLds
        const unsigned n = 16u * k + (lane >> 2);
        w_off[k] = (row_at(n) * fmt.nsp + (((lane & 3u) - (n >> 1)) & 3u)) * 16u;
    }
#pragma unroll
    for (unsigned k = 0; k < 4; k++)                 // (unpadded: sixteen bytes a row; the upper lanes fetch the rows again)
        sc_off[k] = padded ? (row_at(8u * k + (lane >> 3)) * fmt.nsp + (lane & 7u)) * 2u : row_at(j) * fmt.nsp * 2u;
    const unsigned sc_step = padded ? 4u : 2u;
    const unsigned ring_at = L::kRing + wave * L::kRingWave, sc_at = L::kScale + wave * 2048u;
    const uint4* const ring = reinterpret_cast<const uint4*>(raw + ring_at);
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lptr_t)raw);

    auto issue_weights = [&](unsigned step, unsigned slot) {
#pragma unroll
        for (unsigned pl = 0; pl < L::kPlanes; pl++) {
            const char* p = reinterpret_cast<const char*>(C::plane(fmt, pl)) + ((size_t)first * fmt.nsp + step * 4u) * 16u;
#pragma unroll
            for (unsigned k = 0; k < 2; k++) rein_lds_dma16_s(w_off[k], p, lds0 + ring_at + (slot * L::kPlanes + pl) * 2048u + k * 1024u);
        }
    };
    auto issue_acts = [&](unsigned step, unsigned buf) {
        const uint8_t* src = img + ((size_t)step * 2u * n_tt + tile) * REIN_X8_REC;
        const unsigned dst = lds0 + buf * L::kAct;
        const size_t next = (size_t)n_tt * REIN_X8_REC;                  // the step's second pair
#pragma unroll
        for (unsigned k = 0; k < (unsigned)NT; k++) {                    // 4 NT kilobytes of quants: kilobyte q is half q % 2 of record q / 2
            const unsigned q = wave + 4u * k, r = q >> 1, pr = r >= (unsigned)NT ? 1u : 0u, off = (r - pr * NT) * REIN_X8_REC + (q & 1u) * 1024u;
            rein_lds_dma16_s(lane * 16u, src + pr * next + off, dst + pr * NT * REIN_X8_REC + off);
        }
#pragma unroll
        for (unsigned k = 0; k < 2; k++) {
            const unsigned r = wave + 4u * k, pr = r >= (unsigned)NT ? 1u : 0u, off = (r - pr * NT) * REIN_X8_REC + REIN_X8_X;
            if (r < 2u * NT) rein_xh_dma_u32(lane * 4u, src + pr * next + off, dst + pr * NT * REIN_X8_REC + off);
        }
    };
    auto issue_scales = [&](unsigned c) {
        const unsigned dst = lds0 + sc_at + (c & 1u) * 1024u;
        const char* p = reinterpret_cast<const char*>(fmt.dp) + ((size_t)first * fmt.nsp + c * 8u) * 2u;
        if (padded) {
#pragma unroll
            for (unsigned k = 0; k < 4; k++) rein_xh_dma_u16(sc_off[k], p, dst + k * 256u);
        } else {
            rein_lds_dma16_s(sc_off[0], p, dst);
        }
    };

    float bias = REIN_MMQ_MAGIC_F;
    rein_v16i magic, d0[2], d1[2];
    rein_v32f s[2], z32;
#pragma unroll
    for (int v = 0; v < 16; v++) magic[v] = REIN_MMQ_MAGIC_I;
#pragma unroll
    for (int v = 0; v < 32; v++) z32[v] = 0.0f;
    asm volatile("" : "+v"(magic));                  // stays in registers
    asm volatile("" : "+s"(bias));
    d0[0] = d0[1] = d1[0] = d1[1] = magic;
    s[0] = s[1] = z32;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[t][v] = 0.0f;

    __syncthreads();                                 // the LDS may still be read by the caller's previous tile
    issue_weights(c0 * 2u, 0u);
    issue_scales(c0);
    issue_acts(c0 * 2u, 0u);
    const unsigned rot = j >> 1;

    for (unsigned c = c0; c < c1; c++) {
        const unsigned char* const sc_base = raw + sc_at + (c & 1u) * 1024u + (8u * j + h) * sc_step;
#pragma unroll
        for (unsigned u = 0; u < 2; u++) {
            const unsigned step = c * 2u + u;
            const bool more = u == 0u || c + 1u < c1;
            __builtin_amdgcn_sched_barrier(0);
            REIN_WAIT_VMCNT(0);
            __syncthreads();
            if (more) { issue_weights(step + 1u, u ^ 1u); issue_acts(step + 1u, u ^ 1u); }
            if (u == 0u && c + 1u < c1) issue_scales(c + 1u);
            const unsigned char* const act = raw + u * L::kAct + lane * 16u;
            const unsigned char* const dxs = raw + u * L::kAct + REIN_X8_X + lane * 4u;
#pragma unroll
            for (unsigned pr = 0; pr < 2; pr++) {
                const typename C::Small none{};
                rein_v4i b[2];
#pragma unroll
                for (unsigned q = 0; q < 2; q++)
                    b[q] = C::operand_at(ring + (u * L::kPlanes + (L::kPlanes == 2u ? h : 0u)) * 128u + 4u * j + ((2u * pr + q + rot) & 3u), none, 0, h);
                const float sc = rein_h2f(*reinterpret_cast<const uint16_t*>(sc_base + (4u * u + 2u * pr) * sc_step));
                rein_v4i xa[2][2];
                float dx[2];
                auto read = [&](int t) {
                    const unsigned rec = (pr * NT + t) * REIN_X8_REC;
                    xa[t & 1][0] = *reinterpret_cast<const rein_v4i*>(act + rec);
                    xa[t & 1][1] = *reinterpret_cast<const rein_v4i*>(act + rec + 1024u);
                    dx[t & 1] = *reinterpret_cast<const float*>(dxs + rec);
                };
                read(0);
                __builtin_amdgcn_sched_barrier(0);
                // Stage t: tile t's scales and dots in the matrix unit, the elements of the tile before (the last tile of the
                // previous pair for t = 0; nothing times nothing in the very first) under them
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const int now = (int)((2u * u + pr) * NT + t) & 1, old = now ^ 1, tp = (t + NT - 1) % NT;
                    if (t + 1 < NT) read(t + 1);
                    s[now] = __builtin_amdgcn_mfma_f32_32x32x1f32(sc, dx[t & 1], z32, 0, 0, 0);
                    rein_x8_step<0, 16, 0>(acc[tp], d0[old], s[old], bias);
                    REIN_X8_STRETCH(32);
                    d0[now] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b[0], xa[t & 1][0], magic, 0, 0, 0);
                    rein_x8_step<0, 8, 16>(acc[tp], d1[old], s[old], bias);
                    REIN_X8_STRETCH(16);
                    d1[now] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b[1], xa[t & 1][1], magic, 0, 0, 0);
                    rein_x8_step<8, 16, 16>(acc[tp], d1[old], s[old], bias);
                    rein_xh_pin(acc[tp]);
                    REIN_X8_STRETCH(16);
                }
            }
        }
    }
    constexpr int end = (4 * NT - 1) & 1;
    rein_x8_step<0, 16, 0>(acc[NT - 1], d0[end], s[end], bias);
    rein_x8_step<0, 16, 16>(acc[NT - 1], d1[end], s[end], bias);
}

template <int FMT> struct X8Tile {
    static constexpr unsigned kMost = 4, kLeast = 1, kSlots = 512;
    template <int NT>
    static __device__ __forceinline__ void run(const uint8_t* __restrict__ w, const uint8_t* __restrict__ img, unsigned in_dim, unsigned out_dim, unsigned n_tt,
                                               unsigned row_base, unsigned tile, unsigned c0, unsigned c1, unsigned char* const raw, float (&acc)[NT][16])
    {
        rein_x8_acc<FMT, NT>(w, img, in_dim, out_dim, n_tt, row_base, tile, c0, c1, raw, acc);
    }
};
