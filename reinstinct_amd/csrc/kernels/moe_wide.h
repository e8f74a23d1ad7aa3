// Routed experts' FFN on the wide tiles of mmq_exact16.h (Q4_K, Q5_K, Q6_K) and mmq_x8.h (Q8_0): a workgroup owns an expert's group of up to
// MOST 32-token tiles and 128 of its rows, so that a weight is unpacked once for all tokens of the group.
//
// The entries are sorted by expert (moe_expert_sort.hip, tiles of 32); the activations come as the image of those tiles.  What no entry
// belongs to in a tile is never written: a column of the matrix product that nobody stores.
#pragma once

#include "mmq_x8.h"
#include "q8_block.h"
#include "moe_units.h"

// Workgroup i runs on XCD i % 8 and takes row block k % n_block of the (k / n_block)-th unit of that XCD's list (k = i / 8): the row blocks of a
// group, one after the other, share its activations in one L2.
struct XgUnit { unsigned expert, tile, block, tok, n; };                 // n = 0: nothing to do
__device__ __forceinline__ XgUnit rein_xg_unit(const ReinMoeUnit* __restrict__ units, unsigned per_xcd, unsigned n_block)
{
    const unsigned k = blockIdx.x >> 3, at = k / n_block;
    if (at >= per_xcd) return XgUnit{0u, 0u, 0u, 0u, 0u};
    const ReinMoeUnit u = units[(blockIdx.x & 7u) * per_xcd + at];
    return XgUnit{u.expert, u.tile, k - at * n_block, u.tok, u.n};
}

// The image of the sorted entries from the tokens' blocks: eight entries x two superblocks to a workgroup, four threads to a block of 32, as
// rein_xh_quantize.  Entry p is token perm[p] / n_used and goes to slot place[p] % 32 of tile place[p] / 32.  (Quantizing a token again for each
// of its entries, 512 tokens x 8 of 2048: 14.3 us; a superblock to a workgroup and the place worked out of the experts' offsets 11.8.)
template <bool X8>
__device__ __forceinline__ void rein_xg_gather(const BlockQ8* __restrict__ xq, const int* __restrict__ perm, const int* __restrict__ place,
                                               const int* __restrict__ n_sorted, uint8_t* __restrict__ img, unsigned in_dim, unsigned n_used, unsigned n_entries,
                                               unsigned n_tt, unsigned with_xsum)
{
    __shared__ float xsum[2][8][9];
    __shared__ int to[8];
    const XhQuantize w = rein_xh_quantize_who();
    const XhImage image(img, in_dim, n_tt);
    const unsigned at = min(w.tok, n_entries - 1u), sb0 = w.sb + 8u * blockIdx.y, n_super = in_dim >> 8;         // (w.sb is a superblock of every one)
    const unsigned i = (unsigned)perm[at];
    const int slot = place[at];
    const bool live = w.tok < (unsigned)*n_sorted;   // entries of experts that exist
    if (live) {
        const BlockQ8* const from = xq + (size_t)(i / n_used) * (in_dim >> 5) + sb0;
        const unsigned tile = (unsigned)slot >> 5, j = (unsigned)slot & 31u;
        int word[2][2];
        float d[2], sum[2];
#pragma unroll
        for (unsigned k = 0; k < 2; k++) {
            const BlockQ8* const b = from + (2u * blockIdx.y + k < n_super ? 8u * k : 0u);
            word[k][0] = b->qs[w.q]; word[k][1] = b->qs[4u + w.q];
            d[k] = b->d; sum[k] = b->xsum;
        }
#pragma unroll
        for (unsigned k = 0; k < 2; k++) {
            if (2u * blockIdx.y + k >= n_super) break;
            const unsigned sb = sb0 + 8u * k;
            if constexpr (X8) {
                rein_x8_store_words(img + ((size_t)(sb >> 1) * n_tt + tile) * REIN_X8_REC, d[k], word[k], sb & 1u, j, w.q);
            } else {
                XhBlock b;
                b.d = d[k];
#pragma unroll
                for (int v = 0; v < 8; v++) b.q[v] = (int)(int8_t)(word[k][v >> 2] >> (8 * (v & 3)));
                rein_xh_store_block(image, b, tile, sb, j, w.q);
                if (w.q == 0u) xsum[k][sb & 7u][w.tok & 7u] = sum[k];
            }
        }
    }
    if (X8 || !with_xsum) return;
    if (w.q == 0u && (w.sb & 7u) == 0u) to[w.tok & 7u] = live ? slot : -1;
    __syncthreads();
    if (threadIdx.x < 64u) {                         // [superblock][op][lane half][entry]
        const unsigned k = threadIdx.x >> 5, op = (threadIdx.x >> 4) & 1u, hh = (threadIdx.x >> 3) & 1u, t = threadIdx.x & 7u, c = 2u * blockIdx.y + k;
        const int s = to[t];
        if (s < 0 || c >= n_super) return;
        uint32_t o3[4];
#pragma unroll
        for (int v = 0; v < 4; v++) o3[v] = rein_xh_xsum_word(xsum[k][2 * v][t], xsum[k][2 * v + 1][t], op, hh);
        uint8_t* dst = image.xs + ((size_t)c * n_tt + ((unsigned)s >> 5)) * REIN_XH_XS;
        *reinterpret_cast<uint4*>(dst + op * 1024u + (32u * hh + ((unsigned)s & 31u)) * 16u) = make_uint4(o3[0], o3[1], o3[2], o3[3]);
    }
}

// Gate and up projection of 64 columns of ff, SwiGLU and the quantizer: wavefronts 0, 1 run the gate rows of those columns, 2, 3 the up
// rows; the four 32 x 32 tiles of a token tile meet in LDS, and four threads a block turn them into the down projection's image, of
// which a workgroup writes the whole record of a sub-block pair.
enum XgOut : unsigned { REIN_XG_X8 = 0, REIN_XG_XH = 1, REIN_XG_XH_MIN = 2 };        // image of the down projection: int8, fp16, with xsum
template <class Tile, int NT>
__device__ __forceinline__ void rein_xg_swiglu_tiles(const uint8_t* __restrict__ slab, const uint8_t* __restrict__ img, uint8_t* __restrict__ out, unsigned in_dim,
                                                     unsigned out_dim, unsigned n_tt, const XgUnit& u, unsigned out_kind, unsigned char* raw)
{
    constexpr unsigned kPitch = 36;                  // floats of a token's 32 columns
    const unsigned lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 31u, h = lane >> 5;
    const unsigned tile = u.tile;
    float acc[NT][16];
    Tile::template run<NT>(slab, img, in_dim, out_dim, n_tt, u.block * 64u + (wave & 1u) * 32u, tile, 0u, in_dim >> 8, raw, acc);
    float* const meet = reinterpret_cast<float*>(raw);
    float* const sums = meet + 4u * 32u * kPitch;
    const unsigned half = threadIdx.x >> 7, tok = (threadIdx.x >> 2) & 31u, q = threadIdx.x & 3u;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        __syncthreads();
#pragma unroll
        for (int g = 0; g < 4; g++)
            *reinterpret_cast<float4*>(meet + (wave * 32u + j) * kPitch + 8 * g + 4u * h) = make_float4(acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]);
        __syncthreads();
        const float* const gt = meet + (half * 32u + tok) * kPitch + 4u * q;
        const float* const ut = gt + 64u * kPitch;
        const bool live = 32u * t + tok < u.n;
        XhBlock b;
        if (live) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float4 g4 = *reinterpret_cast<const float4*>(gt + 16 * k), u4 = *reinterpret_cast<const float4*>(ut + 16 * k);
                v[4 * k] = rein_silu_det(g4.x) * u4.x; v[4 * k + 1] = rein_silu_det(g4.y) * u4.y;
                v[4 * k + 2] = rein_silu_det(g4.z) * u4.z; v[4 * k + 3] = rein_silu_det(g4.w) * u4.w;
            }
            rein_xh_quantize_values(b, v);
            if (out_kind == REIN_XG_X8) rein_x8_store_block(out + ((size_t)u.block * n_tt + tile + t) * REIN_X8_REC, b, half, tok, q);
            else rein_xh_store_block(XhImage(out, out_dim, n_tt), b, tile + t, 2u * u.block + half, tok, q);
        }
        if (out_kind == REIN_XG_XH_MIN) {
            if (live && q == 0u) sums[half * 32u + tok] = b.sum;
            __syncthreads();
            const unsigned op = threadIdx.x >> 6, hh = (threadIdx.x >> 5) & 1u;              // [op][lane half][token]
            if (threadIdx.x < 128u && 32u * t + j < u.n) {
                uint8_t* dst = XhImage(out, out_dim, n_tt).xs + ((size_t)(u.block >> 2) * n_tt + tile + t) * REIN_XH_XS;
                *reinterpret_cast<uint32_t*>(dst + op * 1024u + (32u * hh + j) * 16u + (u.block & 3u) * 4u) = rein_xh_xsum_word(sums[j], sums[32u + j], op, hh);
            }
        }
    }
}
template <class Tile>
__device__ __forceinline__ void rein_xg_swiglu(const uint8_t* __restrict__ gate, const uint8_t* __restrict__ up, unsigned bytes_per_expert,
                                               const ReinMoeUnit* __restrict__ units, unsigned per_xcd, const uint8_t* __restrict__ img, uint8_t* __restrict__ out,
                                               unsigned in_dim, unsigned out_dim, unsigned n_tt, unsigned out_kind)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char rein_xg_lds[];
    const XgUnit u = rein_xg_unit(units, per_xcd, out_dim >> 6);
    if (u.n == 0u) return;
    // (a select on a scalar condition: the address stays in scalar registers)
    const uint8_t* const s = (__builtin_amdgcn_readfirstlane(threadIdx.x >> 7) ? up : gate) + (size_t)u.expert * bytes_per_expert;
    const unsigned n = (u.n + 31u) >> 5;
    if (n == 1u) { rein_xg_swiglu_tiles<Tile, 1>(s, img, out, in_dim, out_dim, n_tt, u, out_kind, rein_xg_lds); return; }
    if (n == 2u) { rein_xg_swiglu_tiles<Tile, 2>(s, img, out, in_dim, out_dim, n_tt, u, out_kind, rein_xg_lds); return; }
    if constexpr (Tile::kMost == 4u) {
        if (n == 3u) { rein_xg_swiglu_tiles<Tile, 3>(s, img, out, in_dim, out_dim, n_tt, u, out_kind, rein_xg_lds); return; }
        rein_xg_swiglu_tiles<Tile, 4>(s, img, out, in_dim, out_dim, n_tt, u, out_kind, rein_xg_lds);
    }
}

// Down projection: y [sorted entry][out_dim]
template <class Tile, int NT>
__device__ __forceinline__ void rein_xg_rows_tiles(const uint8_t* __restrict__ slab, const uint8_t* __restrict__ img, float* __restrict__ y, unsigned in_dim,
                                                   unsigned out_dim, unsigned n_tt, const XgUnit& u, unsigned char* raw)
{
    const unsigned lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 31u, h = lane >> 5;
    float acc[NT][16];
    Tile::template run<NT>(slab, img, in_dim, out_dim, n_tt, u.block * 128u + wave * 32u, u.tile, 0u, in_dim >> 8, raw, acc);
#pragma unroll
    for (int t = 0; t < NT; t++) {
        if (32u * t + j >= u.n) continue;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const unsigned row = u.block * 128u + wave * 32u + 8u * g + 4u * h;
            if (row < out_dim)
                *reinterpret_cast<float4*>(y + (size_t)(u.tok + 32u * t + j) * out_dim + row) = make_float4(acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]);
        }
    }
}
template <class Tile>
__device__ __forceinline__ void rein_xg_rows(const uint8_t* __restrict__ slab, unsigned bytes_per_expert, const ReinMoeUnit* __restrict__ units, unsigned per_xcd,
                                             const uint8_t* __restrict__ img, float* __restrict__ y, unsigned in_dim, unsigned out_dim, unsigned n_tt)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char rein_xg_lds[];
    const XgUnit u = rein_xg_unit(units, per_xcd, (out_dim + 127u) / 128u);
    if (u.n == 0u) return;
    const uint8_t* const s = slab + (size_t)u.expert * bytes_per_expert;
    const unsigned n = (u.n + 31u) >> 5;
    if (n == 1u) { rein_xg_rows_tiles<Tile, 1>(s, img, y, in_dim, out_dim, n_tt, u, rein_xg_lds); return; }
    if (n == 2u) { rein_xg_rows_tiles<Tile, 2>(s, img, y, in_dim, out_dim, n_tt, u, rein_xg_lds); return; }
    if constexpr (Tile::kMost == 4u) {
        if (n == 3u) { rein_xg_rows_tiles<Tile, 3>(s, img, y, in_dim, out_dim, n_tt, u, rein_xg_lds); return; }
        rein_xg_rows_tiles<Tile, 4>(s, img, y, in_dim, out_dim, n_tt, u, rein_xg_lds);
    }
}
