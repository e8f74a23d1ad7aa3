// MoE expert-routing counting sort, gather and scatter: same entry points and
// arguments as kernels/moe_expert_sort.cpp:27-110 of the reference.
//
//   moe_sort_zero       buf[0..n) = 0
//   moe_sort_histogram  count[e] = number of routing entries with ids[i] == e
//   moe_sort_scan       expert_off[e], tile_off[e] = exclusive prefix sums of
//                       count and ceil(count/bn); entry n_expert holds the totals
//   moe_sort_scatter    perm[expert_off[e] + rank] = i   (rank by atomic counter:
//                       the order inside one expert is not deterministic)
//   moe_gather_xq       xq_dst[p] = xq_src[perm[p] / n_used]   (rows of 40-byte blocks)
//   moe_scatter_rows    dst[perm[p]] = src[p]                  (rows of `dim` floats)
//
// Every kernel is a grid-stride loop, so any launch geometry is correct; the
// scan is one wavefront doing a DPP-free shuffle scan instead of a serial loop.
#include "moe_units.h"

extern "C" __global__ void moe_sort_zero(int* __restrict__ buf, unsigned int n)
{
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) buf[i] = 0;
}

extern "C" __global__ void moe_sort_histogram(const int* __restrict__ ids, int* __restrict__ count,
                                              unsigned int n_entries, unsigned int n_expert)
{
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n_entries; i += gridDim.x * blockDim.x) {
        const int e = ids[i];
        if (e >= 0 && (unsigned)e < n_expert) atomicAdd(&count[e], 1);
    }
}

// Inclusive scan over one wavefront.
__device__ __forceinline__ int rein_wave_scan_incl(int v, unsigned lane)
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(v, o);
        if (lane >= (unsigned)o) v += t;
    }
    return v;
}

// Only wavefront 0 of block 0 works (the reference launches one block of 64).
extern "C" __global__ void moe_sort_scan(const int* __restrict__ count, int* __restrict__ expert_off,
                                         int* __restrict__ tile_off, unsigned int n_expert,
                                         unsigned int bn)
{
    if (blockIdx.x != 0 || threadIdx.x >= 64) return;
    const unsigned lane = threadIdx.x;
    int ebase = 0, tbase = 0;
    for (unsigned e0 = 0; e0 < n_expert; e0 += 64) {
        const unsigned e = e0 + lane;
        const int c = e < n_expert ? count[e] : 0;
        const int t = (int)(((unsigned)c + bn - 1u) / bn);
        const int ce = rein_wave_scan_incl(c, lane);
        const int te = rein_wave_scan_incl(t, lane);
        if (e < n_expert) {
            expert_off[e] = ebase + ce - c;
            tile_off[e]   = tbase + te - t;
        }
        ebase += __shfl(ce, 63);
        tbase += __shfl(te, 63);
    }
    if (lane == 0) {
        expert_off[n_expert] = ebase;
        tile_off[n_expert]   = tbase;
    }
}

extern "C" __global__ void moe_sort_scatter(const int* __restrict__ ids, const int* __restrict__ expert_off,
                                            int* __restrict__ cursor, int* __restrict__ perm,
                                            unsigned int n_entries, unsigned int n_expert)
{
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n_entries; i += gridDim.x * blockDim.x) {
        const int e = ids[i];
        if (e < 0 || (unsigned)e >= n_expert) continue;
        const int rank = atomicAdd(&cursor[e], 1);
        perm[expert_off[e] + rank] = (int)i;
    }
}

// One 40-byte block = five 8-byte words per thread; blockIdx.y strides over entries.
extern "C" __global__ void moe_gather_xq(const unsigned char* __restrict__ xq_src, const int* __restrict__ perm,
                                         unsigned char* __restrict__ xq_dst, unsigned int nsub,
                                         unsigned int n_used, unsigned int n_entries)
{
    for (unsigned p = blockIdx.y; p < n_entries; p += gridDim.y) {
        const unsigned tok = (unsigned)perm[p] / n_used;
        const uint2* s = reinterpret_cast<const uint2*>(xq_src + (size_t)tok * nsub * 40);
        uint2*       d = reinterpret_cast<uint2*>(xq_dst + (size_t)p * nsub * 40);
        for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < nsub * 5; i += gridDim.x * blockDim.x) d[i] = s[i];
    }
}

extern "C" __global__ void moe_scatter_rows(const float* __restrict__ src, const int* __restrict__ perm,
                                            float* __restrict__ dst, unsigned int dim, unsigned int n_entries)
{
    for (unsigned p = blockIdx.y; p < n_entries; p += gridDim.y) {
        const float* s = src + (size_t)p * dim;
        float*       d = dst + (size_t)perm[p] * dim;
        for (unsigned c = blockIdx.x * blockDim.x + threadIdx.x; c < dim; c += gridDim.x * blockDim.x) d[c] = s[c];
    }
}

// moe_sort_scatter that also records where each routing entry went: inv[i] = position
// of entry i in the sorted order (perm[inv[i]] == i).  Lets the combine read the
// sorted expert outputs directly instead of through a scatter pass.
extern "C" __global__ void rein_moe_sort_scatter_inv(const int* __restrict__ ids, const int* __restrict__ expert_off,
                                                     int* __restrict__ cursor, int* __restrict__ perm,
                                                     int* __restrict__ inv, unsigned int n_entries,
                                                     unsigned int n_expert, const int* __restrict__ tile_off, int* __restrict__ place)
{
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n_entries; i += gridDim.x * blockDim.x) {
        const int e = ids[i];
        if (e < 0 || (unsigned)e >= n_expert) { inv[i] = -1; continue; }
        const int rank = atomicAdd(&cursor[e], 1), pos = expert_off[e] + rank;
        perm[pos] = (int)i;
        inv[i] = pos;
        if (place) place[pos] = tile_off[e] * 32 + rank;                 // 32 entries of an expert to a tile
    }
}

// ---- units of the launches on wide tiles (moe_wide.h) -----------------------------------
// A group: up to `most` tiles of one expert, the work that one workgroup does on 128 of the expert's rows.  XCD x takes the x-th eighth
// of the groups of `most` tiles and then of those that are what is left of an expert (the longer ones come first), with totals that differ by
// one at most: a launch lasts as long as its fullest XCD (by eighths of the tiles one had 14 groups and another 18; 512 tokens of 128 experts,
// gate + up 120 -> 110 us).  units [XCD][per_xcd]; n = 0 where there is none.  One wavefront.
__device__ __forceinline__ void rein_moe_list_units(const int* expert_off, const int* tile_off, unsigned n_expert, unsigned most,
                                                    ReinMoeUnit* units, unsigned per_xcd)
{
    const unsigned lane = threadIdx.x & 63u;
    unsigned n_full = 0u, n_rest = 0u;
    for (unsigned e = lane; e < n_expert; e += 64u) {
        const unsigned t = (unsigned)(tile_off[e + 1] - tile_off[e]);
        n_full += t / most;
        n_rest += t % most != 0u;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { n_full += (unsigned)__shfl_xor((int)n_full, o); n_rest += (unsigned)__shfl_xor((int)n_rest, o); }
    // bounds of the XCDs; the rests make the totals even, and a bound that would step back stays
    unsigned f0[9], r0[9];
    f0[0] = r0[0] = 0u;
#pragma unroll
    for (unsigned x = 1; x <= 8u; x++) {
        f0[x] = (unsigned)((unsigned long long)n_full * x / 8u);
        r0[x] = max(r0[x - 1], (unsigned)((unsigned long long)(n_full + n_rest) * x / 8u) - f0[x]);
    }
#pragma unroll
    for (unsigned x = 0; x < 8u; x++)
        for (unsigned k = f0[x + 1] - f0[x] + r0[x + 1] - r0[x] + lane; k < per_xcd; k += 64u) units[x * per_xcd + k] = ReinMoeUnit{0u, 0u, 0u, 0u};
    const auto put = [&](unsigned i, bool full, const ReinMoeUnit& u) {
        unsigned at = 0u;
#pragma unroll
        for (unsigned x = 0; x < 8u; x++) {
            if (full ? i >= f0[x] && i < f0[x + 1] : i >= r0[x] && i < r0[x + 1]) at = x * per_xcd + (full ? i - f0[x] : f0[x + 1] - f0[x] + i - r0[x]);
        }
        units[at] = u;
    };
    unsigned before_full = 0u, before_rest = 0u;
    for (unsigned e0 = 0; e0 < n_expert; e0 += 64u) {
        const unsigned e = e0 + lane;
        const unsigned t0 = e < n_expert ? (unsigned)tile_off[e] : 0u, t = e < n_expert ? (unsigned)tile_off[e + 1] - t0 : 0u;
        const unsigned tok = e < n_expert ? (unsigned)expert_off[e] : 0u, end = e < n_expert ? (unsigned)expert_off[e + 1] : 0u;
        const unsigned f = t / most, rest = t % most != 0u;
        const unsigned in_full = (unsigned)rein_wave_scan_incl((int)f, lane), in_rest = (unsigned)rein_wave_scan_incl((int)rest, lane);
        for (unsigned g = 0; g < f; g++) put(before_full + in_full - f + g, true, ReinMoeUnit{e, t0 + g * most, tok + g * most * 32u, min(end - tok - g * most * 32u, most * 32u)});
        if (rest) put(before_rest + in_rest - 1u, false, ReinMoeUnit{e, t0 + f * most, tok + f * most * 32u, end - tok - f * most * 32u});
        before_full += (unsigned)__shfl((int)in_full, 63);
        before_rest += (unsigned)__shfl((int)in_rest, 63);
    }
}
// (behind the four-launch sort: wavefront 0 lists groups of two, wavefront 1 of four; a null list is left out)
extern "C" __global__ __launch_bounds__(128) void rein_moe_units(const int* __restrict__ expert_off, const int* __restrict__ tile_off, unsigned int n_expert,
                                                                 ReinMoeUnit* __restrict__ units2, unsigned int per_xcd2, ReinMoeUnit* __restrict__ units4,
                                                                 unsigned int per_xcd4)
{
    if (blockIdx.x != 0) return;
    if (threadIdx.x < 64u) { if (units2) rein_moe_list_units(expert_off, tile_off, n_expert, 2u, units2, per_xcd2); }
    else if (units4) rein_moe_list_units(expert_off, tile_off, n_expert, 4u, units4, per_xcd4);
}

// The whole counting sort in one workgroup of 1024 threads, for routing tables small enough
// that launches, not work, are what the four-kernel form costs (512 tokens x top-8 = 4096
// entries): histogram and rank counters live in LDS, wavefront 0 scans, the same threads
// scatter.  Writes count, expert_off, tile_off, perm and (if inv != nullptr) inv exactly as
// moe_sort_zero + moe_sort_histogram + moe_sort_scan + rein_moe_sort_scatter_inv would
// (the order inside one expert is as undetermined here as there).  n_expert <= 2048.
#define REIN_SORT1_MAX_EXPERT 2048
extern "C" __global__ __launch_bounds__(1024)
void rein_moe_sort_one_block(const int* __restrict__ ids, int* __restrict__ count, int* __restrict__ expert_off,
                             int* __restrict__ tile_off, int* __restrict__ perm, int* __restrict__ inv,
                             unsigned int n_entries, unsigned int n_expert, unsigned int bn, int* __restrict__ place,
                             ReinMoeUnit* __restrict__ units2, unsigned int per_xcd2, ReinMoeUnit* __restrict__ units4, unsigned int per_xcd4)
{
    __shared__ int tile[REIN_SORT1_MAX_EXPERT + 1];
    __shared__ int cnt[REIN_SORT1_MAX_EXPERT], off[REIN_SORT1_MAX_EXPERT + 1], cur[REIN_SORT1_MAX_EXPERT];
    if (blockIdx.x != 0 || n_expert > REIN_SORT1_MAX_EXPERT) return;
    for (unsigned e = threadIdx.x; e < n_expert; e += blockDim.x) { cnt[e] = 0; cur[e] = 0; }
    __syncthreads();
    for (unsigned i = threadIdx.x; i < n_entries; i += blockDim.x) {
        const int e = ids[i];
        if (e >= 0 && (unsigned)e < n_expert) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        const unsigned lane = threadIdx.x;
        int ebase = 0, tbase = 0;
        for (unsigned e0 = 0; e0 < n_expert; e0 += 64) {
            const unsigned e = e0 + lane;
            const int c = e < n_expert ? cnt[e] : 0;
            const int t = (int)(((unsigned)c + bn - 1u) / bn);
            const int ce = rein_wave_scan_incl(c, lane);
            const int te = rein_wave_scan_incl(t, lane);
            if (e < n_expert) {
                off[e] = ebase + ce - c;
                tile[e] = tbase + te - t;
                count[e] = c;
                expert_off[e] = ebase + ce - c;
                tile_off[e]   = tbase + te - t;
            }
            ebase += __shfl(ce, 63);
            tbase += __shfl(te, 63);
        }
        if (lane == 0) {
            off[n_expert]  = expert_off[n_expert] = ebase;
            tile[n_expert] = tile_off[n_expert]   = tbase;
        }
    }
    __syncthreads();
    // the last two wavefronts list the units of moe_wide.h, if they are asked for, while the others scatter
    const unsigned wave = threadIdx.x >> 6, listing = units2 || units4 ? 2u : 0u, n_scatter = blockDim.x - 64u * listing;
    if (threadIdx.x >= n_scatter) {
        if (wave == blockDim.x / 64u - 1u) { if (units2) rein_moe_list_units(off, tile, n_expert, 2u, units2, per_xcd2); }
        else if (units4) rein_moe_list_units(off, tile, n_expert, 4u, units4, per_xcd4);
        return;
    }
    for (unsigned i = threadIdx.x; i < n_entries; i += n_scatter) {
        const int e = ids[i];
        if (e < 0 || (unsigned)e >= n_expert) { if (inv) inv[i] = -1; continue; }
        const int rank = atomicAdd(&cur[e], 1), pos = off[e] + rank;
        perm[pos] = (int)i;
        if (inv) inv[i] = pos;
        if (place) place[pos] = tile[e] * 32 + rank;                     // 32 entries of an expert to a tile (bn = 32)
    }
}
