// What the load-time sources share: the row-parallel repack behind rein_repack_for_matvec and
// rein_ingest_for_matvec, and the Q8_0 block quantizer.  Internal to librein.
#pragma once
#include <cstddef>
#include <cstdint>

namespace rein {

// Where the on-disk blocks of one output row are.  A source whose rows have to be converted first writes the
// blocks into `staging` (a row of the format's blocks, one per thread) and returns it.
using RowSource = const uint8_t* (*)(const void* ctx, size_t row, uint8_t* staging);

// Rows 0..out_dim of `fmt` into the repacked layout at dst, split over threads; every byte of dst is written.
// The shape has been checked.  `staged`: the source uses its staging row.
void repack_parallel(int fmt, size_t in_dim, size_t out_dim, uint8_t* dst, RowSource source, const void* ctx, bool staged);

// n_blk blocks of 32 values to Q8_0 blocks (src/quant/q8_0.rs:45-61)
void quantize_q8_0_blocks(const float* x, size_t n_blk, uint8_t* o);

}  // namespace rein
