// Chunked matrix-core form of linear attention with a decay per key channel (chunk_channel.hip), taken by launch_gated_linear_attn for bf16
// prompt portions. Same contract: capturable, no allocation.
#pragma once

#include "rec_launchers.h"

namespace die {

// Whether the sequences of this step go in chunks: dim 64 with vdim 64, 128 or 256, dim 128 with vdim 64 or 128, bf16, and so many rows per
// sequence on average that no such step takes longer. A chunk costs the same for 1 row as for 16, and token by token more workgroups share a
// compute unit. Token by token / in chunks, us, sequences of 16 heads (8 of 64 x 256):
//     64 x 128: 16 sequences of 12 rows 9.0 / 8.7, 32 of 17 18 / 18, 20 19 / 18, 64 of 24 35 / 36, 33 47 / 47, 40 52 / 46, 128 of 33 77 / 82, 40 87 / 82
//     64 x 64: 16 of 12 8.4 / 8.1, 1 of 16 8.2 / 8.5, 32 of 40 19 / 19, 48 21 / 19, 64 of 64 43 / 45      64 x 256: 128 of 17 49 / 51, 24 59 / 51
//     128 x 128: 32 of 17 27 / 29, 20 29 / 29, 128 of 33 129 / 128      128 x 64: 32 of 33 28 / 29, 40 31 / 29, 128 of 64 119 / 129
bool chunk_channel_fits(const GatedLinearArgs& a, int rows, int num_seqs);
hipError_t launch_chunk_channel(const GatedLinearArgs& a, RaggedRows r, hipStream_t s);

}  // namespace die
