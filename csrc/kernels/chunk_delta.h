// Chunked matrix-core form of the gated delta rule (chunk_delta.hip), taken by launch_gated_delta for prompt portions with bf16
// gates. Same contract: capturable, no allocation.
#pragma once

#include "seq_launchers.h"

namespace die {

// Whether launch_chunk_delta takes this step: dim 64 or 128, vdim 64, 128 or 256, bf16 gates, and on average a chunk's 16 rows per
// sequence (bf16, 32 heads, dim = vdim = 128, 16 sequences of 16 rows: 27 us here, 30 us token by token; of 8 rows: 26 and 21).
// With vdim 64 two of six waves consume, and where there are many workgroups the token-by-token kernel's 16 per compute unit hide
// more: 64 rows (64 sequences of 32 rows: 92 us here, 66 us there; of 64 rows: 72 and 72, of 512 rows: 208 and 350).
bool chunk_delta_takes(const GatedDeltaArgs& a, int rows, int num_seqs);
hipError_t launch_chunk_delta(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s);

}  // namespace die
