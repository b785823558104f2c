// Chunked matrix-core form of the gated delta rule (chunk_delta.hip), taken by launch_gated_delta for prompt portions with bf16
// gates. Same contract: capturable, no allocation.
#pragma once

#include "seq_launchers.h"

namespace die {

// Rows from which a sequence of this step goes in chunks: 0 for all of them, more than total_rows for none; in between both kernels are
// launched, each for its own sequences. Chunks: dim 64 or 128, vdim 64, 128 or 256, bf16 gates, on average 16 rows per sequence and more.
//
// A chunk costs the same for 1 row as for 16, and the token-by-token kernel, of which more workgroups share a compute unit, catches up
// where there are many. Both sides in us, 16 heads of 128 x 128 (token by token / in chunks):
//     a workgroup per compute unit (16 sequences):  of 16 rows 20 / 14, 17 rows 22 / 19, 33 rows 37 / 25
//     more (64 sequences):                          of 16 rows 54 / 54, 17 rows 59 / 76, 28 rows 89 / 79, 33 rows 100 / 96
// So with more workgroups than compute units (128 x 256: than half of them) chunks take averages of 16 rows, where every sequence may be
// one chunk, and of 28 and more; a step whose average lies between is divided, as it may hold long portions among decode rows (63 rows
// beside a portion of 1100: token by token 897, so 344), for 2 - 3 us more where it holds none. 64 x 256 fills the waves of either kernel
// and goes in chunks from 16 rows everywhere (64 sequences of 17 rows: 85 / 70). With vdim 64 two of six waves consume: 64 rows;
// with more than two workgroups per compute unit 128 (64 x 64, 64 sequences of 128 rows, 16 heads: 137 / 128), with more than four 256
// (32 heads, of 160 rows: 295 / 300), divided between (of 65 rows: 127 / 174, so 131).
int chunk_delta_cut(const GatedDeltaArgs& a, int rows, int num_seqs);
hipError_t launch_chunk_delta(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s);

}  // namespace die
