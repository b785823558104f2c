// Chunked matrix-core form of the gated delta rule (chunk_delta.hip), taken by launch_gated_delta for prompt portions with bf16
// gates. Same contract: capturable, no allocation.
#pragma once

#include "seq_launchers.h"

namespace die {

// Sets cut, the rows from which a sequence of this step goes in chunks: 0 for all of them, more than `rows` for none; in between both
// kernels are launched, and where the step holds long portions (`divided`) each runs its own sequences, else the token-by-token kernel
// all. Chunks: dim 64 or 128, vdim 64, 128 or 256, bf16 gates, on average 16 rows per sequence and more.
//
// A chunk costs the same for 1 row as for 16, and the token-by-token kernel, of which more workgroups share a compute unit, catches up
// where there are many. 16 heads of 128 x 128, us token by token / in chunks:
//     16 sequences  of 16 rows 20 / 14, 17 rows 22 / 19, 33 rows 37 / 25
//     32            of 18 rows 36 / 40, 22 rows 40 / 40, 15 - 29 rows 45 / 39
//     64            of 16 rows 54 / 54, 17 rows 59 / 76, 22 rows 72 / 76, 24 rows 78 / 77, 12 - 24 rows 65 / 66, 15 - 29 rows 76 / 74
// So chunks take averages of 16 rows, where every sequence may be one chunk, and more; with more than two workgroups per compute unit not
// those of 17 - 20. Such a step may hold long portions among decode rows (63 rows beside a portion of 1100: token by token 897, divided
// 344). Where it holds none, dividing it costs more than it gives (64 sequences of 21 rows, 8 of them of 28: 85 / 93), and one long
// portion must outlast the others: token by token it takes 0.8 us a row, in chunks 0.3, the others 0.05 us a row of theirs (64 sequences,
// 20 rows beside one of 56 / 112 / 224: 88 / 129 / 215, divided 96 / 107 / 133; 256, beside one of 112 / 224 / 448: 276 / 336 / 514, divided
// 302 / 333 / 384). With 256 value columns the workgroup fills the waves of either kernel (128 x 256, 64 sequences of 18 rows 71 / 76, of
// 12 - 24 rows 78 / 73). With vdim 64 two of six waves consume: 64 rows; with more than two workgroups per compute unit 96 (64 x 64, 64
// sequences of 80 / 96 / 112 rows: 88 / 104 / 120 token by token, 91 / 103 / 116 in chunks), with more than four 160 (128 sequences of
// 128 / 160 rows: 238 / 292, in chunks 253 / 301).
void chunk_delta_cut(GatedDeltaArgs& a, int rows, int num_seqs);
// floats of scratch (GatedDeltaArgs::work) that the step needs: 0 where no sequence goes in chunks
int64_t chunk_delta_work(GatedDeltaArgs a, int rows, int num_seqs);
hipError_t launch_chunk_delta(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s);

}  // namespace die
