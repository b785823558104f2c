// Chunked matrix-core form of the gated delta rule (chunk_delta.hip), taken by launch_gated_delta for prompt portions with bf16
// gates. Same contract: capturable, no allocation.
#pragma once

#include "seq_launchers.h"

namespace die {

// Sets cut, the rows from which a sequence of this step goes in chunks: 0 for all of them, more than `rows` for none; in between both
// kernels are launched, and where the step holds long portions (`divided`) each runs its own sequences, else the token-by-token kernel
// all. Chunks: dim 64 or 128, vdim 64, 128 or 256, bf16 gates, from 9 rows per sequence on average, later where workgroups share compute units.
//
// A chunk costs the same for 1 row as for 16, and the token-by-token kernel, of which more workgroups share a compute unit, catches up
// where there are many. The lines are drawn by 8400 steps (equal, ragged and mixed, a decay per head or channel; the choice is 0.6 % from the better
// kernel in the mean of equal steps). 16 heads, a decay per head, us token by token / in chunks:
//     128 x 128: 1 sequence of 12 / 32 / 100 rows 16 / 11, 30 / 15, 81 / 29; 16 of 8 / 12 16 / 15, 20 / 15; 32 of 12 / 14 / 17 / 20 28 / 30, 30 / 30, 36 / 37,
//         39 / 38; 64 of 16 / 17 / 20 / 22 55 / 54, 61 / 68, 68 / 69, 73 / 70
//     64 x 64: 16 of 8 / 12 / 32 9 / 9, 10 / 9, 20 / 14; 64 of 14 / 17 / 20 / 24 24 / 23, 29 / 31, 31 / 31, 35 / 32; 128 of 17 / 24 / 32 44 / 53, 55 / 55, 68 / 58
//     64 x 128: 16 of 8 / 16 11 / 10, 17 / 11; 32 of 12 / 16 / 20 22 / 22, 25 / 22, 30 / 28; 128 of 16 / 17 / 24 68 / 68, 77 / 80, 101 / 82
//     128 x 64, two consuming waves of six: 16 of 12 / 17 14 / 12, 18 / 17; 32 of 20 / 33 / 40 28 / 34, 39 / 42, 43 / 42; 64 of 40 / 48 / 64 66 / 75, 75 / 81, 97 / 95;
//         128 of 48 138 / 158, 192 of 80 317 / 349
//     64 x 256, 128 x 256: 16 of 8 18 / 15, 26 / 28; 128 of 12 154 / 109, 226 / 209
// Steps of 128 value columns, more than two workgroups per compute unit and 17 - 20 rows on average lose to token by token unless they hold long
// portions among decode rows: they are divided (128 sequences, 8 of 200 rows: token by token 226 us, in chunks 121, divided 103). Dividing a step
// without them costs more than it gives, so one long portion must outlast the others: token by token it takes 0.8 us a row, in chunks 0.2, the others
// 0.05 us a row of theirs.
void chunk_delta_cut(GatedDeltaArgs& a, int rows, int num_seqs);
// floats of scratch (GatedDeltaArgs::work) that the step needs: 0 where no sequence goes in chunks
int64_t chunk_delta_work(GatedDeltaArgs a, int rows, int num_seqs);
hipError_t launch_chunk_delta(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s);

}  // namespace die
