// Chunked matrix-core form of the matrix recurrences with one decay per head (chunk_rec.hip), taken by the launchers of
// gated_linear_attn and lightning_attn for bf16 prompt portions. Same contract: capturable, no allocation.
#pragma once

#include "seq_launchers.h"

namespace die {

struct ChunkLinearArgs {
  float* out;              // [T, H * vdim]
  float* nq;               // [T, H], with n_state
  const uint16_t* x;       // [T, *] bf16, row stride xstride: q | k (groups * dim each) at qoff / koff, v (H * vdim) at voff
  int64_t xstride;
  int qoff, koff, voff;
  bool silu;               // q, k, v are silu(x) rounded to bf16
  const float* ab;         // [T, H, abw]: (a, b) = the first two entries; nullptr: a = decay[h], b = 1
  int abw;
  const float* decay;      // [H]
  float* state;            // [slots, H, dim, vdim]
  float* n_state;          // [slots, H, dim] or nullptr
  int heads, groups, dim, vdim;
  float qscale;
  int cut;                 // sequences of fewer rows are left to the token-by-token kernel
};

// Rows from which a sequence of this step goes in chunks: 0 for all of them, more than `rows` for none; in between (with a normaliser)
// both kernels are launched, each for its own sequences. Chunks: dim and vdim 32, 64 or 128, rows of x in whole 16-byte pieces, on
// average more than 8 rows per sequence (states of 128 x 128, at most two workgroups per compute unit: 8).
//
// A chunk costs about as much for one row as for 32. 64 sequences (us, token by token / in chunks): of 9 rows, 64 heads of 128 x 64
// sharing q and k 55 / 50, 16 heads of 128 x 64 with SiLU 18.0 / 16.3; of 8 rows 51 / 51 and 16.5 / 16.1, 16 heads of 64 x 64 with
// SiLU 11.4 / 12.5. Decode rows beside a long portion make such averages as well, and gain more (63 beside 512 rows: 248 / 104 and, with
// normaliser, 264 / 79).
// With a normaliser a workgroup has one wave more, and with many large states the token-by-token kernel is as fast up to 12 rows (16 heads
// of 64 x 128, 64 sequences of 9 rows: 24.6 / 29.1, 12 rows 27.9 / 29.8, 16 rows 31.9 / 30.4; 16 sequences of 9 rows: 10.6 / 8.6): to
// there such steps are divided (9 rows: 27.0). Where one wave stages 128-wide rows alone 24 rows (16 rows: 15.3 / 17.9, 24: 21 / 20.7;
// with SiLU it gains from 9 rows on); many 32 x 128 states cut many operands for few products: 12 rows, with normaliser 24.
int chunk_linear_cut(const ChunkLinearArgs& a, int rows, int num_seqs);
hipError_t launch_chunk_linear(const ChunkLinearArgs& a, RaggedRows r, hipStream_t s);

}  // namespace die
