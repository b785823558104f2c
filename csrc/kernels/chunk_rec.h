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
  int cut = 0, longest = 0;   // (chunk_linear_cut) cut > 0: sequences of so many rows, in divided steps (common.h)
};

// Sets cut, the rows from which a sequence of this step goes in chunks: 0 for all of them, more than `rows` for none; in between (with a
// normaliser) both kernels are launched, and where the step holds long portions (`divided`) each runs its own sequences, else the
// token-by-token kernel all. Chunks: dim and vdim 32, 64 or 128, rows of x in whole 16-byte pieces, on average more than 8 rows per
// sequence (states of 128 x 128, at most two workgroups per compute unit: 8).
//
// A chunk costs about as much for one row as for 32. 64 sequences (us, token by token / in chunks): of 9 rows, 64 heads of 128 x 64
// sharing q and k 55 / 50, 16 heads of 128 x 64 with SiLU 18.0 / 16.3; of 8 rows 51 / 51 and 16.5 / 16.1, 16 heads of 64 x 64 with
// SiLU 11.4 / 12.5. Decode rows beside a long portion make such averages as well, and gain more (63 beside 512 rows: 248 / 104 and, with
// normaliser, 264 / 79).
// With a normaliser a workgroup has one wave more, and with many large states the token-by-token kernel is as fast for a few rows more: 16
// heads of 64 x 128, 32 sequences of 9 rows 14.8 / 13.9; 64 of 9 / 10 / 12 rows 25.1 / 26.2 / 28.2, in chunks 29.5 / 29.6 / 29.8; 128 of 10 / 12 rows
// 46 / 50, in chunks 54 / 54. With more than three such states per compute unit to 10 rows, with more than six to 12, steps are divided if
// they hold long portions. One long portion pays off from about 5/8 of the rows per compute unit on (64 sequences, 10 rows beside one
// of 26 / 52 / 208: 34 / 48 / 121, divided 34 / 37 / 51; 256 sequences, beside one of 52 / 104: 89 / 103, divided 94 / 100).
// Where one wave stages 128-wide rows alone 24 rows (16 rows: 15.3 / 17.9, 24: 21 / 20.7; with SiLU it gains from 9 rows on); many
// 32 x 128 states cut many operands for few products: 12 rows, with normaliser 24.
void chunk_linear_cut(ChunkLinearArgs& a, int rows, int num_seqs);
hipError_t launch_chunk_linear(const ChunkLinearArgs& a, RaggedRows r, hipStream_t s);

}  // namespace die
