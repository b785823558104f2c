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
};

// Rows of a step per sequence, on average, from which the chunked kernel takes it. A chunk costs about as much for one row as
// for 32. 32 sequences of 8 rows (us, token by token / chunk): 64 heads of 128 x 64 29.3 / 28.7, 16 heads of 128 x 128 with SiLU
// 21.2 / 16.9, 16 of 64 x 128 with normaliser 13.7 / 13.7; of 16 rows 39 / 30, 32 / 17.5, 17.2 / 13.7.
constexpr int CHUNK_LINEAR_MIN_ROWS = 8;

// whether launch_chunk_linear takes this step: dim and vdim 32, 64 or 128, rows of x in whole 16-byte pieces, enough rows
bool chunk_linear_takes(const ChunkLinearArgs& a, int rows, int num_seqs);
hipError_t launch_chunk_linear(const ChunkLinearArgs& a, RaggedRows r, hipStream_t s);

}  // namespace die
