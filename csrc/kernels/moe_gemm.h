// Grouped matrix product over expert-sorted rows for prompt-sized steps (moe_gemm.hip). Raw pointers + an explicit stream, no
// allocation, no host read of the expert offsets: capturable.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace die {

// what follows the product: the plain result, silu(g) u, the clamped sigmoid gate, tanh-form gelu(g) u, max(z, 0)^2
enum MoeAct { MOE_ACT_NONE = 0, MOE_ACT_SILU = 1, MOE_ACT_CLAMPED = 2, MOE_ACT_GELU = 3, MOE_ACT_RELU2 = 4 };

struct MoeGemmArgs {
  uint16_t* out;           // [rows, ncols] bf16; row j belongs to the expert e with offsets[e] <= j < offsets[e + 1]
  const uint16_t* x;       // bf16 rows of K (row stride ldx): row j reads x row sorted[j] / topk, without `sorted` row j
  int64_t ldx;
  const uint16_t* w;       // [E, wrows, K] bf16: wrows = ncols, or 2 * ncols = [gate | up] for the gated activations
  const int* offsets;      // [E + 1], on the device; nullptr: `experts` parts of one product over the same `rows` rows (slab)
  const int* sorted;       // [rows] or nullptr: the (token, slot) index of each sorted row
  int topk;
  const float* scale;      // [rows by (token, slot) index] or nullptr: factor of the row's products
  int act;
  float limit, alpha;
  int experts, rows, ncols, K;
  int tile_rows;           // rows of a tile at most: 128, 160, 192, 224 or 256; 64, 96: tiles of 64, 128 weight rows; 0: as the step's rows tile best
  int cus;                 // set by the launcher: compute units of the device
  float* slab = nullptr;   // [experts, rows, ncols] fp32 without `offsets` and activation: part e is the product over the e-th part of K
};
// whether launch_moe_gemm takes these sizes: K a multiple of 64, ncols of 256 (gated: 128), 16-byte aligned rows, offsets of rows
// within 32 bits
bool moe_gemm_takes(const MoeGemmArgs& a);
hipError_t launch_moe_gemm(const MoeGemmArgs& a, hipStream_t s);
// One dense product of 129 and more rows: `parts` fp32 slabs of it (act MOE_ACT_NONE; K a multiple of 64 parts), or, with one part and `out`, its
// activated bf16 rows.
hipError_t launch_dense_gemm(MoeGemmArgs a, hipStream_t s);

}  // namespace die
