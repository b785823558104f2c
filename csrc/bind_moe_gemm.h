// Binding of the grouped expert product, shared by both extensions (each compiles the kernel and this once).
#pragma once

#include <optional>

#include "kernels/moe_gemm.h"

// out [rows, ncols] (rows sorted by expert) = act(x[row] W_e^T): returns false, with nothing launched, where the sizes do not tile or
// the weights are strided views (the library products that the caller has for such cases take any strides).
// tile_rows: 0, or the rows of a tile (tests).
inline bool moe_gemm_op(at::Tensor out, at::Tensor x, at::Tensor w, at::Tensor offsets, std::optional<at::Tensor> sorted, int64_t topk,
                        std::optional<at::Tensor> scale, int64_t act, double limit, double alpha, int64_t tile_rows, hipStream_t stream) {
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 &&
                  out.scalar_type() == at::kBFloat16 && w.is_cuda() && out.is_cuda(),
              "moe_gemm: bf16 device tensors");
  TORCH_CHECK(w.device() == x.device() && out.device() == x.device() && offsets.device() == x.device() &&
                  (!sorted.has_value() || sorted->device() == x.device()) && (!scale.has_value() || scale->device() == x.device()),
              "moe_gemm: one device");
  TORCH_CHECK(x.dim() == 2 && x.stride(1) == 1 && w.dim() == 3 && out.dim() == 2 && out.is_contiguous() && w.size(2) == x.size(1),
              "moe_gemm: x [rows, K], w [E, N, K], out [rows, ncols]");
  TORCH_CHECK(act >= die::MOE_ACT_NONE && act <= die::MOE_ACT_RELU2, "moe_gemm: activation");
  const bool gated = act >= die::MOE_ACT_SILU && act <= die::MOE_ACT_GELU;
  TORCH_CHECK(w.size(1) == out.size(1) * (gated ? 2 : 1), "moe_gemm: w rows");
  TORCH_CHECK(offsets.scalar_type() == at::kInt && offsets.is_contiguous() && offsets.is_cuda() && offsets.numel() >= w.size(0) + 1,
              "moe_gemm: offsets [E + 1] int32");
  die::MoeGemmArgs a;
  a.sorted = nullptr;
  if (sorted.has_value()) {
    TORCH_CHECK(sorted->scalar_type() == at::kInt && sorted->is_contiguous() && sorted->is_cuda() && sorted->numel() == out.size(0) &&
                    topk >= 1 && x.size(0) * topk == out.size(0),
                "moe_gemm: sorted [T * topk] int32");
    a.sorted = sorted->data_ptr<int>();
  } else {
    TORCH_CHECK(x.size(0) == out.size(0), "moe_gemm: one x row per result row");
  }
  a.scale = nullptr;
  if (scale.has_value()) {
    TORCH_CHECK(scale->scalar_type() == at::kFloat && scale->is_contiguous() && scale->is_cuda() && scale->numel() == out.size(0),
                "moe_gemm: scale [rows] fp32");
    a.scale = scale->data_ptr<float>();
  }
  a.out = static_cast<uint16_t*>(out.data_ptr());
  a.x = static_cast<const uint16_t*>(x.data_ptr());
  a.ldx = x.stride(0);
  a.w = static_cast<const uint16_t*>(w.data_ptr());
  a.offsets = offsets.data_ptr<int>();
  a.topk = (int)topk;
  a.act = (int)act;
  a.limit = (float)limit;
  a.alpha = (float)alpha;
  a.tile_rows = (int)tile_rows;
  a.experts = (int)w.size(0);
  a.rows = (int)out.size(0);
  a.ncols = (int)out.size(1);
  a.K = (int)x.size(1);
  if (a.rows == 0) return true;
  if (!w.is_contiguous() || !die::moe_gemm_takes(a)) return false;
  const hipError_t e = die::launch_moe_gemm(a, stream);
  TORCH_CHECK(e == hipSuccess, "moe_gemm: ", hipGetErrorString(e));
  return true;
}
