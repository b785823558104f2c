// out[j] = act(x[row(j)] W_e^T) over rows sorted by expert, one launch for all experts (gfx950, bf16 in and out, fp32 sums).
//
// A workgroup of 8 waves owns a tile of 256 weight rows (gated activations: 128 gate rows and the 128 matching up rows) and BM of
// one expert's rows; which ones it finds from the offsets on the device, so nothing waits for the host. Both operands stream
// through a ring of LDS stages, filled by LDS-DMA (global_load_lds, 16 bytes per lane): W rows as they stand, x rows
// gathered through the sorted order on the way, so there is no gather pass. The LDS image is lane-linear; 16-byte pieces are
// XOR-ed by row, which makes the 32x32x16 fragment reads (32 rows, one piece per lane) conflict-free.
//
// Per stage a wave runs steps of 2 x MT matrix instructions, 16 deep. Fragments are read one step ahead, between the matrix
// instructions; the stage's one barrier stands before its last step, whose fragments are in registers by then. The
// activation runs on the fp32 accumulators (a wave holds gate and up of the same columns), which takes two passes over
// [rows, 2 ff] out, and rounds once where the separate passes rounded twice.
//
// What holds it up at many rows is its traffic into LDS (10.7 TB/s over all CUs; without the matrix instructions the two products of
// 4096 tokens through 8 experts of 4096 x 14336 take 2.75 of their 3.0 ms): no limit of the chip, as 256 x rows are fetched also where
// a tile holds fewer, and as with one workgroup per CU neither a tile's first stages nor its results pass beside another's products. At
// few rows it is the weights' rate from HBM. Both products and their epilogues against one library pair per expert behind a host read
// of the offsets (us, before -> after): 4096 tokens of that shape 2980 -> 2980, 1900 tokens 1628 -> 1340, 300 tokens 913 -> 729; 129 - 255
// tokens, before by the decode kernel in segments of 128 rows, 767 - 808 -> 680 - 722; 8191 tokens, four of 16 experts of 2048 x 1024,
// 870 -> 453; 1000 of them 820 -> 97; 2500 tokens, four of 32 experts of 4096 x 2048, 1594 -> 554.
#include <math.h>

#include "common.h"
#include "moe_gemm.h"

namespace die {

namespace {

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void global_cvoid;

constexpr int BN = 256, TN = 2;                   // weight rows of a tile, 32-row W tiles per wave
constexpr int WN = BN / (32 * TN), NW = 2 * WN;   // waves: 4 along the weight rows, 2 along the x rows
constexpr int ANY_TALL = 0;                       // tile_rows: 192, 224 or 256, as the kernel finds

// At most VM of the wave's LDS-DMA pieces outstanding and its LDS reads done. (The builtin, which the compiler's own waits take
// into account: it would wait for all reads before the first use of any.)
template <int VM> __device__ __forceinline__ void wait_for() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4) << 14 | 7 << 4);
  asm volatile("" ::: "memory");
}
template <int VM> __device__ __forceinline__ void wait_barrier() {
  wait_for<VM>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The functions of gated_act, to the same bf16 values. (__expf has twice the largest error and takes, of the 2955 us of 4096 tokens through
// 8 experts of 4096 x 14336, 18 us less; a division 9 us more.)
template <int ACT> __device__ __forceinline__ float gate(float g, float u, float limit, float alpha) {
  if constexpr (ACT == MOE_ACT_SILU) return gated(g, g) * u;
  if constexpr (ACT == MOE_ACT_GELU) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return gated(g, alpha * g) * (u + 1.0f);
}

// MT: 32-row x tiles per wave (BM = 64 MT rows per workgroup); BK: K of a stage (32 or 64); NS: stages of the ring
// (their products, if the expert's rows end there, are left out: a wave's time goes with its share of the tile's 32-row pieces)
template <int MT, int BK, int NS, int ACT>
__global__ void __launch_bounds__(64 * NW, MT == 4 ? 2 : 4) moe_gemm_kernel(MoeGemmArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BM = 64 * MT;
  constexpr bool GATED = ACT >= MOE_ACT_SILU && ACT <= MOE_ACT_GELU;
  constexpr int NO = GATED ? BN / 2 : BN;           // output columns of a tile
  constexpr int ROWB = 2 * BK, CPR = BK / 8, RPP = 64 / CPR;        // bytes and 16-byte chunks of a stage's row, rows per 1-KiB piece
  constexpr int STAGE = (BN + BM) * ROWB, PW = BN / RPP / NW, PX = BM / RPP / NW, PER = PW + PX;   // pieces per wave and stage
  constexpr int SUB = BK / 16;                                      // steps of one matrix instruction's depth
  static_assert(PW * NW * RPP == BN && PX * NW * RPP == BM, "whole pieces per wave");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- which tile: XCD i (blocks i, i + 8, ...) takes the i-th eighth of the tiles, whose neighbours share weights or x rows
  const int NT = a.ncols / NO;
  int R = a.tile_rows, total = 0;
  if (MT == 4 && R == ANY_TALL) {   // (see tile_height)
    int n[3] = {};
    for (int e = 0; e < a.experts; ++e) {
      const int m = a.offsets[e + 1] - a.offsets[e];
      n[0] += (m + 191) / 192;
      n[1] += (m + 223) / 224;
      n[2] += (m + 255) / 256;
    }
    int least = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int cost = (n[i] * NT + a.cus - 1) / a.cus * (192 + 32 * i + 512);
      if (i == 0 || cost < least) least = cost, R = 192 + 32 * i, total = n[i];
    }
  } else {
    for (int e = 0; e < a.experts; ++e) total += (a.offsets[e + 1] - a.offsets[e] + R - 1) / R;
  }
  total *= NT;
  const int per = (total + 7) / 8, t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || t >= total) return;
  int e = 0, r0 = 0, M = 0, tile = t;
  for (;; ++e) {
    r0 = a.offsets[e];
    M = a.offsets[e + 1] - r0;
    const int n = (M + R - 1) / R * NT;
    if (tile < n) break;
    tile -= n;
  }
  const int mts = (M + R - 1) / R, rows = ((M + mts - 1) / mts + 31) / 32 * 32;     // tiles of even heights
  const int n0 = tile / mts * NO, m0 = tile % mts * rows;                           // x tiles of one weight tile side by side
  r0 += m0;
  M = min(M - m0, rows);

  // ---- the wave's pieces: RPP rows each, chunk c of row r at place c ^ swz(r)
  auto swz = [](int r) { return BK == 64 ? r >> 1 & 7 : r >> 2 & 3; };
  const char* wbase = reinterpret_cast<const char*>(a.w) + (int64_t)e * (GATED ? 2 : 1) * a.ncols * a.K * 2;
  const char* xbase = reinterpret_cast<const char*>(a.x);
  uint32_t off[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int r = RPP * (wave + NW * (p < PW ? p : p - PW)) + lane / CPR;   // row of the W or the x part
    const int col = 16 * (lane % CPR ^ swz(r));
    if (p < PW) {   // 32 TN rows per wave column: with a gate the gate rows, then the matching up rows
      const int wr = GATED ? (r & 16 * TN ? a.ncols : 0) + n0 + r / (32 * TN) * (16 * TN) + r % (16 * TN) : n0 + r;
      off[p] = (uint32_t)wr * (uint32_t)(a.K * 2) + col;
    } else {
      const int j = r0 + min(r, M - 1);
      off[p] = (uint32_t)(a.sorted != nullptr ? a.sorted[j] / a.topk : j) * (uint32_t)(a.ldx * 2) + col;
    }
  }
  const int nst = a.K / BK;
  auto issue = [&](int s) {
    char* st = smem + s % NS * STAGE;
    const int64_t k = (int64_t)min(s, nst - 1) * ROWB;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const char* src = (p < PW ? wbase : xbase) + k + off[p];
      char* to = st + (p < PW ? wave + NW * p : BN / RPP + wave + NW * (p - PW)) * 1024;
      __builtin_amdgcn_global_load_lds((global_cvoid*)src, (lds_void*)to, 16, 0, 0);
    }
  };

  const int wn = wave % WN, wm = wave / WN, fr = lane & 31, hi = lane >> 5;
  // a fragment of step kk: 32 rows from `row`, chunk 2 kk + hi of each
  auto load = [&](int s, int kk, int row) {
    const char* p = smem + s % NS * STAGE + (row + fr) * ROWB + 16 * ((2 * kk + hi) ^ swz(fr));
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(p));
  };
  f32x16_t acc[TN][MT] = {};
#pragma unroll
  for (int p = 0; p < NS; ++p) issue(p);
  // (past the last stage the last one is fetched again, into a place that nothing reads any more: no branch stands between the
  // fragments' reads and their use, so every wait is for what is needed only)
  auto run = [&](auto count) {
    constexpr int MC = decltype(count)::value, MX = MC > 0 ? MC : 1, NF = MC > 0 ? TN + MC : 0;
    bf16x8_t wf[2][TN], xf[2][MX];   // [parity of the step][tile]
    auto frag = [&](int s, int kk, int i) {   // those of W, then the x tiles
      if (i < TN)
        wf[kk & 1][i] = load(s, kk, 32 * (TN * wn + i));
      else
        xf[kk & 1][i - TN] = load(s, kk, BN + 32 * (2 * (i - TN) + wm));
    };
    // The products of step kk. The next step's fragments (stage s, step next; next < 0: none) are read behind the first two pairs, so
    // that their latency passes under the rest, and `then` follows the third.
    auto step = [&](int kk, int s, int next, auto&& then) {
      static_for<MX>([&](auto mi) {
        constexpr int m = decltype(mi)::value;
        if constexpr (m < MC) {
#pragma unroll
          for (int n = 0; n < TN; ++n)
            acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[kk & 1][n], xf[kk & 1][m], acc[n][m], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (next >= 0) {
#pragma unroll
          for (int i = 0; i < NF; ++i)
            if (m == (MX > 1 && i >= (NF + 1) / 2 ? 1 : 0)) frag(s, next, i);
        }
        if constexpr (m == (MX > 2 ? 2 : MX - 1)) then();
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    wait_barrier<(NS - 1) * PER>();
#pragma unroll
    for (int i = 0; i < NF; ++i) frag(0, 0, i);
#pragma unroll 1
    for (int s = 0; s + 1 < nst; ++s) {
      static_for<SUB - 1>([&](auto ki) {
        wait_for<63>();   // the step's fragments, read during the last one's products
        step(decltype(ki)::value, s, decltype(ki)::value + 1, [] {});
      });
      // stage s + 1 has landed when only the stages behind it are outstanding; behind the barrier every wave has read all of stage s,
      // whose place in the ring stage s + NS takes
      wait_barrier<(NS - 2) * PER>();
      step(SUB - 1, s + 1, 0, [&] { issue(s + NS); });
    }
    static_for<SUB>([&](auto ki) {
      constexpr int kk = decltype(ki)::value;
      wait_for<63>();
      step(kk, nst - 1, kk + 1 < SUB ? kk + 1 : -1, [] {});
    });
  };
  const int mc = ((M + 31) / 32 + 1 - wm) / 2;   // the wave's 32-row pieces of x: wm, wm + 2, ...
  if constexpr (MT == 4) {
    if (mc == 4) run(IntC<4>{});
    if (mc == 3) run(IntC<3>{});
  }
  if (mc == 2) run(IntC<2>{});
  if (mc == 1) run(IntC<1>{});
  if (mc == 0) run(IntC<0>{});
  wait_for<0>();   // no LDS-DMA outlives the workgroup

  // ---- results: x row in the lane, weight rows 8 g + 4 hi + 0 .. 3 of a 32-row tile in the registers
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = 32 * (2 * m + wm) + fr;
    const float sc = a.scale != nullptr ? a.scale[a.sorted != nullptr ? a.sorted[r0 + min(row, M - 1)] : r0 + min(row, M - 1)] : 1.0f;
    uint16_t* op = a.out + (int64_t)(r0 + row) * a.ncols + n0 + (GATED ? 16 : 32) * TN * wn + 4 * hi;
#pragma unroll
    for (int n = 0; n < (GATED ? TN / 2 : TN); ++n)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (GATED)
            y[i] = gate<ACT>(acc[n][m][4 * g + i] * sc, acc[TN / 2 + n][m][4 * g + i] * sc, a.limit, a.alpha);
          else
            y[i] = acc[n][m][4 * g + i] * sc;
          if constexpr (ACT == MOE_ACT_RELU2) y[i] = fmaxf(y[i], 0.f) * fmaxf(y[i], 0.f);
        }
        if (row < M) *reinterpret_cast<uint2*>(op + 32 * n + 8 * g) = make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
      }
  }
}

template <int MT, int BK, int NS, int ACT> hipError_t launch_one(const MoeGemmArgs& a, hipStream_t s) {
  constexpr int BM = 64 * MT, NO = ACT >= MOE_ACT_SILU && ACT <= MOE_ACT_GELU ? BN / 2 : BN;
  constexpr size_t smem = (size_t)NS * (BN + BM) * 2 * BK;
  auto* fn = moe_gemm_kernel<MT, BK, NS, ACT>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (e != hipSuccess) return e;
  // at most one tile more per expert than its rows fill; blocks beyond the tiles that there are leave at once
  const int64_t mts = a.rows / (a.tile_rows == ANY_TALL ? 192 : a.tile_rows) + (a.experts < a.rows ? a.experts : a.rows);
  const int64_t blocks = (mts * (a.ncols / NO) + 7) / 8 * 8;
  hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(64 * NW), smem, s, a);
  return hipGetLastError();
}
// Tile heights. Up to 96 rows per expert two workgroups per CU with tiles of 128 rows (75 rows per expert of 4096 x 14336: 739 us for
// both products, with tall tiles 794); above, one workgroup per CU and tiles of 192, 224 or 256 rows. Which of them depends on how the
// experts' rows come out, so the kernel chooses from the offsets: the height whose rounds over the CUs cost least, a round being its
// rows plus what goes with any height (weights, and x rows that are fetched either way). Over 660 steps (11 widths, 100 - 2048 rows per
// expert: equal, random, skewed) that is within 0.2 % of the best height on average and 3 % at most; chosen from the average rows per
// expert, with half a tile for the remainders, it was 4.7 % and 78 %. (Both products at 192 / 224 / 256 rows, us: 425 rows per expert
// of 4096 x 14336 1768 / 1640 / 1276, 750 of 2048 x 2048 296 / 216 / 225, 1500 of 2048 x 1024 399 / 343 / 348.)
int tile_height(const MoeGemmArgs& a) { return a.rows <= 96 * a.experts ? 128 : ANY_TALL; }
template <int ACT> hipError_t launch_act(MoeGemmArgs a, hipStream_t s) {
  if (a.tile_rows == 0) a.tile_rows = tile_height(a);
  a.cus = num_cus();
  return a.tile_rows != 128 ? launch_one<4, 64, 2, ACT>(a, s) : launch_one<2, 32, 3, ACT>(a, s);
}

}  // namespace

bool moe_gemm_takes(const MoeGemmArgs& a) {
  const bool gated = a.act >= MOE_ACT_SILU && a.act <= MOE_ACT_GELU;
  auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const int64_t xrows = a.sorted != nullptr ? a.rows / a.topk : a.rows;
  return a.K >= 64 && a.K % 64 == 0 && a.ncols > 0 && a.ncols % (gated ? BN / 2 : BN) == 0 && a.ldx % 8 == 0 && a16(a.x) && a16(a.w) &&
         a16(a.out) && xrows * a.ldx * 2 < (int64_t(1) << 32) && (int64_t)2 * a.ncols * a.K * 2 < (int64_t(1) << 32);
}

hipError_t launch_moe_gemm(const MoeGemmArgs& a, hipStream_t s) {
  if (a.rows == 0) return hipSuccess;
  if (a.rows < 0 || a.experts < 1 || a.topk < 1 || !moe_gemm_takes(a)) return hipErrorInvalidValue;
  if (a.tile_rows != 0 && a.tile_rows != 128 && (a.tile_rows < 192 || a.tile_rows > 256 || a.tile_rows % 32 != 0)) return hipErrorInvalidValue;
  switch (a.act) {
    case MOE_ACT_NONE: return launch_act<MOE_ACT_NONE>(a, s);
    case MOE_ACT_SILU: return launch_act<MOE_ACT_SILU>(a, s);
    case MOE_ACT_CLAMPED: return launch_act<MOE_ACT_CLAMPED>(a, s);
    case MOE_ACT_GELU: return launch_act<MOE_ACT_GELU>(a, s);
    case MOE_ACT_RELU2: return launch_act<MOE_ACT_RELU2>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace die
