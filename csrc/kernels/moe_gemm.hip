// out[j] = act(x[row(j)] W_e^T) over rows sorted by expert, one launch for all experts (gfx950, bf16 in and out, fp32 sums).
//
// A tile is 256 weight rows (gated activations: 128 gate rows and the 128 matching up rows) by up to 256 of one expert's rows. One
// workgroup of 8 waves per CU goes from tile to tile; which ones it finds from the offsets on the device, so nothing waits for the host.
// Both operands stream through LDS, filled by LDS-DMA (global_load_lds, 16 bytes per lane): W rows as they stand, x rows gathered
// through the sorted order on the way, so there is no gather pass. A unit is the W or the x rows of a stage of 64 K (whole 128-byte
// lines); five units fit, so that while one stage is read the next and half of the one behind it are on their way, and while a tile's
// results are formed and stored the first units of the next tile. The LDS image is lane-linear; 16-byte pieces are XOR-ed by row,
// which makes the fragment reads (16 or 32 rows, one piece per lane) conflict-free.
//
// The waves are two groups, one wave of each per SIMD, half a stage apart: while one group's 32 matrix instructions run, the other
// reads its next fragments and issues its fetches, and a barrier exchanges them. (Both waves of a SIMD reading and multiplying at their
// own pace left the matrix cores waiting for fragments: a stage took 2500 - 2900 cycles, now 2000 - 2500 of 2048.) The activation runs
// on the fp32 accumulators (a wave holds gate and up of the same columns), which takes two passes over [rows, 2 ff] out, and rounds
// once where the separate passes rounded twice.
//
// What holds it up at many rows is power: under the products the clock falls to 1.6 - 1.8 GHz. So the tiles are 16x16x32 products: at the power limit
// a wave of 64 x 128 results runs 1.85 - 1.88 PFLOP/s with them from LDS on normal values and 1.60 - 1.64 with 32x32x16 (without the limit, on zeros, both are the
// same), the rows of x gone through there and back so that each product shares an operand with the one before it (1.88 against 1.83 - 1.85). The fetches
// into LDS take most of the rest: a copy of this kernel without them ran 1.28 times as fast, one with all of them from L2 1.09 times. (Waves of 128 x 128 results, one
// per SIMD, read a third less LDS; as a kernel they ran 7 - 20 % slower, as nothing runs beside its epilogues.) At few rows it is the weights' rate from HBM.
// Each product alone, back to back over three sets of rows and weights, 32x32x16 -> 16x16x32, us: 8 gated experts of 4096 x 14336, two of them, 3000 tokens 1371 -> 1192 (1.18 PFLOP/s)
// and 665 -> 590, 1075 tokens 644 -> 588 and 300 -> 279; four of 16 of 2048 x 1024, 8000 tokens 151 -> 137 and 149 -> 139; four of 32 of 4096 x 2048, 3000 tokens 223 -> 205 and 217 -> 208; two of 8
// gated ones of 2048 x 2048, 1500 tokens 66 -> 65 and 41 -> 41. (By the profiler, whose passes run at lower and lower clocks, the median of 12 at 4096 tokens 1925 -> 1685 and 995 -> 898.)
#include <math.h>

#include <algorithm>

#include "common.h"
#include "moe_gate.h"

namespace die {

namespace {

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void global_cvoid;

constexpr int BN = 256, BM = 256, TN = 2;         // weight rows and x rows of a tile, 32-row W tiles per wave
constexpr int WN = BN / (32 * TN), NW = 2 * WN;   // waves: 4 along the weight rows, 2 along the x rows
constexpr int BK = 64, ROWB = 2 * BK;             // K of a stage, bytes of a stage's row
constexpr int UNIT = BN * ROWB, NU = 5;           // a stage's W or x rows in LDS; places of the ring
constexpr int PC = UNIT / 1024 / NW;              // 1-KiB pieces (8 rows) of a unit per wave
static_assert(NU * UNIT <= 160 * 1024, "LDS of a compute unit");

__device__ __forceinline__ void fence() { asm volatile("" ::: "memory"); }
// at most VM of the wave's LDS-DMA pieces and stores outstanding / its LDS reads done
template <int VM> __device__ __forceinline__ void wait_vm() {
  fence();
  __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4) << 14 | 7 << 4 | 15 << 8);
  fence();
}
__device__ __forceinline__ void wait_lds() {
  fence();
  __builtin_amdgcn_s_waitcnt(15 | 3 << 14 | 7 << 4);
  fence();
}
__device__ __forceinline__ void barrier() {
  __builtin_amdgcn_sched_barrier(0);
  fence();
  __builtin_amdgcn_s_barrier();
  fence();
  __builtin_amdgcn_sched_barrier(0);
}

// inclusive sums over the lanes of a wave
template <int CTRL> __device__ __forceinline__ int from_before(int x) { return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, false); }
__device__ __forceinline__ int scan64(int x, int lane) {
  x += from_before<0x111>(x);
  x += from_before<0x112>(x);
  x += from_before<0x114>(x);
  x += from_before<0x118>(x);
  const int a = __builtin_amdgcn_readlane(x, 15), b = __builtin_amdgcn_readlane(x, 31), c = __builtin_amdgcn_readlane(x, 47);
  return x + (lane >= 16 ? a : 0) + (lane >= 32 ? b : 0) + (lane >= 48 ? c : 0);
}

// What a launch goes through: rows of experts by offsets; one product's rows; one product's, with a part of K in the place of an expert. (Known to the compiler, so that an
// expert's two offsets are loaded together: behind a test of the pointer they were loaded one after the other, per tile.)
constexpr int OF_EXPERTS = 0, OF_ONE = 1, OF_PARTS = 2;
// the first row of expert i <= experts, and the one behind its last
template <int OF> __device__ __forceinline__ int first_row(const MoeGemmArgs& a, int i) { return OF == OF_EXPERTS ? a.offsets[min(i, a.experts)] : 0; }
template <int OF> __device__ __forceinline__ int end_row(const MoeGemmArgs& a, int i) {
  return OF == OF_EXPERTS ? a.offsets[min(i + 1, a.experts)] : i < a.experts ? a.rows : 0;
}

struct Tile {
  int e, n0, r0, M;   // expert, first output column, first of M rows
  int turn;           // the stage of K that it starts with
};
// Weight rows are K apart, mostly a power of two: tiles that go through K in step ask the same few memory channels for their pieces. So
// each starts at a K of its own, spread by the golden ratio, and goes round. Experts of one tile of rows, us in step / so, at 64 rows each: 32 of
// 4096 x 2048 132 / 107 and 135 / 109, 8 gated ones of 4096 x 4096 135 / 109, of 2048 x 2048 43 / 39. Experts of more tiles stay in step, as these
// share the weights through L2 (4096 x 4096, 1000 rows each: in step 523, from places of their own 548), and so do launches that leave more than
// half of the CUs idle (16 of 2048 x 1024, 256 rows: 33.0 / 34.6).
__device__ __forceinline__ int first_stage(int n, int nst) { return (int)((uint64_t)((uint32_t)n * 2654435769u) * (uint32_t)nst >> 32); }
__device__ __forceinline__ int stage_of(int s, int turn, int nst) { return s + turn >= nst ? s + turn - nst : s + turn; }
template <int OF> __device__ __forceinline__ int stages(const MoeGemmArgs& a) { return OF == OF_PARTS ? a.K / (BK * a.experts) : a.K / BK; }   // of a tile
// The tiles of the launch, found from the offsets by every wave (lane i looks at experts i, i + 64, ...). Tiles of an expert are as even
// as 32-row pieces allow, at most R rows. XCD i (blocks i, i + 8, ...) takes the i-th eighth of the list, whose neighbours share
// weights or x rows; its CUs take turns. What is left for less than a turn of all of them is cut into `parts` by rows.
//
// R and parts are those that cost least. A tile's time goes with 128 + its rows (2048 K, all CUs busy: 256 rows 66 us, 192 46, 128 36,
// 64 26); of the whole, 0.7 go with the turns of the CU that has most and 0.3 with the mean of all, as CUs that rest leave the others a
// higher clock. Over 43 products (200 - 16000 tokens of 5 expert sizes, random routing) that is within 1.8 % of the best R and parts on average;
// the same R without parts 4.9 %, 256 rows without parts 14 %. (Candidates are weighed by a lane each: one after the other they took 5 us.)
template <int OF> struct Plan {
  int R = 0, per = 0, count = 0, full = 0, parts = 1;   // count: tiles of the own XCD
  int NT, cpx;
  const MoeGemmArgs& a;
  int lane;
  __device__ __forceinline__ Plan(const MoeGemmArgs& args, int nt, int lane_) : NT(nt), a(args), lane(lane_) {
    constexpr int NH = 5;   // heights 256, 224, .. 128: lanes 4 i + log2(parts)
    int n = 1, filled = 0;  // tiles of the lane's height; rows in whole 32-row pieces
    for (int b = 0; b < a.experts; b += 64) {
      const int m = end_row<OF>(a, b + lane) - first_row<OF>(a, b + lane);
      filled += 32 * __builtin_amdgcn_readlane(scan64((m + 31) / 32, lane), 63);
#pragma unroll
      for (int i = 0; i < NH; ++i) {
        const int k = __builtin_amdgcn_readlane(scan64((m + 255 - 32 * i) / (256 - 32 * i), lane), 63);
        n = lane / 4 == i ? (b == 0 ? k : n + k) : n;
      }
    }
    cpx = max(a.cus / 8, 1);
    const int h = 256 - 32 * min(lane / 4, NH - 1), c = 1 << (lane & 3), p = (n * NT + 7) / 8, turns = p / cpx, rem = p - turns * cpx;
    const float mean = (float)filled / (float)n, whole = 128.f + mean, cut = 128.f + fmaxf(mean / (float)c, 32.f);
    float cost = 0.7f * ((float)turns * whole + (float)((rem * c + cpx - 1) / cpx) * cut) +
                 0.3f * ((float)turns * whole + (float)(rem * c) / (float)cpx * cut);
    const bool out = lane >= 4 * NH || (lane & 3) == 3 || (a.tile_rows != 0 && (a.tile_rows != h || c > 1));
    cost = out ? __builtin_inff() : cost;
    float least = cost;
#pragma unroll
    for (int d = 1; d < 32; d *= 2) least = fminf(least, __shfl_xor(least, d, 64));
    const int best = __builtin_amdgcn_readfirstlane(__builtin_ctzll(__builtin_amdgcn_ballot_w64(cost == least) | 1ull << 63));
    R = __builtin_amdgcn_readlane(h, best);
    parts = __builtin_amdgcn_readlane(c, best);
    per = __builtin_amdgcn_readlane(p, best);
    const int total = __builtin_amdgcn_readlane(n * NT, best);
    full = per / cpx * cpx;
    count = min(max(total - (int)(blockIdx.x & 7) * per, 0), per);
  }
  // the block's first job from job j on
  __device__ __forceinline__ bool find(int& j, Tile& t) const {
    for (;; j += cpx) {
      if (j >= min(full, count) + max(count - full, 0) * parts) return false;
      int tile = (int)(blockIdx.x & 7) * per + j, part = 0, cut = 1;
      if (j >= full) {
        tile += (j - full) / parts - (j - full);
        part = (j - full) % parts;
        cut = parts;
      }
      int o0, o1, before, b = 0;
      uint64_t beyond;
      for (;; b += 64) {
        o0 = first_row<OF>(a, b + lane), o1 = end_row<OF>(a, b + lane);
        const int own = (o1 - o0 + R - 1) / R * NT, upto = scan64(own, lane);
        beyond = __builtin_amdgcn_ballot_w64(upto > tile);
        before = upto - own;
        if (beyond != 0 || b + 64 >= a.experts) break;
        tile -= __builtin_amdgcn_readlane(upto, 63);
      }
      if (beyond == 0) return false;
      const int l = __builtin_ctzll(beyond);
      tile -= __builtin_amdgcn_readlane(before, l);
      t.e = b + l;
      t.r0 = __builtin_amdgcn_readlane(o0, l);
      t.M = __builtin_amdgcn_readlane(o1, l) - t.r0;
      // up to 8 x tiles go over all weight tiles together, so that an XCD's CUs share both
      const int mts = (t.M + R - 1) / R, rows = ((t.M + mts - 1) / mts + 31) / 32 * 32;
      const int groups = (mts + 7) / 8, gs = (mts + groups - 1) / groups, g = tile / (gs * NT), gm = min(gs, mts - g * gs);
      tile -= g * gs * NT;
      const int h = (rows / 32 + cut - 1) / cut * 32, m0 = (g * gs + tile % gm) * rows + part * h;
      t.n0 = tile / gm;
      t.turn = mts == 1 ? first_stage(t.e * NT + t.n0, stages<OF>(a)) : 0;   // (used where the launch asks for it)
      t.M = min(min(t.M - m0, rows - part * h), h);
      t.r0 += m0;
      if (t.M > 0) return true;
    }
  }
};

// The activation on one value of a result column (with a gate: its gate and up sums).
template <int ACT> __device__ __forceinline__ float activated(float g, float u, const MoeGemmArgs& a) {
  if constexpr (ACT >= MOE_ACT_SILU && ACT <= MOE_ACT_GELU) return moe_gate<ACT>(g, u, a.limit, a.alpha);
  if constexpr (ACT == MOE_ACT_RELU2) return fmaxf(g, 0.f) * fmaxf(g, 0.f);
  return g;
}

// A lane's results of 32 TN weight rows by 32x32 products: z(n, i) is register i of the n-th 32-row tile (weight rows 8 g + 4 hi + 0 .. 3 of it for
// i = 4 g ..). Lanes 32 apart exchange halves of neighbouring g, so that each stores 8 columns at `op`, its own 8 hi columns on.
template <int ACT, class Z> __device__ __forceinline__ void store_row(Z z, uint16_t* op, bool in, const MoeGemmArgs& a) {
  constexpr bool GATED = ACT >= MOE_ACT_SILU && ACT <= MOE_ACT_GELU;
#pragma unroll
  for (int n = 0; n < (GATED ? TN / 2 : TN); ++n)
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      uint32_t p[2][2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = activated<ACT>(z(n, 4 * (g + q) + i), GATED ? z(TN / 2 + n, 4 * (g + q) + i) : 0.f, a);
        p[q][0] = pack2(y[0], y[1]), p[q][1] = pack2(y[2], y[3]);
      }
      const auto u = __builtin_amdgcn_permlane32_swap(p[0][0], p[1][0], false, false);
      const auto v = __builtin_amdgcn_permlane32_swap(p[0][1], p[1][1], false, false);
      if (in) *reinterpret_cast<uint4*>(op + 32 * n + 8 * g) = make_uint4(u[0], v[0], u[1], v[1]);
    }
}
// The same by 16x16 products: z(n, i) is register i of the n-th 16-row tile (weight rows 4 (lane / 16) + i of it). Lanes 16 apart exchange their
// columns of neighbouring tiles; each stores 8 columns at `op`, its own 16 (lane / 16 % 2) + 8 (lane / 32) columns on.
template <int ACT, class Z> __device__ __forceinline__ void store_row16(Z z, uint16_t* op, bool in, const MoeGemmArgs& a) {
  constexpr bool GATED = ACT >= MOE_ACT_SILU && ACT <= MOE_ACT_GELU;
#pragma unroll
  for (int n = 0; n < (GATED ? TN : 2 * TN); n += 2) {
    uint32_t p[2][2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = activated<ACT>(z(n + q, i), GATED ? z(TN + n + q, i) : 0.f, a);
      p[q][0] = pack2(y[0], y[1]), p[q][1] = pack2(y[2], y[3]);
    }
    const auto u = __builtin_amdgcn_permlane16_swap(p[0][0], p[1][0], false, false);
    const auto v = __builtin_amdgcn_permlane16_swap(p[0][1], p[1][1], false, false);
    if (in) *reinterpret_cast<uint4*>(op + 16 * n) = make_uint4(u[0], v[0], u[1], v[1]);
  }
}

template <int ACT, bool TURN, int OF = OF_EXPERTS>
__global__ void __launch_bounds__(64 * NW, 2) moe_gemm_kernel(MoeGemmArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr bool GATED = ACT >= MOE_ACT_SILU && ACT <= MOE_ACT_GELU;
  constexpr int NO = GATED ? BN / 2 : BN;           // output columns of a tile
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wm = wave / WN, fr = lane & 15, lg = lane >> 4;
  constexpr bool SLAB = OF == OF_PARTS;
  const int nst = stages<OF>(a);

  const Plan<OF> plan(a, a.ncols / NO, lane);
  int job = (int)(blockIdx.x >> 3);
  Tile t, next;
  if (!plan.find(job, t)) return;

  // ---- the wave's pieces of a unit: 8 rows each, 16-byte chunk c of row r at place c ^ swz(r)
  auto swz = [](int r) { return r >> 1 & 7; };
  const char *wbase, *xbase;
  uint32_t woff[PC], xoff[PC];
  int xr[PC];
  auto rows_of = [&](const Tile& u) {   // the x rows of the wave's pieces
#pragma unroll
    for (int p = 0; p < PC; ++p) xr[p] = u.r0 + min(8 * (wave + NW * p) + lane / 8, u.M - 1);
    if (a.sorted != nullptr) {
#pragma unroll
      for (int p = 0; p < PC; ++p) xr[p] = a.sorted[xr[p]];
    }
  };
  int turn = 0;
  auto offsets_of = [&](const Tile& u) {
    turn = TURN ? u.turn : 0;
    const int64_t part = SLAB ? (int64_t)u.e * nst * ROWB : 0;   // of a row
    wbase = reinterpret_cast<const char*>(a.w) + (SLAB ? part : (int64_t)u.e * (GATED ? 2 : 1) * a.ncols * a.K * 2);
    xbase = reinterpret_cast<const char*>(a.x) + part;
#pragma unroll
    for (int p = 0; p < PC; ++p) {
      const int r = 8 * (wave + NW * p) + lane / 8, col = 16 * (lane % 8 ^ swz(r));
      // 32 TN rows per wave column: with a gate the gate rows, then the matching up rows
      const int wr = GATED ? (r & 16 * TN ? a.ncols : 0) + u.n0 * NO + r / (32 * TN) * (16 * TN) + r % (16 * TN) : u.n0 * NO + r;
      woff[p] = (uint32_t)wr * (uint32_t)(a.K * 2) + col;
      const uint32_t row = a.sorted != nullptr && a.topk > 1 ? (uint32_t)xr[p] / (uint32_t)a.topk : (uint32_t)xr[p];
      xoff[p] = row * (uint32_t)(a.ldx * 2) + col;
    }
  };
  auto issue_w = [&](int s, int slot) {
    if constexpr (TURN) s = stage_of(s, turn, nst);
#pragma unroll
    for (int p = 0; p < PC; ++p)
      __builtin_amdgcn_global_load_lds((global_cvoid*)(wbase + (int64_t)s * ROWB + woff[p]),
                                       (lds_void*)(smem + slot * UNIT + (wave + NW * p) * 1024), 16, 0, 0);
  };
  auto issue_x = [&](int s, int slot, int pieces) {
    if constexpr (TURN) s = stage_of(s, turn, nst);
#pragma unroll
    for (int p = 0; p < PC; ++p)
      if (p < pieces)
        __builtin_amdgcn_global_load_lds((global_cvoid*)(xbase + (int64_t)s * ROWB + xoff[p]),
                                         (lds_void*)(smem + slot * UNIT + (wave + NW * p) * 1024), 16, 0, 0);
  };
  auto begin = [&](const Tile& u) {   // the first units of a tile, into places 0, 1, 2
    offsets_of(u);
    issue_w(0, 0);
    issue_x(0, 1, (u.M + 63) / 64);
    if (nst > 1) issue_w(1, 2);
  };
  int lo[BK / 32];   // a fragment of 16 rows: the lane's place at step kk
#pragma unroll
  for (int kk = 0; kk < BK / 32; ++kk) lo[kk] = fr * ROWB + 16 * ((4 * kk + lg) ^ swz(fr));

  rows_of(t);
  begin(t);
  for (;;) {
    job += plan.cpx;
    const bool more = plan.find(job, next);
    if (more) rows_of(next);
    const int nx = (t.M + 63) / 64, mc = ((t.M + 31) / 32 + 1 - wm) / 2;   // 64-row pieces of x that are fetched; the wave's 32-row pieces
    auto run = [&](auto mc_) {
    constexpr int MC = decltype(mc_)::value, MT = 2 * MC, MX = MT > 0 ? MT : 1, NT = 2 * TN;   // 16-row tiles of x, of W
    f32x4_t acc[NT][MX] = {};
    bf16x8_t wf[NT], xf[MX];
    auto products = [&] {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < NT; ++i) {   // (there and back: one operand stays at every product)
          const int n = m & 1 ? NT - 1 - i : i;
          acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[n], xf[m], acc[n][m], 0, 0, 0);
        }
      __builtin_amdgcn_s_setprio(0);
    };
      auto load = [&](int ws, int xs, auto half) {   // fragments of half a stage
        const char* wp = smem + ws * UNIT + 32 * TN * wn * ROWB;
        const char* xp = smem + xs * UNIT + 32 * wm * ROWB;
        const int l = lo[decltype(half)::value];
#pragma unroll
        for (int n = 0; n < NT; ++n) wf[n] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(wp + 16 * n * ROWB + l));
#pragma unroll
        for (int m = 0; m < MT; ++m)
          xf[m] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(xp + (64 * (m / 2) + 16 * (m % 2)) * ROWB + l));
      };
      wait_vm<0>();
      barrier();
      if (wm == 1) barrier();
      int ws = 0, xs = 1;
#pragma unroll 1
      for (int s = 1; s < nst; ++s) {   // stage s - 1
        int sx = xs + 2, sw = ws + 4;   // places of x(s), W(s + 1): those that stage s - 2 has left
        sx = sx >= NU ? sx - NU : sx;
        sw = sw >= NU ? sw - NU : sw;
        load(ws, xs, IntC<0>{});
        issue_x(s, sx, nx);
        wait_lds();
        barrier();
        products();
        barrier();
        load(ws, xs, IntC<1>{});
        const bool ahead = s + 1 < nst;
        if (ahead) issue_w(s + 1, sw);
        if (wm == 1) {   // stage s is there
          if (ahead) wait_vm<PC>(); else wait_vm<0>();
        }
        wait_lds();
        barrier();
        products();
        if (wm == 0) {
          if (ahead) wait_vm<PC>(); else wait_vm<0>();
        }
        barrier();
        ws += 2;
        ws = ws >= NU ? ws - NU : ws;
        xs = sx;
      }
      load(ws, xs, IntC<0>{});
      wait_lds();
      barrier();
      products();
      barrier();
      load(ws, xs, IntC<1>{});
      wait_lds();
      barrier();
      if (wm == 1 && more) begin(next);   // (no wave reads this tile's units any more)
      products();
      barrier();
      if (wm == 0 && more) begin(next);

    // ---- results: x row in the lane, weight rows in the registers
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int row = 32 * (2 * (m / 2) + wm) + 16 * (m % 2) + fr, rr = t.r0 + min(row, t.M - 1);
      if constexpr (SLAB) {
        float* sp = a.slab + ((int64_t)t.e * a.rows + rr) * a.ncols + t.n0 * NO + 32 * TN * wn + 4 * lg;
        if (row < t.M) {
#pragma unroll
          for (int n = 0; n < NT; ++n) *reinterpret_cast<f32x4_t*>(sp + 16 * n) = acc[n][m];
        }
        continue;
      }
      const float sc = a.scale != nullptr ? a.scale[a.sorted != nullptr ? a.sorted[rr] : rr] : 1.0f;
      uint16_t* op = a.out + (int64_t)rr * a.ncols + t.n0 * NO + (GATED ? 16 : 32) * TN * wn + 16 * (lg & 1) + 8 * (lg >> 1);
      store_row16<ACT>([&](int n, int i) __attribute__((always_inline)) { return acc[n][m][i] * sc; }, op, row < t.M, a);
    }
    };
    if (mc == 4) run(IntC<4>{});
    else if (mc == 3) run(IntC<3>{});
    else if (mc == 2) run(IntC<2>{});
    else if (mc == 1) run(IntC<1>{});
    else run(IntC<0>{});
    if (wm == 0) barrier();   // (the second waves' last products)
    if (!more) return;
    t = next;
  }
}

// ---- few tiles: 64 NB weight rows (with a gate 32 NB and the 32 NB matching ones) by up to 256 rows, one tile per workgroup
// Where tiles of 256 weight rows leave compute units idle, these are four times or twice as many, and what is left to bound them is the weights'
// rate from HBM and, with many rows, LDS (x rows are read once per 64 weight rows). A stage is 64 K of both operands, the same LDS image as above; as many
// stages as LDS holds are on their way, one barrier each. The waves are 2 or 4 along the x rows, NB along the weight rows, and what is left (2 or 4)
// groups along K of a stage, whose sums meet in LDS at the end: two waves per SIMD have work, and a wave that has more x rows reads less.
// us, tiles of 256 weight rows / 64 / 128, at 32, 64, 96, 128 and 160 rows per expert:
//   16 experts of 2048 x 1024, 256 tiles of 64     29 29 30 30 31 / 15 18 19 24 25        / 18 23 24 30 31
//   8 of 2048 x 2048, 256                          28 29 30 30 30 / 15 17 18 23 24        / 17 22 24 30 30
//   16 of 1024 x 2048, 512                         19 20 20 23 24 / 18 22 24 29 31        / 15 17 17 21 21
//   8 gated of 2048 x 2048, 512                    40 39 40 42 43 / 34 40 44 51 53        / 29 32 33 38 39
//   8 of 4096 x 4096, 512                          68 67 70 73 77 / 57 64 71 84 90        / 51 54 56 63 69
//   8 of 14336 x 4096, 512                         233 224 237 248 263 / 170 210 241 285 331   / 166 181 206 239 270
//   32 of 4096 x 2048, 1024                        102 107 115 125 134 / 109 126 141 163 177   / 100 108 112 132 147
//   8 gated of 4096 x 14336, 3584                  352 361 373 402 429 / 363 452 495 575 614   / 323 361 379 457 485
// So steps of up to a tile of 64 per CU take these up to 192 rows per expert on average (27 of 32 us; from 257 rows they are two tiles), of up to two
// those of 128 rows up to 144; larger ones up to 60 - 80 (few_tiles). (Two workgroups per CU, each with half the LDS and tiles of 64 by up to 128 rows: 15 17 19 27 for
// the third, 55 61 68 108 for the fifth.)
constexpr int FN = 32 * TN, FUNIT = FN * ROWB;   // weight rows of a tile, bytes of 64 rows of a stage

constexpr int FEW_LDS = 160 * 1024;

template <int ACT, int NB, int OF = OF_EXPERTS>
__global__ void __launch_bounds__(64 * NW, 2) moe_gemm_few_kernel(MoeGemmArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr bool GATED = ACT >= MOE_ACT_SILU && ACT <= MOE_ACT_GELU;
  constexpr int NO = (GATED ? FN / 2 : FN) * NB;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 31, hi = lane >> 5;
  constexpr bool SLAB = OF == OF_PARTS;
  const int nst = stages<OF>(a), NT = a.ncols / NO;

  // ---- the workgroup's tile: XCD i (blocks i, i + 8, ..) takes the i-th eighth of the list, whose neighbours share x rows or weights
  int total = 0;
  for (int b = 0; b < a.experts; b += 64) {
    const int m = end_row<OF>(a, b + lane) - first_row<OF>(a, b + lane);
    total += __builtin_amdgcn_readlane(scan64((m + BM - 1) / BM * NT, lane), 63);
  }
  const int per = (total + 7) / 8;
  int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || tile >= total) return;
  Tile t;
  for (int b = 0;; b += 64) {
    const int o0 = first_row<OF>(a, b + lane), o1 = end_row<OF>(a, b + lane);
    const int own = (o1 - o0 + BM - 1) / BM * NT, upto = scan64(own, lane);
    const uint64_t beyond = __builtin_amdgcn_ballot_w64(upto > tile);
    if (beyond == 0) {   // (there is one: tile < total)
      tile -= __builtin_amdgcn_readlane(upto, 63);
      continue;
    }
    const int l = __builtin_ctzll(beyond);
    tile -= __builtin_amdgcn_readlane(upto - own, l);
    t.e = b + l;
    t.r0 = __builtin_amdgcn_readlane(o0, l);
    t.M = __builtin_amdgcn_readlane(o1, l) - t.r0;
    break;
  }
  {
    const int mts = (t.M + BM - 1) / BM, rows = ((t.M + mts - 1) / mts + 31) / 32 * 32, m0 = tile % mts * rows;
    t.n0 = tile / mts;
    t.M = min(t.M - m0, rows);
    t.r0 += m0;
    if (t.M <= 0) return;
  }

  t.turn = first_stage(t.e * NT + t.n0, nst);
  auto run = [&](auto mx_) __attribute__((always_inline)) {
    constexpr int MX = decltype(mx_)::value;             // 64-row pieces of x
    constexpr int SLOT = FUNIT * (NB + MX), D = FEW_LDS / SLOT < 8 ? FEW_LDS / SLOT : 8;   // a stage in LDS, stages that it holds
    constexpr int MW = NB == 1 && MX % 2 == 0 ? 4 : 2, KG = NW / MW / NB;   // waves along the x rows, along K
    constexpr int MT = 2 * MX / MW, KS = BK / 16 / KG;   // 32-row tiles and 16-K steps of a wave
    const int wm = wave % MW, wn = wave / MW % NB, kg = wave / (MW * NB);
    // ---- the wave's pieces of a stage: 8 rows each, 16-byte chunk c of row r at place c ^ (r >> 1 & 7)
    const int r8 = 8 * wave + lane / 8, col = 16 * (lane % 8 ^ (r8 >> 1 & 7)) + (SLAB ? t.e * nst * ROWB : 0);
    const char* wp[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
      wp[b] = reinterpret_cast<const char*>(a.w) + ((SLAB ? 0 : (int64_t)t.e * (GATED ? 2 : 1) * a.ncols) + t.n0 * NO + b * (NO / NB) +
                                                     (GATED ? (r8 & 32 ? a.ncols : 0) + r8 % 32 : r8)) * a.K * 2 + col;
    const char* xp[MX];
#pragma unroll
    for (int p = 0; p < MX; ++p) {
      int row = t.r0 + min(r8 + 64 * p, t.M - 1);
      if (a.sorted != nullptr) row = a.topk > 1 ? a.sorted[row] / a.topk : a.sorted[row];
      xp[p] = reinterpret_cast<const char*>(a.x) + (int64_t)row * a.ldx * 2 + col;
    }
    auto issue = [&](int s, int slot) __attribute__((always_inline)) {
      s = stage_of(s, t.turn, nst);
#pragma unroll
      for (int b = 0; b < NB; ++b)
        __builtin_amdgcn_global_load_lds((global_cvoid*)(wp[b] + (int64_t)s * ROWB), (lds_void*)(smem + slot * SLOT + FUNIT * b + wave * 1024), 16, 0, 0);
#pragma unroll
      for (int p = 0; p < MX; ++p)
        __builtin_amdgcn_global_load_lds((global_cvoid*)(xp[p] + (int64_t)s * ROWB),
                                         (lds_void*)(smem + slot * SLOT + FUNIT * (NB + p) + wave * 1024), 16, 0, 0);
    };
    int lo[KS];   // a fragment of 32 rows: the lane's place at step kk
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) lo[kk] = fr * ROWB + 16 * ((2 * (KS * kg + kk) + hi) ^ (fr >> 1 & 7));
    f32x16_t acc[TN][MT] = {};
#pragma unroll
    for (int s = 0; s < D - 1; ++s)
      if (s < nst) issue(s, s);
    int slot = 0;
#pragma unroll 1
    for (int s = 0; s < nst; ++s) {
      // stage s is there once no more than the stages behind it are on their way
      const int behind = min(D - 2, nst - 1 - s);
      if (behind == D - 2) wait_vm<(D - 2) * (NB + MX)>();
      else if (D > 7 && behind == 5) wait_vm<5 * (NB + MX)>();
      else if (D > 6 && behind == 4) wait_vm<4 * (NB + MX)>();
      else if (D > 5 && behind == 3) wait_vm<3 * (NB + MX)>();
      else if (D > 4 && behind == 2) wait_vm<2 * (NB + MX)>();
      else if (D > 3 && behind == 1) wait_vm<NB + MX>();
      else wait_vm<0>();
      wait_lds();   // (the reads of stage s - 1, whose place is filled next)
      barrier();
      if (s + D - 1 < nst) issue(s + D - 1, slot == 0 ? D - 1 : slot - 1);
      const char* wl = smem + slot * SLOT;
      bf16x8_t wf[KS][TN], xf[KS][MT];
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
#pragma unroll
        for (int n = 0; n < TN; ++n) wf[kk][n] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(wl + FUNIT * wn + 32 * n * ROWB + lo[kk]));
#pragma unroll
        for (int m = 0; m < MT; ++m)
          xf[kk][m] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(wl + FUNIT * NB + 32 * (wm + MW * m) * ROWB + lo[kk]));
      }
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int n = 0; n < TN; ++n) acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[kk][n], xf[kk][m], acc[n][m], 0, 0, 0);
      slot = slot == D - 1 ? 0 : slot + 1;
    }
    // ---- the groups' sums, the first group's last
    wait_lds();
    barrier();
    float* sums = reinterpret_cast<float*>(smem);
    static_assert((KG - 1) * MW * NB * MT * TN * 16 * 256 <= FEW_LDS, "LDS of a compute unit");
    auto place = [&](int g, int m, int n, int i) __attribute__((always_inline)) { return (((((g - 1) * NB + wn) * MW + wm) * MT + m) * TN + n) * 1024 + 64 * i + lane; };
    if (kg > 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int i = 0; i < 16; ++i) sums[place(kg, m, n, i)] = acc[n][m][i];
    }
    wait_lds();
    barrier();
    if (kg > 0) return;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int g = 1; g < KG; ++g)
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[n][m][i] += sums[place(g, m, n, i)];
      const int row = 32 * (wm + MW * m) + fr, rr = t.r0 + min(row, t.M - 1);
      if constexpr (SLAB) {   // (register 4 g + i: weight row 8 g + 4 hi + i)
        float* sp = a.slab + ((int64_t)t.e * a.rows + rr) * a.ncols + t.n0 * NO + wn * FN + 4 * hi;
        if (row < t.M) {
#pragma unroll
          for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int g = 0; g < 4; ++g)
              *reinterpret_cast<f32x4_t*>(sp + 32 * n + 8 * g) = f32x4_t{acc[n][m][4 * g], acc[n][m][4 * g + 1], acc[n][m][4 * g + 2], acc[n][m][4 * g + 3]};
        }
        continue;
      }
      const float sc = a.scale != nullptr ? a.scale[a.sorted != nullptr ? a.sorted[rr] : rr] : 1.0f;
      uint16_t* op = a.out + (int64_t)rr * a.ncols + t.n0 * NO + wn * (NO / NB) + 8 * hi;
      store_row<ACT>([&](int n, int i) __attribute__((always_inline)) { return acc[n][m][i] * sc; }, op, row < t.M, a);
    }
  };
  const int mx = (t.M + 63) / 64;
  if (mx == 1) run(IntC<1>{});
  else if (mx == 2) run(IntC<2>{});
  else if (mx == 3) run(IntC<3>{});
  else run(IntC<4>{});
}

// `tile_rows` of the tiles of 64 and 128 weight rows; what a step takes. Beyond two turns of tiles of 64 those of 128 are faster where experts have few rows, up to four turns a few
// more (whole tiles / 128, layers of 8 experts, gated, on cold weights, us: width 4096 x 14336, 50 rows each 521 / 505, 75 551 / 559; 4096 x 4096, 50 174 / 167, 62 179 / 174, 75 185 / 182,
// 112 193 / 193; 32 of 4096 x 2048, 87 254 / 256).
enum { ROWS_WHOLE = 0, ROWS_64 = 64, ROWS_128 = 96 };
inline int few_tiles(const MoeGemmArgs& a) {
  const int no = a.act >= MOE_ACT_SILU && a.act <= MOE_ACT_GELU ? FN / 2 : FN;
  const int64_t tiles = (int64_t)std::min(a.experts, a.rows) * (a.ncols / no);   // of experts of up to 256 rows
  if (tiles <= a.cus && a.rows <= 192 * (int64_t)a.experts) return ROWS_64;
  return a.rows <= (tiles <= 2 * a.cus ? 144 : tiles <= 4 * a.cus ? 80 : 60) * (int64_t)a.experts ? ROWS_128 : ROWS_WHOLE;
}

template <int ACT, int NB, int OF = OF_EXPERTS> hipError_t launch_few(const MoeGemmArgs& a, hipStream_t s) {
  auto* fn = moe_gemm_few_kernel<ACT, NB, OF>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, FEW_LDS);
  if (e != hipSuccess) return e;
  constexpr int NO = (ACT >= MOE_ACT_SILU && ACT <= MOE_ACT_GELU ? FN / 2 : FN) * NB;
  const int64_t mts = OF != OF_EXPERTS ? a.experts * (int64_t)((a.rows + BM - 1) / BM) : std::min(a.experts, a.rows) + a.rows / BM;   // at most
  const int64_t tiles = mts * (a.ncols / NO);
  hipLaunchKernelGGL(fn, dim3((unsigned)(8 * ((tiles + 7) / 8))), dim3(64 * NW), FEW_LDS, s, a);
  return hipGetLastError();
}

template <int ACT, int OF> hipError_t launch_whole(const MoeGemmArgs& a, bool turn, hipStream_t s) {
  auto* fn = turn ? moe_gemm_kernel<ACT, true, OF> : moe_gemm_kernel<ACT, false, OF>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, NU * UNIT);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(8 * std::max(a.cus / 8, 1)), dim3(64 * NW), NU * UNIT, s, a);
  return hipGetLastError();
}

template <int ACT> hipError_t launch_act(MoeGemmArgs a, hipStream_t s) {
  a.cus = num_cus();
  const int few = a.tile_rows != 0 ? a.tile_rows : few_tiles(a);
  if (few == ROWS_64) return launch_few<ACT, 1>(a, s);
  if (few == ROWS_128) return launch_few<ACT, 2>(a, s);
  // (at most one row tile per expert on average: the places cost 0.6 % where they are all the first, 8 of 4096 x 14336, 1024 rows each)
  constexpr int NO = ACT >= MOE_ACT_SILU && ACT <= MOE_ACT_GELU ? BN / 2 : BN;
  const bool turn = a.rows <= (int64_t)BM * a.experts && 2 * (int64_t)a.experts * (a.ncols / NO) >= a.cus;
  return launch_whole<ACT, OF_EXPERTS>(a, turn, s);
}

template <int ACT, int OF> hipError_t launch_dense(const MoeGemmArgs& a, hipStream_t s) {
  const bool one = a.rows <= BM;
  if (a.tile_rows == ROWS_64) return launch_few<ACT, 1, OF>(a, s);
  if (a.tile_rows == ROWS_128) return launch_few<ACT, 2, OF>(a, s);
  return launch_whole<ACT, OF>(a, one, s);
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
  if (a.tile_rows != 0 && a.tile_rows != ROWS_64 && a.tile_rows != ROWS_128 && (a.tile_rows < 128 || a.tile_rows > 256 || a.tile_rows % 32 != 0)) return hipErrorInvalidValue;
  switch (a.act) {
    case MOE_ACT_NONE: return launch_act<MOE_ACT_NONE>(a, s);
    case MOE_ACT_SILU: return launch_act<MOE_ACT_SILU>(a, s);
    case MOE_ACT_CLAMPED: return launch_act<MOE_ACT_CLAMPED>(a, s);
    case MOE_ACT_GELU: return launch_act<MOE_ACT_GELU>(a, s);
    case MOE_ACT_RELU2: return launch_act<MOE_ACT_RELU2>(a, s);
    default: return hipErrorInvalidValue;
  }
}

// Dense products of prompt steps of a few row tiles by the same kernels. 4096 weight rows are 16 - 32 tiles a row tile, so the parts of K are what fills the
// chip: they go as the "experts" of one set of rows, each into an fp32 slab, which the pass behind the product (norm statistics, RoPE) sums. At 4096 x 14336
// weights 129 rows take 34 us and 3.5 TB/s (34 with 7 parts, 38 with 4 of 64-row tiles), 442 55 (0.94 PFLOP/s), where the library's 64 x 64 and 64 x 128 tiles
// take 55 and 86; the bound is the fetch of the tiles into LDS (10 TB/s). A gate and up product has tiles enough, and its activation on the sums saves
// [rows, 2 ff] out and back: 442 rows of 4096 x 28672 105 -> 96. Which steps take it: prompt_slab_parts, prompt_silu_tiles in src/ops.
hipError_t launch_dense_gemm(MoeGemmArgs a, hipStream_t s) {
  if (a.rows == 0) return hipSuccess;
  const bool slab = a.slab != nullptr;
  if (a.rows < 0 || a.experts < 1 || a.topk != 1 || a.offsets != nullptr || a.sorted != nullptr || !moe_gemm_takes(a)) return hipErrorInvalidValue;
  if (slab ? a.act != MOE_ACT_NONE || a.K % (BK * a.experts) != 0 : a.experts != 1 || a.act != MOE_ACT_SILU) return hipErrorInvalidValue;
  if (a.tile_rows != 0 && a.tile_rows != ROWS_64 && a.tile_rows != ROWS_128 && (a.tile_rows < 128 || a.tile_rows > 256 || a.tile_rows % 32 != 0)) return hipErrorInvalidValue;
  a.cus = num_cus();
  return slab ? launch_dense<MOE_ACT_NONE, OF_PARTS>(a, s) : launch_dense<MOE_ACT_SILU, OF_ONE>(a, s);
}

}  // namespace die
