// S <- diag(g_t) S + k_t v_t^T, o_t = S^T q_t of bf16 prompt portions, g_t = sigmoid(z_t + bias)^(1 / tau) per key channel, in chunks of 16
// tokens on the matrix cores (gfx950). State, decays and results are fp32 and keep their 24 bits.
//
// With G_i = g_1 .. g_i (elementwise over the key channels) and, for j <= i, P_ij = sum_d q_i g_(j+1) .. g_i k_j, a chunk is
//     o = (G q) S + P v        S <- diag(G_16) S + (k G_16 / G)^T v
// All products of decays are multiplied up from their tokens (no quotients), so any decay is fine, zero ones too.
//
// A workgroup is one (sequence, head). One wave per 32 value columns consumes: it owns its columns of S in accumulators, whose layout (row
// 4 (lane / 16) + r in register r) is an operand's with the contraction in another order. D / 32 waves scale q and k by their decays, D / 32
// more form P (a lane runs w = k_j g_(j+1) .. g_i down a column); a step ahead, one barrier per chunk.
//
// fp32 operands enter as three bf16 parts of 8 bits each (exact); against each other the six largest of nine products are formed, against
// v, which is bf16, all three. The products of lower parts are summed apart; the state is rounded once per chunk.
//
// Bound by instruction issue of a consuming and a helping wave per SIMD. 16 heads of 64 x 128 (us, token by token / in chunks): 16 x 1024 tokens 372 / 140, one
// sequence of 1024 319 / 132, 32 x 300 ragged 151 / 82, 1 x 64 of 32 heads 24 / 13. Distance from 64 bits 0.86 - 0.95 of that token by token.
//
// The parts of an infinity are NaN. A wave that finds results or state of its columns not finite goes through the portion once more, token by
// token from the state as it was, and puts what that gives in the place of what is not finite: infinities stay what they are.
#include "chunk_channel.h"
#include "chunk_parts.h"
#include "lane_reduce.h"

namespace die {

namespace {

// Rows k, q of two neighbouring channels and 4 neighbouring tokens on every lane, and their decays: a wave covers 32 channels of a
// chunk (lane % 16: the pair of channels, lane / 16: the quarter of the tokens).
template <int D> struct Rows {
  const bf16_t *kb, *qb, *zb;   // the portion's rows: the head's k, q, z
  int64_t xstride, zstride;
  int L, t0;
  uint32_t d2;
  float inv_tau, bias0, bias1;
  uint32_t k[4], q[4], z[4];   // as loaded
  __device__ __forceinline__ Rows(const GatedLinearArgs& a, int q0, int rows, int h, int pw, int lane) {
    const int g = h / (a.heads / a.groups);
    const bf16_t* x = reinterpret_cast<const bf16_t*>(a.x) + (int64_t)q0 * a.xstride + g * D;
    kb = x + a.koff, qb = x + a.qoff;
    zb = reinterpret_cast<const bf16_t*>(a.z) + (int64_t)q0 * a.zstride + h * D;
    xstride = a.xstride, zstride = a.zstride;
    L = rows, t0 = 4 * (lane >> 4), d2 = 32 * pw + 2 * (lane & 15);
    inv_tau = a.inv_tau, bias0 = a.z_bias[h * D + d2], bias1 = a.z_bias[h * D + d2 + 1];
  }
  __device__ __forceinline__ void fetch(int n) {   // rows of chunk n, at any 2 bytes; beyond the portion its last one
    const uint32_t last = L - n * CT - 1;
    const int64_t row0 = n * CT;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint32_t row = min((uint32_t)(t0 + t), last), at = 2 * (row * (uint32_t)xstride + d2);
      k[t] = *at_bytes<uint32_at2>(kb + row0 * xstride, at);
      q[t] = *at_bytes<uint32_at2>(qb + row0 * xstride, at);
      z[t] = *at_bytes<uint32_at2>(zb + row0 * zstride, 2 * (row * (uint32_t)zstride + d2));
    }
  }
  static __device__ __forceinline__ float decay(float x, float inv_tau) {   // exp(-softplus(-x) / tau), softplus_of<true> with its logarithm ahead of the choice
    const float e = exp_of<true>(-fabsf(x));
    float l = 0.6931471805599453f * __builtin_amdgcn_logf(1.0f + e);
    asm volatile("" : "+v"(l));
    l = e < 9.765625e-4f ? e - 0.5f * e * e : l;
    return exp_of<true>(-(fmaxf(-x, 0.f) + l) * inv_tau);
  }
  // the fetched values -> rows and decays of chunk n (tokens beyond the portion: k = q = 0, g = 1)
  __device__ __forceinline__ void finish(int n, float2 (&ko)[4], float2 (&qo)[4], float2 (&go)[4]) {
    const int last = L - n * CT - 1;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool in = t0 + t <= last;
      asm volatile("" : "+v"(k[t]), "+v"(q[t]), "+v"(z[t]));   // (converted here, not where they are loaded and would be waited for)
      float gx = decay(__uint_as_float(z[t] << 16) + bias0, inv_tau), gy = decay(__uint_as_float(z[t] & 0xffff0000u) + bias1, inv_tau);
      asm volatile("" : "+v"(gx), "+v"(gy));
      const uint32_t kw = in ? k[t] : 0u, qw = in ? q[t] : 0u;
      ko[t] = make_float2(__uint_as_float(kw << 16), __uint_as_float(kw & 0xffff0000u));
      qo[t] = make_float2(__uint_as_float(qw << 16), __uint_as_float(qw & 0xffff0000u));
      go[t] = make_float2(in ? gx : 1.0f, in ? gy : 1.0f);
    }
  }
};

__device__ __forceinline__ bool finite(float x) { return fabsf(x) < INFINITY; }

// A wave's 32 columns of a portion token by token, S [D, 32] (LDS) their state; a lane has one column and half of the channels. o: row 0's
// results, state: what the chunks left, both replaced where they are not finite. (Loops that are not unrolled: a rare way is not to cost the
// kernel registers.)
template <int D, int V>
__device__ __forceinline__ void token_by_token(const GatedLinearArgs& a, int q0, int L, int h, float* S, float* o, float* state) {
  const int lane = threadIdx.x & 63, half = lane >> 5, v0 = (threadIdx.x >> 6) * 32 + (lane & 31);
  const bf16_t* x = reinterpret_cast<const bf16_t*>(a.x) + (int64_t)q0 * a.xstride;
  const bf16_t* z = reinterpret_cast<const bf16_t*>(a.z) + (int64_t)q0 * a.zstride + h * D;
  const int g = h / (a.heads / a.groups) * D;
  float* const own = S + (lane & 31);
#pragma unroll 1
  for (int t = 0; t < L; ++t, x += a.xstride, z += a.zstride) {
    const float v = bf2f(x[a.voff + h * V + v0]);
    float y = 0.f;
#pragma unroll 1
    for (int d = half * (D / 2); d < (half + 1) * (D / 2); ++d) {
      const float s = fmaf(own[32 * d], Rows<D>::decay(bf2f(z[d]) + a.z_bias[h * D + d], a.inv_tau), bf2f(x[a.koff + g + d]) * v);
      own[32 * d] = s;
      y = fmaf(s, bf2f(x[a.qoff + g + d]), y);
    }
    y = xor32_sum(y) * a.qscale;
    float* const at = o + (int64_t)t * a.heads * V + v0;
    if (half == 0 && !finite(*at)) *at = y;
  }
#pragma unroll 1
  for (int d = half * (D / 2); d < (half + 1) * (D / 2); ++d)
    if (!finite(state[d * V + v0])) state[d * V + v0] = own[32 * d];
}

// LDS of a workgroup, in bytes
template <int D> struct Lds {
  static constexpr int NP = D / 32, KP = D + 4;                // waves of either kind of helper; pitch of raw rows (floats)
  static constexpr int XP = 2 * D + 16, DP = 8 * CT + 16;      // pitch of a part's row of G q; of a channel of k G_16 / G
  static constexpr int SX = 3 * CT * XP, SK = D * DP + 4 * D;  // parts of G q; k G_16 / G and G_16: two chunks each
  static constexpr int kd = 2 * SX, pp = kd + 2 * SK;          // P in parts, as pieces in the order of the lanes, two chunks
  static constexpr int raw = pp + 2 * 2048;                    // k | q | decays of the chunk whose P is formed
  static constexpr int part = raw + 12 * CT * KP;              // partial P of every wave, two chunks
  static constexpr int total = part + 2 * 4 * NP * CT * TP;
};

template <int D, int V>
__global__ void __launch_bounds__(2 * V + 4 * D, 1) chunk_channel_kernel(GatedLinearArgs a, RaggedRows r) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  using Z = Lds<D>;
  constexpr int NB = 2, NC = V / (16 * NB), ND = D / 16, NP = Z::NP;
  const int H = a.heads, h = blockIdx.x, s = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int q0 = __builtin_amdgcn_readfirstlane(r.cu_q[s]);
  const int L = __builtin_amdgcn_readfirstlane(r.cu_q[s + 1]) - q0;
  if (L <= 0) return;
  const int nch = (L + CT - 1) / CT;

  if (wave >= NC + NP) {
    // ------------------------------------------------------------------------------------------------ P
    const int pw = wave - NC - NP;
    Rows<D> rows(a, q0, L, h, pw, lane);
    float* const raw = reinterpret_cast<float*>(sm + Z::raw);
    constexpr int KP = Z::KP;
    auto pairs = [&](int n) {   // of chunk n, over the wave's 32 channels; then the loads of the next one
      float2 k[4], q[4], g[4];
      rows.finish(n, k, q, g);
      rows.fetch(min(n + 1, nch - 1));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (a wave reads the channels that it wrote)
      float* to = raw + 4 * lg * KP + 32 * pw + 2 * li;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        *reinterpret_cast<float2*>(to + t * KP) = k[t];
        *reinterpret_cast<float2*>(to + (CT + t) * KP) = q[t];
        *reinterpret_cast<float2*>(to + (2 * CT + t) * KP) = g[t];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      // 4 channels per lane: lane j < 8 (of 8 for the channels) runs down column j, rows j .. 15, then down column 15 - j: 17 steps for any j
      const int j = lane & 7, turn = CT - j;
      const float* ra = raw + 32 * pw + 4 * (lane >> 3) + j * KP;
      const float* rb = ra - j * KP - KP;
      f32x4_t w = {}, at[2][3];
      auto row = [&](int t) {   // k, q, decays of step t's row
        const float* r = (t < turn ? ra : rb) + t * KP;
        at[t & 1][0] = ld4(r), at[t & 1][1] = ld4(r + CT * KP), at[t & 1][2] = ld4(r + 2 * CT * KP);
      };
      float p[CT + 1];
      row(0);
#pragma unroll
      for (int t = 0; t <= CT; ++t) {
        if (t < CT) row(t + 1);
        __builtin_amdgcn_sched_barrier(0);   // (a step's reads stay ahead of the step before it)
        const f32x4_t* x = at[t & 1];
        const bool own = t == 0 || (t > CT / 2 && t == turn);
        p[t] = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = w[e] * x[2][e];
          w[e] = own ? x[0][e] : v;
          p[t] = fmaf(x[1][e], w[e], p[t]);
        }
      }
      // sums over the 8 lanes of a column: of 8 steps, one is left to each of them
      float* pm = reinterpret_cast<float*>(sm + Z::part) + (n % 2 * NP + pw) * (CT * TP);
      auto put = [&](int t, float x) { pm[t < turn ? (j + t) * TP + j : (t - 1) * TP + CT - 1 - j] = x; };
      const bool b3 = lane & 8, b4 = lane & 16;
      auto two = [](float x, float y) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
      };
      auto four = [](float x, float y) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
      };
#pragma unroll
      for (int u = 0; u < CT; u += 8) {
        const float x = four(two(p[u], p[u + 1]), two(p[u + 2], p[u + 3])), y = four(two(p[u + 4], p[u + 5]), two(p[u + 6], p[u + 7]));
        const float give = dpp_ror8(b3 ? x : y);
        put(u + (b3 ? 4 : 0) + (b4 ? 2 : 0) + (lane >> 5), (b3 ? y : x) + give);
      }
      float y = xor16_sum(xor32_sum(p[CT]));
      y += dpp_ror8(y);
      if (lane < 8) put(CT, y);
    };
    auto sum = [&](int n) {   // P of chunk n from its partial sums, behind a barrier
      if (pw != 0) return;
      const float* pm = reinterpret_cast<const float*>(sm + Z::part) + n % 2 * NP * (CT * TP) + li * TP + 4 * lg;
      f32x4_t p = ld4(pm);
#pragma unroll
      for (int w = 1; w < NP; ++w) p += ld4(pm + w * CT * TP);
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = 4 * lg + e <= li ? p[e] : 0.f;
      uint32_t x[3], y[3];
      split3(p[0], p[1], x);
      split3(p[2], p[3], y);
      uint4* to = reinterpret_cast<uint4*>(sm + Z::pp + n % 2 * 2048) + lane;
      to[0] = make_uint4(x[0], y[0], x[1], y[1]);
      to[64] = make_uint4(x[0], y[0], x[2], y[2]);
    };
    rows.fetch(0);
    pairs(0);
    __syncthreads();
    sum(0);
    if (nch > 1) pairs(1);
    __syncthreads();
    for (int n = 0; n < nch; ++n) {
      if (n + 1 < nch) sum(n + 1);
      if (n + 2 < nch) pairs(n + 2);
      __syncthreads();
    }
    return;
  }

  if (wave >= NC) {
    // ------------------------------------------------------------------------------------------------ scaled rows
    const int pw = wave - NC, d2 = 32 * pw + 2 * li;
    Rows<D> rows(a, q0, L, h, pw, lane);
    auto scale = [&](int n) {   // of chunk n; then the loads of the next one
      float2 k[4], q[4], g[4];
      rows.finish(n, k, q, g);
      rows.fetch(min(n + 1, nch - 1));
      const float2 all = make_float2(g[0].x * g[1].x * (g[2].x * g[3].x), g[0].y * g[1].y * (g[2].y * g[3].y));
      float2 G, P;
      around(all.x, lg, G.x, P.x);
      around(all.y, lg, G.y, P.y);
      char* to = sm + n % 2 * Z::SX + 4 * lg * Z::XP;
      to += 2 * ((d2 & ~31) + 8 * (d2 >> 2 & 3) + 4 * (d2 >> 4 & 1) + (d2 & 3));   // in the order of the accumulators' rows
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        G.x *= g[t].x;
        G.y *= g[t].y;
        uint32_t p[3];
        split3(q[t].x, G.x, q[t].y, G.y, p);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint32_t*>(to + (i * CT + t) * Z::XP) = p[i];
      }
      char* kd = sm + Z::kd + n % 2 * Z::SK;
      float x0[4], x1[4], y0[4], y1[4];
#pragma unroll
      for (int t = 3; t >= 0; --t) {
        x0[t] = k[t].x, y0[t] = P.x;
        x1[t] = k[t].y, y1[t] = P.y;
        P.x *= g[t].x;
        P.y *= g[t].y;
      }
      split_store(kd + d2 * Z::DP + 32 * lg, x0, y0);
      split_store(kd + (d2 + 1) * Z::DP + 32 * lg, x1, y1);
      if (lg == 3) *reinterpret_cast<float2*>(kd + D * Z::DP + 4 * d2) = G;
    };
    rows.fetch(0);
    __syncthreads();
    scale(0);
    __syncthreads();
    for (int n = 0; n < nch; ++n) {
      if (n + 1 < nch) scale(n + 1);
      __syncthreads();
    }
    return;
  }

  // -------------------------------------------------------------------------------------------------- consumers
  const int v0 = 16 * NB * wave + li;
  const bool fresh = r.positions[q0] <= 0;
  float* st = a.state + ((int64_t)__builtin_amdgcn_readfirstlane(r.state_slots[s]) * H + h) * (D * V);
  uint32_t so = 4 * lg * V + v0;
  uint16_t vr[NB][4];   // values of the current chunk, as loaded
  const bf16_t* vb = reinterpret_cast<const bf16_t*>(a.x) + (int64_t)q0 * a.xstride + a.voff + h * V;
  auto fetch = [&](int n) {
    const uint32_t last = L - n * CT - 1;
    const bf16_t* x = vb + (int64_t)(n * CT) * a.xstride;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t at = 2 * (min((uint32_t)(4 * lg + e), last) * (uint32_t)a.xstride + v0);
#pragma unroll
      for (int c = 0; c < NB; ++c) vr[c][e] = *at_bytes<uint16_t>(x, at + 32 * c);
    }
  };
  fetch(0);
  f32x4_t S[ND][NB];
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float y = st[so + (16 * t + e) * V + 16 * c];
        S[t][c][e] = fresh ? 0.f : y;   // (a new sequence reads its slot but not its content)
      }
  float odd_sum = 0.f;   // 0 as long as all results are finite
  __syncthreads();
  __syncthreads();
  for (int n = 0; n < nch; ++n) {
    // ---- (G q) S: 32 channels of 16 columns at a time, the next ones' parts cut beside the products of the current ones
    f32x4_t qs[NB] = {}, ql[NB] = {};   // ql: the products of lower parts
    const char* xa = sm + n % 2 * Z::SX + li * Z::XP + 16 * lg;
    bf16x8_t qf[2][3], sf[2][3];
    auto rows_of = [&](int t) {
#pragma unroll
      for (int i = 0; i < 3; ++i) qf[t & 1][i] = ldf(xa + i * CT * Z::XP + 64 * t);
    };
    auto cut = [&](int b) {
      float x[8];
      uint32_t p[3][4];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = S[2 * (b / NB) + e / 4][b % NB][e % 4];
      split3<4>(x, p);
#pragma unroll
      for (int i = 0; i < 3; ++i) sf[b & 1][i] = frag(p[i][0], p[i][1], p[i][2], p[i][3]);
    };
    rows_of(0);
    cut(0);
#pragma unroll
    for (int b = 0; b < ND / 2 * NB; ++b) {
      const int t = b / NB, c = b % NB;
      __builtin_amdgcn_sched_barrier(0);
      if (c == 0 && t + 1 < ND / 2) rows_of(t + 1);
      if (b + 1 < ND / 2 * NB) cut(b + 1);
#pragma unroll
      for (int i = 0; i < 3; ++i)   // all but the products below 2^-24 of the largest
#pragma unroll
        for (int j = 0; i + j < 3; ++j) (i + j > 0 ? ql : qs)[c] = mm(qf[t & 1][i], sf[b & 1][j], (i + j > 0 ? ql : qs)[c]);
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- the values as operands: 4 tokens of a column
    uint32_t va[NB], vc[NB];
    const bool whole = n * CT + CT <= L;
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      va[c] = vr[c][0] | (uint32_t)vr[c][1] << 16;
      vc[c] = vr[c][2] | (uint32_t)vr[c][3] << 16;
      asm volatile("" : "+v"(va[c]), "+v"(vc[c]));
    }
    if (!whole) {   // (rows beyond the portion: a zero weight times an infinite value would count)
      const int left = L - n * CT - 4 * lg;
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        va[c] &= (left > 0 ? 0xffffu : 0u) | (left > 1 ? 0xffff0000u : 0u);
        vc[c] &= (left > 2 ? 0xffffu : 0u) | (left > 3 ? 0xffff0000u : 0u);
      }
    }
    fetch(min(n + 1, nch - 1));
    // a zero of P times an infinite or NaN value of a later token would reach earlier rows: such values enter P v as zeros and the rows from
    // their token on become NaN
    uint32_t za[NB], zc[NB], top = 0;
    int first[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      za[c] = va[c], zc[c] = vc[c], first[c] = CT;
      top |= ((va[c] & 0x7f807f80u) + 0x00800080u) | ((vc[c] & 0x7f807f80u) + 0x00800080u);
    }
    const bool odd = __ballot((top & 0x80008000u) != 0) != 0;
    if (odd) {
#pragma unroll
      for (int c = 0; c < NB; ++c) {
#pragma unroll
        for (int e = 3; e >= 0; --e) {
          uint32_t& w = e < 2 ? za[c] : zc[c];
          const uint32_t half = e & 1 ? 0xffff0000u : 0xffffu, inf = 0x7f807f80u & half;
          if ((w & inf) == inf) first[c] = 4 * lg + e, w &= ~half;
        }
        first[c] = min(first[c], __shfl_xor(first[c], 16, 64));
        first[c] = min(first[c], __shfl_xor(first[c], 32, 64));
      }
    }
    const uint4* pp = reinterpret_cast<const uint4*>(sm + Z::pp + n % 2 * 2048) + lane;
    const bf16x8_t p0 = __builtin_bit_cast(bf16x8_t, pp[0]), p1 = __builtin_bit_cast(bf16x8_t, pp[64]);
#pragma unroll
    for (int c = 0; c < NB; ++c) {   // (h, m) v and l v
      ql[c] = mm(p1, frag(0u, 0u, za[c], zc[c]), ql[c]);
      qs[c] = mm(p0, frag(za[c], zc[c], za[c], zc[c]), qs[c]);
    }
    float* op = a.out + ((int64_t)(q0 + n * CT) * H + h) * V;
    const uint32_t hv = H * V, at = 4 * (4 * lg * hv + v0);
    f32x4_t o[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[c][e] = (qs[c][e] + ql[c][e]) * a.qscale;
        if (odd) o[c][e] = 4 * lg + e >= first[c] ? __builtin_nanf("") : o[c][e];
        odd_sum = fmaf(o[c][e], 0.f, odd_sum);
      }
    if (whole) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < NB; ++c) *const_cast<float*>(at_bytes<float>(op + (int64_t)e * hv + 16 * c, at)) = o[c][e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n * CT + 4 * lg + e < L) {
#pragma unroll
          for (int c = 0; c < NB; ++c) *const_cast<float*>(at_bytes<float>(op + (int64_t)e * hv + 16 * c, at)) = o[c][e];
        }
    }
    // ---- the state: 16 channels' products beside the sums of the ones before
    const char* ka = sm + Z::kd + n % 2 * Z::SK + li * Z::DP + 32 * lg;
    const float* end = reinterpret_cast<const float*>(sm + Z::kd + n % 2 * Z::SK + D * Z::DP) + 4 * lg;   // G_16
    bf16x8_t k0[2], k1[2], v2[NB], v1[NB];
    f32x4_t G[2], x[2][NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) v2[c] = frag(va[c], vc[c], va[c], vc[c]), v1[c] = frag(0u, 0u, va[c], vc[c]);
    auto load = [&](int t) {
      k0[t & 1] = ldf(ka + 16 * t * Z::DP), k1[t & 1] = ldf(ka + 16 * t * Z::DP + 16);
      G[t & 1] = ld4(end + 16 * t);
    };
    auto add = [&](int t) {
#pragma unroll
      for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[t][c][e] = fmaf(S[t][c][e], G[t & 1][e], x[t & 1][c][e]);   // one rounding of the state per chunk
    };
    load(0);
#pragma unroll
    for (int t = 0; t < ND; ++t) {
      __builtin_amdgcn_sched_barrier(0);
      if (t > 0) add(t - 1);
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        const f32x4_t zero = {};
        x[t & 1][c] = mm(k0[t & 1], v2[c], mm(k1[t & 1], v1[c], zero));
      }
      if (t + 1 < ND) load(t + 1);
    }
    add(ND - 1);
    __syncthreads();
  }
  asm volatile("" : "+v"(so));   // the loads' offsets are formed again, not kept through the loop
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) odd_sum = fmaf(S[t][c][e], 0.f, odd_sum);
  const bool again = __ballot(odd_sum != 0.f) != 0;
  float* const was = reinterpret_cast<float*>(sm) + wave * (D * 16 * NB);   // the state's columns as they were (nothing else is in LDS any more)
  if (again) {
#pragma unroll 1
    for (int i = lane; i < D * 16 * NB; i += 64) was[i] = fresh ? 0.f : st[i / (16 * NB) * V + 16 * NB * wave + i % (16 * NB)];
    __threadfence();
  }
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) st[so + (16 * t + e) * V + 16 * c] = S[t][c][e];
  if (again) {
    __threadfence();
    token_by_token<D, V>(a, q0, L, h, was, a.out + ((int64_t)q0 * H + h) * V, st);
  }
}

template <int D, int V> hipError_t launch_one(const GatedLinearArgs& a, RaggedRows r, hipStream_t s) {
  constexpr size_t smem = Lds<D>::total > 4 * D * V ? Lds<D>::total : 4 * D * V;   // (the chunks', then the whole state where it is gone through again)
  static_assert(smem <= 160 * 1024, "LDS of a compute unit");
  const auto fn = chunk_channel_kernel<D, V>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(a.heads, r.num_seqs), dim3(2 * V + 4 * D), smem, s, a, r);
  return hipGetLastError();
}

}  // namespace

bool chunk_channel_fits(const GatedLinearArgs& a, int rows, int num_seqs) {
  const bool sizes = (a.dim == 64 && (a.vdim == 64 || a.vdim == 128 || a.vdim == 256)) || (a.dim == 128 && (a.vdim == 64 || a.vdim == 128));
  const bool near = a.xstride < (1 << 26) && a.zstride < (1 << 26);   // (offsets within a chunk are 32-bit)
  const int64_t n = num_seqs, wgs = a.heads * n, cus = num_cus();
  const bool narrow = a.vdim == 64, wide = a.vdim == 256;
  const int from = wgs <= cus ? (narrow && a.dim == 64 ? 17 : wide ? 16 : 14) : wgs <= 2 * cus ? (narrow ? 48 : 20) : narrow ? 80 : wide ? 24 : 36;
  return !a.f32 && a.z != nullptr && sizes && near && rows >= from * n;
}

hipError_t launch_chunk_channel(const GatedLinearArgs& a, RaggedRows r, hipStream_t s) {
  if (a.dim == 64) return a.vdim == 64 ? launch_one<64, 64>(a, r, s) : a.vdim == 128 ? launch_one<64, 128>(a, r, s) : launch_one<64, 256>(a, r, s);
  return a.vdim == 64 ? launch_one<128, 64>(a, r, s) : launch_one<128, 128>(a, r, s);
}

}  // namespace die
