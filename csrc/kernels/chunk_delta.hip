// The gated delta rule S <- diag(g_t) S, u_t = beta_t (v_t - S^T k_t), S <- S + k_t u_t^T, o_t = S^T q_t of prompt portions in
// chunks of 16 tokens on the matrix cores (gfx950), normed and gated. State, operands and sums are fp32, as in the token-by-token
// kernel, in another order; decays, norm and gate are the same functions to the bit (hardware exponentials, a reciprocal and a
// reciprocal root in norm and gate took 2 - 4 % less and rounded 12 of 262144 gated values to the other neighbour).
//
// With G_i = g_1 .. g_i (elementwise over the key channels) and, for j <= i, M_ij = sum_d k_i g_(j+1) .. g_i k_j and P_ij the same
// with q_i, a chunk is
//     u = T B (v - (G k) S),  T = (I + B tril(M, -1))^-1        o = (G q) S + P u        S <- diag(G_16) S + (k G_16 / G)^T u
// All products of decays are multiplied up from their tokens (no quotients), so any decay is fine, zero ones too.
//
// A workgroup is one (sequence, head). One wave per 32 value columns consumes: it owns its columns of S in accumulators, whose
// layout (row 4 (lane / 16) + r in register r) is an operand's with the contraction in another order, so that S, v and u are
// operands as they stand. D / 32 more waves produce what does not depend on S: decays, scaled k and q (into LDS), M and P
// (a lane runs w = k_j g_(j+1) .. g_i down a column), and T by substitution. Two barriers per chunk:
//     consume (G k) S, (G q) S of chunk n      | M, P of n + 1, decays of n + 2
//     consume u, o, S of chunk n               | T of n + 1, scaled k and q of n + 2
//
// fp32 operands enter as three bf16 parts of 8 bits each (exact), of whose nine products the six largest are formed (the rest are
// below 2^-25 of the whole): the fp32 matrix instructions run at the vector units' rate and in their place (7.2 us a chunk; these
// 5.0). Where a sum enters the state, lower parts are summed apart and added once, and of T the part below its diagonal is
// multiplied; the state is rounded once per chunk instead of twice per token. Its error against 64 bits (2-norm; 1 - 16 sequences of
// 32 - 1400 rows, 12 draws each) is 0.2 - 1.0e-7, 0.90 - 0.93 of that of the token-by-token kernel, decays per head and per channel.
//
// An infinite key or value makes the rows from its token on and the state NaN (a part of an infinity is NaN), where token by token some
// of them may stay infinite; earlier rows and other sequences are as they are.
//
// Bound by the issue of vector and matrix instructions of the two waves per SIMD (LDS leaves one workgroup per compute unit):
// per chunk 700 vector and 150 matrix instructions of a consuming wave beside 900 of a producing one, 11000 cycles. 16 sequences of
// 300 - 1000 rows, 16 heads, dim = vdim = 128, decays per channel: 914 -> 325 us; one sequence of 1024 rows: 874 -> 310 us.
#include "chunk_delta.h"
#include "common.h"
#include "lane_reduce.h"

namespace die {

namespace {

constexpr int CT = 16;        // tokens of a chunk
constexpr int TP = CT + 4;    // pitch of the 16-wide arrays (floats): 16-byte reads of 16 rows fall on different banks

__device__ __forceinline__ f32x4_t mm(float a, float b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float dpp_ror8(float x) {   // of lane ^ 8
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false));
}
// the value of lane E of the own quad
template <int E> __device__ __forceinline__ float of_quad(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), E * 0x55, 0xf, 0xf, true));
}
__device__ __forceinline__ f32x4_t ld4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }

// x = h + m + l in bf16 parts, exact (8 bits each, rounded to nearest): pairs of values, packed
__device__ __forceinline__ void split3(float x, float y, uint32_t (&p)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    p[i] = pack2(x, y);
    x -= __uint_as_float(p[i] << 16);
    y -= __uint_as_float(p[i] & 0xffff0000u);
  }
}
// 4 consecutive places of a contraction as operands of 8 places: (h, m) and (h, l)
__device__ __forceinline__ void split_store(char* to, const float* x) {
  uint32_t a[3], b[3];
  split3(x[0], x[1], a);
  split3(x[2], x[3], b);
  *reinterpret_cast<uint4*>(to) = make_uint4(a[0], b[0], a[1], b[1]);
  *reinterpret_cast<uint4*>(to + 16) = make_uint4(a[0], b[0], a[2], b[2]);
}
__device__ __forceinline__ bf16x8_t ldf(const char* p) { return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(p)); }
__device__ __forceinline__ bf16x8_t frag(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return __builtin_bit_cast(bf16x8_t, make_uint4(a, b, c, d));
}
__device__ __forceinline__ f32x4_t mm(bf16x8_t a, bf16x8_t b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// LDS of a workgroup, in bytes
template <int D, int NC> struct Lds {
  static constexpr int KP = D + 4, NP = D / 32;              // pitch of raw rows (floats), producing waves
  static constexpr int XP = 2 * D + 16, DP = 8 * CT + 16;    // pitch of a part's row of G k, G q; of a channel of k G_16 / G, a row of P
  static constexpr int SX = 6 * CT * XP;                     // (k, q) x 3 parts of G x; two chunks
  static constexpr int SK = D * DP + 4 * D + 4 * CT;         // k G_16 / G, G_16, beta; three chunks
  static constexpr int kd = 2 * SX;
  static constexpr int raw = kd + 3 * SK;                    // k | q rows of the chunk whose pairs are formed
  static constexpr int gates = raw + 8 * CT * KP;            // decays of two chunks
  static constexpr int part = gates + 8 * CT * KP;           // partial M | P of every producing wave
  static constexpr int low = part + 8 * NP * CT * TP;        // B tril(M)
  static constexpr int STP = 4 * CT * TP + CT * DP;          // T | P; two chunks
  static constexpr int tp = low + 4 * CT * TP;
  static constexpr int ssq = tp + 2 * STP;                   // sums of squares of the consuming waves, two chunks
  static constexpr int total = ssq + 8 * NC * CT;
  static_assert(total <= 160 * 1024, "LDS of a compute unit");
};

template <int D, int NC, bool CD>
__global__ void __launch_bounds__(64 * NC + 2 * D, 1) chunk_delta_kernel(GatedDeltaArgs a, RaggedRows r) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  using Z = Lds<D, NC>;
  constexpr int V = 32 * NC, ND = D / 16, KP = Z::KP, NP = Z::NP;
  const DeltaShape& sh = a.sh;
  const int H = sh.heads, GH = sh.kv_heads, C = sh.channels();
  const int h = blockIdx.x, s = blockIdx.y, kh = h / (H / GH);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int q0 = __builtin_amdgcn_readfirstlane(r.cu_q ? r.cu_q[s] : s);
  const int L = __builtin_amdgcn_readfirstlane(r.cu_q ? r.cu_q[s + 1] - q0 : 1);
  if (L <= 0 || L < a.cut) return;
  if (a.cut > 0 && !divided(r.cu_q, r.num_seqs, r.total_rows, a.cut, a.longest)) return;
  const int nch = (L + CT - 1) / CT;

  if (wave >= NC) {
    // ------------------------------------------------------------------------------------------------ producers
    const int pw = wave - NC, pt = 64 * pw + lane;
    const int d = pt % D;       // gates: channel d, all tokens or half of them
    const bool isq = pt >= D;
    constexpr int HT = CD ? CT / 2 : CT;   // decays per thread: per channel half of a chunk's, per head all of them
    const int t0 = CD && isq ? HT : 0;
    const int d2 = 2 * (pt % (D / 2)), hf = pt / (D / 2) % 2;   // rows: channels d2, d2 + 1 of q (isq) or k, half hf of the tokens
    const float expA = CD ? expf(a.A_log[h]) : 0.f, zb = CD ? a.z_bias[h * D + d] : 0.f;
    const float* src = a.qkv32 + (isq ? 0 : GH * D) + kh * D + d2;
    const bf16_t* zs = reinterpret_cast<const bf16_t*>(a.z) + h * D + d;
    const int bw = CD ? H : 2 * H;
    float2 x[CT / 2];
    float gz[HT], bt = 0.f;
    float* const raw = reinterpret_cast<float*>(sm + Z::raw);
    float* const gates_at = reinterpret_cast<float*>(sm + Z::gates);
    float* const part = reinterpret_cast<float*>(sm + Z::part);
    auto fetch_gates = [&](int n) {
      const int64_t row0 = q0 + n * CT;
      const int last = L - n * CT - 1;
      const bf16_t* zr = zs + row0 * a.zstride;
      const float* gr = a.bg + row0 * bw + H + h;
#pragma unroll
      for (int t = 0; t < HT; ++t) {
        const int row = min(t0 + t, last);
        gz[t] = CD ? bf2f(zr[row * (int)a.zstride]) : gr[row * bw];
      }
    };
    auto gates = [&](int n) {   // the decays of chunk n to LDS, then the loads of the next ones
      float* to = gates_at + n % 2 * CT * KP + t0 * KP + d;
      const int last = L - n * CT - 1;
      float g[HT];
#pragma unroll
      for (int t = 0; t < HT; ++t) {
        g[t] = gz[t];
        if constexpr (CD) {   // softplus_of<true>, its logarithm ahead of the choice
          const float z = gz[t] + zb, e = exp_of<true>(-fabsf(z));
          float l = 0.6931471805599453f * __builtin_amdgcn_logf(1.0f + e);
          asm volatile("" : "+v"(l));
          l = e < 9.765625e-4f ? e - 0.5f * e * e : l;
          g[t] = exp_of<true>(-expA * (fmaxf(z, 0.f) + l));
        }
      }
#pragma unroll
      for (int t = 0; t < HT; ++t)   // (tokens beyond the portion: k = q = beta = 0, g = 1)
        if (CD || !isq) to[t * KP] = t0 + t <= last ? g[t] : 1.0f;
      if (n + 1 < nch) fetch_gates(n + 1);
    };
    auto fetch = [&](int n) {
      const int64_t row0 = q0 + n * CT;
      const int last = L - n * CT - 1;
#pragma unroll
      for (int t = 0; t < CT / 2; ++t) {
        const float* r = src + row0 * C;
        const int i = min(CT / 2 * hf + t, last) * C;
        x[t] = make_float2(r[i], r[i + 1]);
      }
      if (pt < CT) bt = a.bg[(row0 + min(pt, last)) * bw + h];
    };
    auto scale = [&](int n) {   // scaled rows and raw rows of chunk n; then the loads of the next one
      constexpr int HR = CT / 2;
      const float* gs = gates_at + n % 2 * CT * KP + d2;
      float2 g[HR], o[HR];   // decays of the own and of the other half
#pragma unroll
      for (int t = 0; t < HR; ++t) {
        g[t] = *reinterpret_cast<const float2*>(gs + (HR * hf + t) * KP);
        o[t] = *reinterpret_cast<const float2*>(gs + (HR - HR * hf + t) * KP);
      }
      float2 all = o[0];
#pragma unroll
      for (int t = 1; t < HR; ++t) all.x *= o[t].x, all.y *= o[t].y;
      float2 G = hf ? all : make_float2(1.0f, 1.0f);
      char* to = sm + n % 2 * Z::SX + (isq ? 3 * CT * Z::XP : 0) + HR * hf * Z::XP;
      to += 2 * ((d2 & ~31) + 8 * (d2 >> 2 & 3) + 4 * (d2 >> 4 & 1) + (d2 & 3));   // in the order of the accumulators' rows
      float* rw = raw + (isq ? CT * KP : 0) + HR * hf * KP + d2;
#pragma unroll
      for (int t = 0; t < HR; ++t) {
        const bool in = n * CT + HR * hf + t < L;
        x[t].x = in ? x[t].x : 0.f;
        x[t].y = in ? x[t].y : 0.f;
        G.x *= g[t].x;
        G.y *= g[t].y;
        uint32_t p[3];
        split3(x[t].x * G.x, x[t].y * G.y, p);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint32_t*>(to + (i * CT + t) * Z::XP) = p[i];
        *reinterpret_cast<float2*>(rw + t * KP) = x[t];
      }
      char* kd = sm + Z::kd + n % 3 * Z::SK;
      float* end = reinterpret_cast<float*>(kd + D * Z::DP);   // G_16, beta
      if (!isq) {
        float2 P = hf ? make_float2(1.0f, 1.0f) : all;
        float y0[HR], y1[HR];
#pragma unroll
        for (int t = HR - 1; t >= 0; --t) {
          y0[t] = x[t].x * P.x;
          y1[t] = x[t].y * P.y;
          P.x *= g[t].x;
          P.y *= g[t].y;
        }
#pragma unroll
        for (int t = 0; t < HR; t += 4) {
          split_store(kd + d2 * Z::DP + 8 * (HR * hf + t), y0 + t);
          split_store(kd + (d2 + 1) * Z::DP + 8 * (HR * hf + t), y1 + t);
        }
        if (hf) *reinterpret_cast<float2*>(end + d2) = G;
      }
      if (pt < CT) end[D + pt] = n * CT + pt < L ? bt : 0.f;
      if (n + 1 < nch) fetch(n + 1);
    };
    auto pairs = [&](int n) {   // of the chunk whose raw rows are staged, over the wave's 32 channels, 4 per lane
      // lane j < 8 (of 8 for the channels) runs down column j, rows j .. 15, then down column 15 - j: 17 steps for any j
      const int j = lane & 7, turn = CT - j;
      const bool b3 = lane & 8, b4 = lane & 16;
      const float* ra = raw + 32 * pw + 4 * (lane >> 3) + j * KP;
      const float* rb = ra - j * KP - KP;
      const int og = (Z::gates - Z::raw) / 4 + n % 2 * CT * KP;
      f32x4_t w = {}, at[2][3];
      auto row = [&](int t) {   // k, q, decays of step t's row
        const float* r = (t < turn ? ra : rb) + t * KP;
        at[t & 1][0] = ld4(r), at[t & 1][1] = ld4(r + CT * KP), at[t & 1][2] = ld4(r + og);
      };
      float* pm = part + (lane >> 5) * (NP * CT * TP) + pw * CT * TP;   // low lanes keep M, high ones P
      auto put = [&](int t, float x) { pm[t < turn ? (j + t) * TP + j : (t - 1) * TP + CT - 1 - j] = x; };
      float one = 0.f, two = 0.f;
      row(0);
#pragma unroll
      for (int t = 0; t <= CT; ++t) {
        if (t < CT) row(t + 1);
        if constexpr (NC < 8) __builtin_amdgcn_sched_barrier(0);   // (a step's reads stay ahead of the step before it)
        const f32x4_t* x = at[t & 1];
        const bool own = t == 0 || (t > CT / 2 && t == turn);
        float m = 0.f, p = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = w[e] * x[2][e];
          w[e] = own ? x[0][e] : v;
          m = fmaf(x[0][e], w[e], m);
          p = fmaf(x[1][e], w[e], p);
        }
        // sums over the lanes of a column: 4 steps' values are left in one register
        float y;
        {
          const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(p), false, false);
          y = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }
        if (t == CT) {
          y = xor16_sum(y);
          y += dpp_ror8(y);
          if (!b3 && !b4) put(t, y);
        } else if (t % 2 == 0) {
          one = y;
        } else {
          const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(one), __float_as_uint(y), false, false);
          y = __uint_as_float(r[0]) + __uint_as_float(r[1]);
          if (t % 4 == 1) {
            two = y;
          } else {
            const float give = dpp_ror8(b3 ? two : y);
            put(t - 3 + (b3 ? 2 : 0) + (b4 ? 1 : 0), (b3 ? y : two) + give);
          }
        }
      }
    };
    auto solve = [&](int n) {   // T and P of chunk n, by the last wave
      if (pw != NP - 1) return;
      const float beta = reinterpret_cast<const float*>(sm + Z::kd + n % 3 * Z::SK + D * Z::DP)[D + li];
      f32x4_t m = {}, p = {};
      const float* pm = part + li * TP + 4 * lg;
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        m += ld4(pm + q * CT * TP);
        p += ld4(pm + (NP + q) * CT * TP);
      }
      float* lo = reinterpret_cast<float*>(sm + Z::low);
      float* T = reinterpret_cast<float*>(sm + Z::tp + n % 2 * Z::STP);
#pragma unroll
      for (int e = 0; e < 4; ++e) {   // row li, columns 4 lg ..
        const int j = 4 * lg + e;
        m[e] = j < li ? beta * m[e] : 0.f;
        p[e] = j <= li ? p[e] : 0.f;
      }
      *reinterpret_cast<f32x4_t*>(lo + li * TP + 4 * lg) = m;
      const float pe[4] = {p[0], p[1], p[2], p[3]};
      split_store(reinterpret_cast<char*>(T + CT * TP) + li * Z::DP + 32 * lg, pe);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      // lane (li, lg): rows 4 lg .. of column li of the inverse; 4 rows are solved at a time and passed to the ones below
      f32x4_t c[4][4];   // rows 4 lg + r of B tril(M), columns 4 b ..
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) c[b][r] = ld4(lo + (4 * lg + r) * TP + 4 * b);
      float t[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) t[r] = 4 * lg + r == li ? 1.0f : 0.f;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        float x[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x[r] = t[r];
#pragma unroll
          for (int k = 0; k < r; ++k) x[r] = fmaf(-c[b][r][k], x[k], x[r]);
        }
        float y[4], z[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = b < 3 ? __shfl(x[r], 16 * b + li, 64) : 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          z[r] = t[r];
#pragma unroll
          for (int k = 0; k < 4; ++k) z[r] = fmaf(-c[b][r][k], y[k], z[r]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] = lg == b ? x[r] : lg > b ? z[r] : t[r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) T[(4 * lg + r) * TP + li] = 4 * lg + r > li ? t[r] : 0.f;   // (T - 1)
    };
    fetch_gates(0);
    fetch(0);
    gates(0);
    __syncthreads();
    scale(0);
    if (nch > 1) gates(1);
    __syncthreads();
    pairs(0);
    __syncthreads();
    solve(0);
    if (nch > 1) scale(1);
    __syncthreads();
    for (int n = 0; n < nch; ++n) {
      if (n + 1 < nch) pairs(n + 1);
      if (n + 2 < nch) gates(n + 2);
      __syncthreads();
      if (n + 1 < nch) solve(n + 1);
      if (n + 2 < nch) scale(n + 2);
      __syncthreads();
    }
    return;
  }

  // -------------------------------------------------------------------------------------------------- consumers
  const int v0 = 32 * wave + li;
  const bool fresh = r.positions[q0] <= 0;
  float* st = a.state + ((int64_t)__builtin_amdgcn_readfirstlane(r.state_slots[s]) * H + h) * (D * V);
  uint32_t so = 4 * lg * V + v0;
  f32x4_t S[ND][2];
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float y = st[so + (16 * t + e) * V + 16 * c];
        S[t][c][e] = fresh ? 0.f : y;   // (a new sequence reads its slot but not its content)
      }
  const float nw[2] = {a.norm_w[v0], a.norm_w[v0 + 16]};
  float vv[2][4], gt[2][4], gd[2][4];   // values and gates of the current chunk, gates of the one whose results are pending
  f32x4_t o[2];
  auto fetch = [&](int n) {
    const int64_t row0 = q0 + n * CT;
    const float* vr = a.qkv32 + row0 * C + 2 * GH * D + h * V;
    const bf16_t* gr = reinterpret_cast<const bf16_t*>(a.gate) + row0 * a.gstride + h * V;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = min(4 * lg + e, L - n * CT - 1);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        vv[c][e] = vr[row * C + v0 + 16 * c];
        gt[c][e] = bf2f(gr[row * (int)a.gstride + v0 + 16 * c]);
      }
    }
  };
  float y[2][4];
  auto norm = [&](int n) {   // the results of chunk n: their sums of squares are complete behind a barrier
    const float* q = reinterpret_cast<const float*>(sm + Z::ssq) + n % 2 * NC * CT + 4 * lg;
    f32x4_t ss = {};
#pragma unroll
    for (int w = 0; w < NC; ++w) ss += ld4(q + w * CT);
    // (the four rows' factors by four lanes, one each)
    const float own = (lane & 2) != 0 ? ((lane & 1) != 0 ? ss[3] : ss[2]) : ((lane & 1) != 0 ? ss[1] : ss[0]);
    const float f = a.mult / sqrtf(own * (1.0f / V) + a.eps);
    const float rs[4] = {of_quad<0>(f), of_quad<1>(f), of_quad<2>(f), of_quad<3>(f)};
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int c = 0; c < 2; ++c) y[c][e] = o[c][e] * rs[e] * nw[c] * gated(a.gate_sigmoid ? 1.0f : gd[c][e], gd[c][e]);
  };
  auto store = [&](int n) {
    bf16_t* to = reinterpret_cast<bf16_t*>(a.out) + (int64_t)(q0 + n * CT) * a.ostride + h * V;
#pragma unroll
    for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(y[0][e]), "+v"(y[1][e]));   // all formed here, not behind the conditions
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n * CT + 4 * lg + e < L) {
        to[(4 * lg + e) * (int)a.ostride + v0] = f2bf(y[0][e]);
        to[(4 * lg + e) * (int)a.ostride + v0 + 16] = f2bf(y[1][e]);
      }
  };
  fetch(0);
  __syncthreads();
  __syncthreads();
  __syncthreads();
  __syncthreads();
  for (int n = 0; n < nch; ++n) {
    const char* kd = sm + Z::kd + n % 3 * Z::SK;
    const float* end = reinterpret_cast<const float*>(kd + D * Z::DP) + 4 * lg;   // G_16, beta
    if (n > 0) norm(n - 1);   // (before the loop's first products: the two run side by side)
    f32x4_t ks[2] = {}, qs[2] = {}, kl[2] = {};   // kl: the products of lower parts, so that ks is rounded once per 32 channels
    const char* xa = sm + n % 2 * Z::SX + li * Z::XP + 16 * lg;
#pragma unroll
    for (int t = 0; t < ND; t += 2) {
      bf16x8_t kf[3], qf[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        kf[i] = ldf(xa + i * CT * Z::XP + 32 * t);
        qf[i] = ldf(xa + (3 + i) * CT * Z::XP + 32 * t);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        uint32_t p[4][3];
#pragma unroll
        for (int e = 0; e < 4; ++e) split3(S[t + e / 2][c][2 * (e & 1)], S[t + e / 2][c][2 * (e & 1) + 1], p[e]);
        bf16x8_t sf[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) sf[i] = frag(p[0][i], p[1][i], p[2][i], p[3][i]);
#pragma unroll
        for (int i = 0; i < 3; ++i)   // all but the products below 2^-24 of the largest
#pragma unroll
          for (int j = 0; i + j < 3; ++j) {
            (i + j > 0 ? kl : ks)[c] = mm(kf[i], sf[j], (i + j > 0 ? kl : ks)[c]);
            qs[c] = mm(qf[i], sf[j], qs[c]);
          }
      }
    }
    if (n > 0) store(n - 1);
    __syncthreads();
    const f32x4_t beta = ld4(end + D);
    f32x4_t R[2], U[2] = {};
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        R[c][e] = n * CT + 4 * lg + e < L ? beta[e] * (vv[c][e] - (ks[c][e] + kl[c][e])) : 0.f;
        gd[c][e] = gt[c][e];
      }
    if (n + 1 < nch) fetch(n + 1);
    // a zero of T or P times an infinity or NaN of a later token would reach earlier rows: such values enter the products as zeros
    // and the rows from their token on become NaN
    int first[2] = {CT, CT};   // first such token of the lane's columns
    auto take_out = [&](f32x4_t (&x)[2]) {
      bool bad = false;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) bad = bad || !(fabsf(x[c][e]) < __builtin_inff());
      if (__ballot(bad) == 0) return;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int e = 3; e >= 0; --e)
          if (!(fabsf(x[c][e]) < __builtin_inff())) first[c] = min(first[c], 4 * lg + e), x[c][e] = 0.f;
        first[c] = min(first[c], __shfl_xor(first[c], 16, 64));
        first[c] = min(first[c], __shfl_xor(first[c], 32, 64));
      }
    };
    take_out(R);
    const float* T = reinterpret_cast<const float*>(sm + Z::tp + n % 2 * Z::STP);
    const f32x4_t tf = ld4(T + li * TP + 4 * lg);
    const char* pp = reinterpret_cast<const char*>(T + CT * TP) + li * Z::DP + 32 * lg;
    const bf16x8_t p0 = ldf(pp), p1 = ldf(pp + 16);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int c = 0; c < 2; ++c) U[c] = mm(tf[e], R[c][e], U[c]);
#pragma unroll
    for (int c = 0; c < 2; ++c) U[c] += R[c];
    take_out(U);
    bf16x8_t uf[2][3];   // (h, h), (m, m), (l, h): against (h, m), (h, m), (h, l) the same products as above and m m
    auto parts = [&]() {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        uint32_t x[3], y[3];
        split3(U[c][0], U[c][1], x);
        split3(U[c][2], U[c][3], y);
        uf[c][0] = frag(x[0], y[0], x[0], y[0]);
        uf[c][1] = frag(x[1], y[1], x[1], y[1]);
        uf[c][2] = frag(x[2], y[2], x[0], y[0]);
      }
    };
    parts();
#pragma unroll
    for (int c = 0; c < 2; ++c) o[c] = mm(p0, uf[c][0], mm(p0, uf[c][1], mm(p1, uf[c][2], qs[c])));
    if (__ballot(min(first[0], first[1]) < CT) != 0) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * lg + e >= first[c]) o[c][e] = U[c][e] = __builtin_nanf("");
      parts();
    }
    f32x4_t ss;
#pragma unroll
    for (int e = 0; e < 4; ++e) ss[e] = group_sum<16>(o[0][e] * o[0][e] + o[1][e] * o[1][e]);
    if (li == 0) *reinterpret_cast<f32x4_t*>(sm + Z::ssq + 4 * (n % 2 * NC * CT + wave * CT + 4 * lg)) = ss;
    const char* ka = kd + li * Z::DP + 32 * lg;
#pragma unroll
    for (int t = 0; t < ND; ++t) {
      const bf16x8_t k0 = ldf(ka + 16 * t * Z::DP), k1 = ldf(ka + 16 * t * Z::DP + 16);
      const f32x4_t G = ld4(end + 16 * t);
      f32x4_t x[2] = {};
#pragma unroll
      for (int i = 2; i >= 0; --i)
#pragma unroll
        for (int c = 0; c < 2; ++c) x[c] = mm(i < 2 ? k0 : k1, uf[c][i], x[c]);
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[t][c][e] = fmaf(S[t][c][e], G[e], x[c][e]);   // one rounding of the state per chunk
    }
    __syncthreads();
  }
  norm(nch - 1);
  store(nch - 1);
  asm volatile("" : "+v"(so));   // the loads' offsets are formed again, not kept through the loop
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) st[so + (16 * t + e) * V + 16 * c] = S[t][c][e];
}

template <int D, int NC> hipError_t launch_one(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s) {
  constexpr size_t smem = Lds<D, NC>::total;
  auto* fn = a.z != nullptr ? chunk_delta_kernel<D, NC, true> : chunk_delta_kernel<D, NC, false>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(a.sh.heads, r.num_seqs), dim3(64 * NC + 2 * D), smem, s, a, r);
  return hipGetLastError();
}
template <int D> hipError_t launch_d(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s) {
  switch (a.sh.vdim / 32) {
    case 2: return launch_one<D, 2>(a, r, s);
    case 4: return launch_one<D, 4>(a, r, s);
    case 8: return launch_one<D, 8>(a, r, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

void chunk_delta_cut(GatedDeltaArgs& a, int rows, int num_seqs) {
  const int d = a.sh.dim, v = a.sh.vdim, none = rows + 1;
  // offsets within a chunk are 32-bit
  const bool near = a.gstride < (1 << 26) && a.ostride < (1 << 26) && (a.z == nullptr || a.zstride < (1 << 26));
  a.cut = none;
  if (a.f32 || !near || (d != 64 && d != 128) || (v != 64 && v != 128 && v != 256)) return;
  const int64_t wgs = (int64_t)a.sh.heads * num_seqs, cus = num_cus();
  const bool many = v < 256 && wgs > 2 * cus;
  const int64_t from = v == 64 ? 64 : CT, all = !many ? from : v == 128 ? 21 : wgs > 4 * cus ? 160 : 96;
  if (rows >= all * num_seqs || (v != 64 && rows >= CT * num_seqs && rows < (CT + 1) * num_seqs)) {
    a.cut = 0;
  } else if (rows >= from * num_seqs) {
    a.cut = v == 64 ? (int)all : 28;
    a.longest = (int)(rows * (int64_t)a.sh.heads / (2 * cus)) + 30;
  }
}

hipError_t launch_chunk_delta(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s) {
  switch (a.sh.dim) {
    case 64: return launch_d<64>(a, r, s);
    case 128: return launch_d<128>(a, r, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace die
