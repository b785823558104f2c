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
// What does not depend on the state, M, P and T, is formed for all chunks at once by a kernel of its own, chunk_pairs_kernel, a workgroup per
// (chunk, head): decays per channel by a lane that runs w = k_j g_(j+1) .. g_i down a column, one decay for all channels as products on
// the matrix cores, weighed afterwards; T by substitution.
//
// The serial part, chunk_delta_kernel, is a workgroup per (sequence, head). One wave per 32 value columns consumes: it owns its columns of
// S in accumulators, whose layout (row 4 (lane / 16) + r in register r) is an operand's with the contraction in another order, so that
// S, v and u are operands as they stand. Up to four helping waves scale k and q by their decays (into LDS, a chunk ahead) and norm, gate and
// store the results of the chunk before. One barrier per chunk. Steps of about a chunk per sequence form M, P and T inside (launch_one).
//
// fp32 operands enter as three bf16 parts of 8 bits each (exact), of whose nine products the six largest are formed (the rest are
// below 2^-25 of the whole): the fp32 matrix instructions run at the vector units' rate and in their place. Where a sum enters the state,
// lower parts are summed apart and added once, and of T the part below its diagonal is multiplied; the state is rounded once per chunk
// instead of twice per token, scaled rows not at all before they are cut. Its error against 64 bits (2-norm; 1 - 16 sequences of
// 16 - 1400 rows) is 0.2 - 1.0e-7, 0.90 - 0.93 of that of the token-by-token kernel, decays per head and per channel.
//
// An infinite key or value makes the rows from its token on and the state NaN (a part of an infinity is NaN), where token by token some
// of them may stay infinite; earlier rows and other sequences are as they are.
//
// Bound by instruction issue of the two waves per SIMD: per chunk some 530 vector and 158 matrix instructions of a consuming wave beside 650 of a
// helping one, each 4.5 - 5 cycles of its SIMD whatever it does (conversions and exponentials 8; 7800 cycles a chunk), and under a full load by
// power (1.8 GHz). Loads stand where no condition is around them and their values are converted where they are used: behind a condition, or
// converted early, they were waited for at once, 2000 cycles a chunk. Products and the cutting of the next operands alternate, as a wave issues
// in order. With M, P and T inside, every chunk, and norm and gate by the consuming waves, a chunk took 5.0 us instead of 3.3: 16 heads of 128 x 128, decays
// per channel, one sequence of 1024 rows 316 -> 220 us, 16 of 500 - 1000 336 -> 316, 3 x 180 rows (decays per head) 62 -> 49; 64 x 64, one of 1024 194 -> 130.
#include "chunk_delta.h"
#include "chunk_parts.h"
#include "lane_reduce.h"

namespace die {

namespace {

// What a chunk's serial part takes ready made, per (chunk, head): T - 1, and P in parts, as 16-byte pieces in the order of the lanes
constexpr int WORK = 3 * 64 * 4;   // floats
// the first chunk of sequence s, whose rows start at q0: room for every sequence's last, partly filled one
__device__ __forceinline__ int first_chunk(int q0, int s) { return q0 / CT + s; }

// Rows k, q of two neighbouring channels and 4 neighbouring tokens on every lane, and their decays: a wave covers 32 channels of a
// chunk (lane % 16: the pair of channels, lane / 16: the quarter of the tokens).
template <int D, bool CD> struct Rows {
  const float *kb, *qb, *gb, *bb;   // the portion's rows: the head's k, q, decay, beta
  const bf16_t* zb;
  int C, bw, L, t0;
  uint32_t d2;
  int64_t zstride;
  float expA, bias0, bias1;
  float2_at4 k[4], q[4];
  uint32_t g[4];   // as loaded (two bf16 values of z, or the head's decay): converted at the load they would be waited for there
  __device__ __forceinline__ Rows(const GatedDeltaArgs& a, int q0, int rows, int h, int pw, int lane) {
    const DeltaShape& sh = a.sh;
    const int H = sh.heads, GH = sh.kv_heads;
    C = sh.channels(), bw = CD ? H : 2 * H, L = rows, t0 = 4 * (lane >> 4), d2 = 32 * pw + 2 * (lane & 15);
    qb = a.qkv32 + (int64_t)q0 * C + h / (H / GH) * D;
    kb = qb + GH * D;
    bb = a.bg + (int64_t)q0 * bw + h;
    gb = bb + H;
    zb = reinterpret_cast<const bf16_t*>(a.z) + (int64_t)q0 * a.zstride + h * D;
    zstride = a.zstride;
    if constexpr (CD) expA = expf(a.A_log[h]), bias0 = a.z_bias[h * D + d2], bias1 = a.z_bias[h * D + d2 + 1];
  }
  __device__ __forceinline__ void fetch(int n) {   // raw rows of chunk n; beyond the portion its last one
    const uint32_t last = L - n * CT - 1;
    const int64_t row0 = n * CT;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint32_t row = min((uint32_t)(t0 + t), last), at = 4 * (row * C + d2);
      k[t] = *at_bytes<float2_at4>(kb + row0 * C, at);
      q[t] = *at_bytes<float2_at4>(qb + row0 * C, at);
      if constexpr (CD)
        g[t] = *at_bytes<uint32_at2>(zb + row0 * zstride, 2 * (row * (uint32_t)zstride + d2));   // (z at any 2 bytes)
      else
        g[t] = *at_bytes<uint32_t>(gb + row0 * bw, 4 * (row * bw));
    }
  }
  // k and q of token lane % 16, channels 32 pw + 8 (lane / 16) .. + 7 as operands; its decay
  __device__ __forceinline__ float rows_of_pairs(int n, int pw, int lane, bf16x8_t (&kf)[3], bf16x8_t (&qf)[3]) const {
    const uint32_t row = min(lane & 15, L - n * CT - 1), at = 4 * (row * C + 32 * pw + 8 * (lane >> 4));
    const int64_t row0 = n * CT;
    float2_at4 x[2][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[0][e] = *at_bytes<float2_at4>(kb + row0 * C, at + 8 * e);
      x[1][e] = *at_bytes<float2_at4>(qb + row0 * C, at + 8 * e);
    }
    const float g = *at_bytes<float>(gb + row0 * bw, 4 * (row * bw));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float v[8];
      uint32_t p[3][4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[2 * e] = x[i][e][0], v[2 * e + 1] = x[i][e][1];
      split3<4>(v, p);
#pragma unroll
      for (int j = 0; j < 3; ++j) (i ? qf : kf)[j] = frag(p[j][0], p[j][1], p[j][2], p[j][3]);
    }
    return g;
  }
  __device__ __forceinline__ float beta(int n, int lane) const {   // of token lane % 16, as loaded
    const int last = L - n * CT - 1;
    return bb[(int64_t)(n * CT + min(lane & 15, last)) * bw];
  }
  __device__ __forceinline__ float decay(float x, float bias) const {   // softplus_of<true>, its logarithm ahead of the choice
    const float z = x + bias, e = exp_of<true>(-fabsf(z));
    float l = 0.6931471805599453f * __builtin_amdgcn_logf(1.0f + e);
    asm volatile("" : "+v"(l));
    l = e < 9.765625e-4f ? e - 0.5f * e * e : l;
    return exp_of<true>(-expA * (fmaxf(z, 0.f) + l));
  }
  // the fetched values -> rows and decays of chunk n (tokens beyond the portion: k = q = 0, g = 1)
  __device__ __forceinline__ void finish(int n, float2 (&ko)[4], float2 (&qo)[4], float2 (&go)[4]) const {
    const int last = L - n * CT - 1;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool in = t0 + t <= last;
      uint32_t w = g[t];
      asm volatile("" : "+v"(w));
      float gx = __uint_as_float(w), gy = gx;
      if constexpr (CD) gx = decay(__uint_as_float(w << 16), bias0), gy = decay(__uint_as_float(w & 0xffff0000u), bias1);
      asm volatile("" : "+v"(gx), "+v"(gy));   // (formed for every token, not behind the condition)
      ko[t] = make_float2(in ? k[t].x : 0.f, in ? k[t].y : 0.f);
      qo[t] = make_float2(in ? q[t].x : 0.f, in ? q[t].y : 0.f);
      go[t] = make_float2(in ? gx : 1.0f, in ? gy : 1.0f);
    }
  }
};

// ------------------------------------------------------------------------------------------------ M, P and T of every chunk
// LDS of a workgroup, in floats
template <int D> struct PairLds {
  static constexpr int KP = D + 4, NP = D / 32;
  static constexpr int gates = 2 * CT * KP, part = gates + CT * KP, low = part + 2 * NP * CT * TP, total = low + CT * TP;
};

// M, P and T of one chunk, by D / 32 waves: M and P over 32 channels each, the last one solves. One barrier, of the whole workgroup.
template <int D, bool CD>
__device__ __forceinline__ void form_pairs(Rows<D, CD>& rows, float* raw, float* to, int n, float beta, int pw, int lane) {
  using Z = PairLds<D>;
  constexpr int KP = Z::KP, NP = Z::NP;
  const int li = lane & 15, lg = lane >> 4;
  const int last = rows.L - n * CT - 1;
  beta = li <= last ? beta : 0.f;
  float* const part = raw + Z::part;
  float own = 0.f;
  if constexpr (!CD) {   // one decay for all channels: M and P without it on the matrix cores, each wave over its 32 channels
    f32x4_t m = {}, p = {};
    bf16x8_t kf[3], qf[3];
    own = rows.rows_of_pairs(n, pw, lane, kf, qf);
#pragma unroll
    for (int i = 2; i >= 0; --i)
#pragma unroll
      for (int j = 2 - i; j >= 0; --j) {
        m = mm(kf[i], kf[j], m);
        p = mm(qf[i], kf[j], p);
      }
    float* pm = part + pw * CT * TP + 4 * lg * TP + li;
#pragma unroll
    for (int r = 0; r < 4; ++r) pm[r * TP] = m[r], pm[NP * CT * TP + r * TP] = p[r];
  } else {
    rows.fetch(n);
    float2 k[4], q[4], g[4];
    rows.finish(n, k, q, g);
    float* to = raw + 4 * lg * KP + 32 * pw + 2 * li;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      *reinterpret_cast<float2*>(to + t * KP) = k[t];
      *reinterpret_cast<float2*>(to + (CT + t) * KP) = q[t];
      *reinterpret_cast<float2*>(to + (2 * CT + t) * KP) = g[t];
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (a wave reads the channels that it wrote)
  __builtin_amdgcn_wave_barrier();
  if constexpr (CD) {
    // over the wave's 32 channels, 4 per lane: lane j < 8 (of 8 for the channels) runs down column j, rows j .. 15, then down column
    // 15 - j: 17 steps for any j
    const int j = lane & 7, turn = CT - j;
    const bool b3 = lane & 8, b4 = lane & 16;
    const float* ra = raw + 32 * pw + 4 * (lane >> 3) + j * KP;
    const float* rb = ra - j * KP - KP;
    f32x4_t w = {}, at[2][3];
    auto row = [&](int t) {   // k, q, decays of step t's row
      const float* r = (t < turn ? ra : rb) + t * KP;
      at[t & 1][0] = ld4(r), at[t & 1][1] = ld4(r + CT * KP), at[t & 1][2] = ld4(r + 2 * CT * KP);
    };
    float* pm = part + (lane >> 5) * (NP * CT * TP) + pw * CT * TP;   // low lanes keep M, high ones P
    auto put = [&](int t, float x) { pm[t < turn ? (j + t) * TP + j : (t - 1) * TP + CT - 1 - j] = x; };
    float one = 0.f, two = 0.f;
    row(0);
#pragma unroll
    for (int t = 0; t <= CT; ++t) {
      if (t < CT) row(t + 1);
      __builtin_amdgcn_sched_barrier(0);   // (a step's reads stay ahead of the step before it)
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
  }
  __syncthreads();
  if (pw != NP - 1) return;
  f32x4_t m = {}, p = {};
  const float* pm = part + li * TP + 4 * lg;
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    m += ld4(pm + q * CT * TP);
    p += ld4(pm + (NP + q) * CT * TP);
  }
  if constexpr (!CD) {   // decays from a column's token to the row's, multiplied up from theirs
    float w = 1.0f;
    f32x4_t W = {1.0f, 1.0f, 1.0f, 1.0f};
#pragma unroll
    for (int j = CT - 2; j >= 0; --j) {
      w = j < li ? w * __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(own), j + 1)) : w;
      W[j & 3] = j >> 2 == lg ? w : W[j & 3];
    }
    m *= W;
    p *= W;
  }
  float* lo = raw + Z::low;
#pragma unroll
  for (int e = 0; e < 4; ++e) {   // row li, columns 4 lg ..
    const int j = 4 * lg + e;
    m[e] = j < li ? beta * m[e] : 0.f;
    p[e] = j <= li ? p[e] : 0.f;
  }
  *reinterpret_cast<f32x4_t*>(lo + li * TP + 4 * lg) = m;
  {
    uint32_t x[3], y[3];
    split3(p[0], p[1], x);
    split3(p[2], p[3], y);
    *reinterpret_cast<uint4*>(to + 256 + 4 * lane) = make_uint4(x[0], y[0], x[1], y[1]);
    *reinterpret_cast<uint4*>(to + 512 + 4 * lane) = make_uint4(x[0], y[0], x[2], y[2]);
  }
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
  // T - 1, to where a row's lanes read it: column li of row 4 lg + r is value li % 4 of lane 4 lg + r + 16 (li / 4)
#pragma unroll
  for (int r = 0; r < 4; ++r) to[4 * (4 * lg + r + 16 * (li >> 2)) + (li & 3)] = 4 * lg + r > li ? t[r] : 0.f;
}

// One workgroup per (chunk, head).
template <int D, bool CD>
__global__ void __launch_bounds__(2 * D) chunk_pairs_kernel(GatedDeltaArgs a, RaggedRows r, float* work) {
  __shared__ __attribute__((aligned(16))) float raw[PairLds<D>::total];   // k | q | decays of the chunk, partial M | P of every wave, B tril(M)
  const int h = blockIdx.x % a.sh.heads, at = blockIdx.x / a.sh.heads;
  const int pw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  int s = -1;   // the sequence whose chunk this is: the last one that starts here or before
  for (int i = 0; i < r.num_seqs; i += 64) {
    const bool before = i + lane < r.num_seqs && first_chunk(r.cu_q[min(i + lane, r.num_seqs)], i + lane) <= at;
    s += __builtin_popcountll(__ballot(before));
  }
  s = __builtin_amdgcn_readfirstlane(s);
  if (s < 0) return;
  const int q0 = __builtin_amdgcn_readfirstlane(r.cu_q[s]), L = __builtin_amdgcn_readfirstlane(r.cu_q[s + 1]) - q0;
  const int n = at - first_chunk(q0, s);
  if (n * CT >= L || L < a.cut) return;
  if (a.cut > 0 && !divided(r.cu_q, r.num_seqs, r.total_rows, a.cut, a.longest)) return;
  Rows<D, CD> rows(a, q0, L, h, pw, lane);
  form_pairs(rows, raw, work + ((int64_t)at * a.sh.heads + h) * WORK, n, rows.beta(n, lane), pw, lane);
}

// ---------------------------------------------------------------------------------------------------------- the serial part
// LDS of a workgroup, in bytes
template <int D, int V> struct Lds {
  static constexpr int XP = 2 * D + 16, DP = 8 * CT + 16;    // pitch of a part's row of G k, G q; of a channel of k G_16 / G
  static constexpr int OP = V + 4;                           // pitch of a token's results (floats)
  static constexpr int SX = 6 * CT * XP;                     // (k, q) x 3 parts of G x; two chunks
  static constexpr int SK = D * DP + 4 * D + 4 * CT;         // k G_16 / G, G_16, beta; two chunks
  static constexpr int kd = 2 * SX;
  static constexpr int res = kd + 2 * SK;                    // results, two chunks
  static constexpr int total = res + 8 * CT * OP;
  static_assert(total <= 160 * 1024, "LDS of a compute unit");
};

// waves that scale rows (32 channels each) and finish results (a share of the chunk's tokens)
template <int D, int V> constexpr int helpers() { return D / 32 > 4 || V <= D ? D / 32 : V / 32 < 4 ? V / 32 : 4; }

template <int D, int V, bool CD>
__global__ void __launch_bounds__((2 * V + 64 * helpers<D, V>()), 1) chunk_delta_kernel(GatedDeltaArgs a, RaggedRows r, float* work, bool pairs) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  constexpr int NB = 2, NC = V / (16 * NB), ND = D / 16, NH = helpers<D, V>();   // consuming waves of 16 NB columns each
  using Z = Lds<D, V>;
  const DeltaShape& sh = a.sh;
  const int H = sh.heads, GH = sh.kv_heads, C = sh.channels();
  const int h = blockIdx.x, s = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int q0 = __builtin_amdgcn_readfirstlane(r.cu_q ? r.cu_q[s] : s);
  const int L = __builtin_amdgcn_readfirstlane(r.cu_q ? r.cu_q[s + 1] - q0 : 1);
  if (L <= 0 || L < a.cut) return;
  if (a.cut > 0 && !divided(r.cu_q, r.num_seqs, r.total_rows, a.cut, a.longest)) return;
  const int nch = (L + CT - 1) / CT;
  float* const made = work + ((int64_t)first_chunk(q0, s) * H + h) * WORK;   // of the first chunk; the next ones' H * WORK further
  auto pairs_of = [&](int n) __attribute__((always_inline)) {   // with `pairs`: chunk n's, in LDS of their own
    if (n >= nch || wave < NC || wave >= NC + D / 32) {
      __syncthreads();
    } else {
      Rows<D, CD> rows(a, q0, L, h, wave - NC, lane);
      form_pairs(rows, reinterpret_cast<float*>(sm + Z::total), made + (int64_t)n * H * WORK, n, rows.beta(n, lane), wave - NC, lane);
    }
  };
  auto first_pairs = [&]() __attribute__((always_inline)) {   // (behind the first loads)
    if (!pairs) return;
    pairs_of(0);
    if (nch == 1) return;
    __syncthreads();
    pairs_of(1);
  };

  if (wave >= NC) {
    // ------------------------------------------------------------------------------------------------ producers
    const int pw = wave - NC, pt = 64 * pw + lane;
    // results: 64 NH / 16 lanes a token, columns fc + FL i
    constexpr int FL = 4 * NH, FN = V / FL;
    const int ft = pt / FL, fc = pt % FL;
    float nw[FN];
    uint32_t gt[FN];   // (as loaded)
#pragma unroll
    for (int i = 0; i < FN; ++i) nw[i] = a.norm_w[fc + FL * i];
    const bf16_t* gp = reinterpret_cast<const bf16_t*>(a.gate) + (int64_t)q0 * a.gstride + h * V + fc;
    bf16_t* const op = reinterpret_cast<bf16_t*>(a.out) + (int64_t)q0 * a.ostride + h * V + fc;
    auto fetch_gates = [&](int n) {
      const bf16_t* g = gp + (int64_t)(n * CT) * a.gstride + min(ft, L - n * CT - 1) * (int)a.gstride;
#pragma unroll
      for (int i = 0; i < FN; ++i) gt[i] = g[FL * i];
    };
    auto finish = [&](int n) {   // norm and gate of chunk n
      const float* res = reinterpret_cast<const float*>(sm + Z::res) + (n % 2 * CT + ft) * Z::OP + fc;
      float o[FN], ss = 0.f;
#pragma unroll
      for (int i = 0; i < FN; ++i) o[i] = res[FL * i], ss = fmaf(o[i], o[i], ss);
      if constexpr (FL < 16) ss = group_sum<8>(ss);
      if constexpr (FL >= 16) ss = group_sum<16>(ss);
      const float rs = a.mult / sqrtf(ss * (1.0f / V) + a.eps);
      float y[FN];
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        asm volatile("" : "+v"(gt[i]));
        const float g = __uint_as_float(gt[i] << 16);
        y[i] = o[i] * rs * nw[i] * gated(a.gate_sigmoid ? 1.0f : g, g);
      }
      bf16_t* to = op + (int64_t)(n * CT) * a.ostride + ft * (int)a.ostride;
      if (n * CT + ft < L) {
#pragma unroll
        for (int i = 0; i < FN; ++i) to[FL * i] = f2bf(y[i]);
      }
      fetch_gates(min(n + 1, nch - 1));   // (without a condition, behind which loads would be waited for)
    };
    static_assert(FL == 8 || FL == 16, "lanes of a token");
    if (D / 32 < NH && pw >= D / 32) {   // (rows are all taken)
      fetch_gates(0);
      first_pairs();
      __syncthreads();
      for (int n = 0; n < nch; ++n) {
        if (pairs) pairs_of(n + 2);
        if (n > 0) finish(n - 1);
        __syncthreads();
      }
      finish(nch - 1);
      return;
    }
    const int d2 = 32 * pw + 2 * li;
    Rows<D, CD> rows(a, q0, L, h, pw, lane);
    float bt = 0.f;
    auto fetch = [&](int n) {
      rows.fetch(n);
      bt = rows.beta(n, lane);
    };
    auto scale = [&](int n) {   // scaled rows of chunk n; then the loads of the next one
      float2 k[4], q[4], g[4];
      rows.finish(n, k, q, g);
      const float b = n * CT + pt < L ? bt : 0.f;
      fetch(min(n + 1, nch - 1));
      float2 all = make_float2(g[0].x * g[1].x * (g[2].x * g[3].x), g[0].y * g[1].y * (g[2].y * g[3].y));
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
        split3(k[t].x, G.x, k[t].y, G.y, p);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint32_t*>(to + (i * CT + t) * Z::XP) = p[i];
        split3(q[t].x, G.x, q[t].y, G.y, p);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint32_t*>(to + ((3 + i) * CT + t) * Z::XP) = p[i];
      }
      char* kd = sm + Z::kd + n % 2 * Z::SK;
      float* end = reinterpret_cast<float*>(kd + D * Z::DP);   // G_16, beta
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
      if (lg == 3) *reinterpret_cast<float2*>(end + d2) = G;
      if (pt < CT) end[D + pt] = b;
    };
    fetch(0);
    fetch_gates(0);
    first_pairs();
    scale(0);
    __syncthreads();
    for (int n = 0; n < nch; ++n) {
      if (pairs) pairs_of(n + 2);   // (a chunk before its consumers load them)
      if (n + 1 < nch) scale(n + 1);
      if (n > 0) finish(n - 1);
      __syncthreads();
    }
    finish(nch - 1);
    return;
  }

  // -------------------------------------------------------------------------------------------------- consumers
  const int v0 = 16 * NB * wave + li;
  const bool fresh = r.positions[q0] <= 0;
  float* st = a.state + ((int64_t)__builtin_amdgcn_readfirstlane(r.state_slots[s]) * H + h) * (D * V);
  uint32_t so = 4 * lg * V + v0;
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
  const uint4* wp = reinterpret_cast<const uint4*>(made) + lane;
  uint4 tp[3];   // T - 1, P of the current chunk
  float vv[NB][4];   // values of the current chunk
  auto fetch = [&](int n) {
    const int64_t row0 = q0 + n * CT;
    const float* vr = a.qkv32 + row0 * C + 2 * GH * D + h * V;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = min(4 * lg + e, L - n * CT - 1);
#pragma unroll
      for (int c = 0; c < NB; ++c) vv[c][e] = vr[row * C + v0 + 16 * c];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) tp[i] = wp[n * H * (WORK / 4) + 64 * i];
  };
  first_pairs();
  if (!pairs) fetch(0);
  __syncthreads();
  if (pairs) fetch(0);
  for (int n = 0; n < nch; ++n) {
    const char* kd = sm + Z::kd + n % 2 * Z::SK;
    const float* end = reinterpret_cast<const float*>(kd + D * Z::DP) + 4 * lg;   // G_16, beta
    f32x4_t ks[NB] = {}, qs[NB] = {}, kl[NB] = {};   // kl: the products of lower parts, so that ks is rounded once per 32 channels
    const char* xa = sm + n % 2 * Z::SX + li * Z::XP + 16 * lg;
    // 32 channels of 16 columns at a time; the next ones' parts are cut between the products of the current ones, as a wave's instructions
    // issue in order and a product keeps the next one waiting for 16 cycles
    bf16x8_t kf[2][3], qf[2][3], sf[2][3];
    auto rows_of = [&](int t, bf16x8_t (&k)[3], bf16x8_t (&q)[3]) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        k[i] = ldf(xa + i * CT * Z::XP + 64 * t);
        q[i] = ldf(xa + (3 + i) * CT * Z::XP + 64 * t);
      }
    };
    auto cut = [&](int t, int c, bf16x8_t (&f)[3]) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = S[2 * t + e / 4][c][e % 4];
      uint32_t p[3][4];
      split3<4>(x, p);
#pragma unroll
      for (int i = 0; i < 3; ++i) f[i] = frag(p[i][0], p[i][1], p[i][2], p[i][3]);
    };
    rows_of(0, kf[0], qf[0]);
    cut(0, 0, sf[0]);
#pragma unroll
    for (int b = 0; b < ND / 2 * NB; ++b) {
      const int t = b / NB, c = b % NB;
      __builtin_amdgcn_sched_barrier(0);
      if (c == 0 && t + 1 < ND / 2) rows_of(t + 1, kf[(t + 1) & 1], qf[(t + 1) & 1]);
      if (b + 1 < ND / 2 * NB) cut((b + 1) / NB, (b + 1) % NB, sf[(b + 1) & 1]);
#pragma unroll
      for (int i = 0; i < 3; ++i)   // all but the products below 2^-24 of the largest
#pragma unroll
        for (int j = 0; i + j < 3; ++j) {
          (i + j > 0 ? kl : ks)[c] = mm(kf[t & 1][i], sf[b & 1][j], (i + j > 0 ? kl : ks)[c]);
          qs[c] = mm(qf[t & 1][i], sf[b & 1][j], qs[c]);
        }
#pragma unroll
      for (int m = 0; m < 12; ++m) {   // a product, then what issues while it runs
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (m < 3) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (pairs) __syncthreads();   // (the one inside pairs_of)
    const f32x4_t beta = ld4(end + D);
    f32x4_t R[NB], U[NB] = {};
    const f32x4_t tf = __builtin_bit_cast(f32x4_t, tp[0]);
    const bf16x8_t p0 = __builtin_bit_cast(bf16x8_t, tp[1]), p1 = __builtin_bit_cast(bf16x8_t, tp[2]);
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) R[c][e] = n * CT + 4 * lg + e < L ? beta[e] * (vv[c][e] - (ks[c][e] + kl[c][e])) : 0.f;
    fetch(min(n + 1, nch - 1));
    // a zero of T or P times an infinity or NaN of a later token would reach earlier rows: such values enter the products as zeros
    // and the rows from their token on become NaN
    int first[NB];   // first such token of the lane's columns
#pragma unroll
    for (int c = 0; c < NB; ++c) first[c] = CT;
    auto take_out = [&](f32x4_t (&x)[NB]) {
      bool bad = false;
#pragma unroll
      for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) bad = bad || !(fabsf(x[c][e]) < __builtin_inff());
      if (__ballot(bad) == 0) return;
#pragma unroll
      for (int c = 0; c < NB; ++c) {
#pragma unroll
        for (int e = 3; e >= 0; --e)
          if (!(fabsf(x[c][e]) < __builtin_inff())) first[c] = min(first[c], 4 * lg + e), x[c][e] = 0.f;
        first[c] = min(first[c], __shfl_xor(first[c], 16, 64));
        first[c] = min(first[c], __shfl_xor(first[c], 32, 64));
      }
    };
    take_out(R);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int c = 0; c < NB; ++c) U[c] = mm(tf[e], R[c][e], U[c]);
#pragma unroll
    for (int c = 0; c < NB; ++c) U[c] += R[c];
    take_out(U);
    bf16x8_t uf[NB][3];   // (h, h), (m, m), (l, h): against (h, m), (h, m), (h, l) the same products as above and m m
    auto parts = [&]() {
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        uint32_t x[3], y[3];
        split3(U[c][0], U[c][1], x);
        split3(U[c][2], U[c][3], y);
        uf[c][0] = frag(x[0], y[0], x[0], y[0]);
        uf[c][1] = frag(x[1], y[1], x[1], y[1]);
        uf[c][2] = frag(x[2], y[2], x[0], y[0]);
      }
    };
    parts();
    f32x4_t o[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) o[c] = mm(p0, uf[c][0], mm(p0, uf[c][1], mm(p1, uf[c][2], qs[c])));
    bool odd = false;
#pragma unroll
    for (int c = 0; c < NB; ++c) odd = odd || first[c] < CT;
    if (__ballot(odd) != 0) {
#pragma unroll
      for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * lg + e >= first[c]) o[c][e] = U[c][e] = __builtin_nanf("");
      parts();
    }
    float* res = reinterpret_cast<float*>(sm + Z::res) + (n % 2 * CT + 4 * lg) * Z::OP + v0;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int c = 0; c < NB; ++c) res[e * Z::OP + 16 * c] = o[c][e];
    const char* ka = kd + li * Z::DP + 32 * lg;
    bf16x8_t k0[2], k1[2];
    f32x4_t G[2], x[2][NB];
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
    for (int t = 0; t < ND; ++t) {   // (16 channels' products beside the sums of the ones before)
      __builtin_amdgcn_sched_barrier(0);
      if (t > 0) add(t - 1);
#pragma unroll
      for (int c = 0; c < NB; ++c) x[t & 1][c] = {};
#pragma unroll
      for (int i = 2; i >= 0; --i)
#pragma unroll
        for (int c = 0; c < NB; ++c) x[t & 1][c] = mm(i < 2 ? k0[t & 1] : k1[t & 1], uf[c][i], x[t & 1][c]);
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
      for (int e = 0; e < 4; ++e) st[so + (16 * t + e) * V + 16 * c] = S[t][c][e];
}

template <int D, int V, bool CD> hipError_t launch_one(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s) {
  constexpr size_t smem = Lds<D, V>::total;
  const auto fn = chunk_delta_kernel<D, V, CD>;
  // Where portions have a chunk on average, pairs are formed inside, two chunks ahead: the launch of its own, which longer portions gain from,
  // takes longer than they do (16 tokens of 1 / 16 / 64 sequences, 16 heads of 128 x 128: 12.5 / 19.4 / 59 us with it, 10.6 / 15.9 / 54 without; only
  // many of 64 x 128 are faster with it, 128 of 16 tokens 68 / 73), and with one workgroup per compute unit two chunks do not pay for it either (16 x
  // 22: 22.2 / 21.2). An average hides long portions, whose chain is up to twice as long with pairs inside (1000 tokens beside 63 rows of a token, 64 x
  // 128, 191 / 314; before there were two forms 267): where the longest is known to have more than two chunks, the launch of its own is taken.
  constexpr size_t own = 4 * PairLds<D>::total, most = smem + own <= 160 * 1024 ? smem + own : smem;
  const int64_t wgs = (int64_t)a.sh.heads * r.num_seqs, cus = num_cus();
  const bool few = r.total_rows <= (CT + 1) * r.num_seqs ? D != 64 || V != 128 || wgs <= 2 * cus
                                                         : wgs <= cus && 2 * wgs > cus && r.total_rows <= 2 * CT * r.num_seqs;
  const bool inside = most > smem && few && r.max_rows <= 2 * CT;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
  if (e != hipSuccess) return e;
  if (!inside)
    hipLaunchKernelGGL((chunk_pairs_kernel<D, CD>), dim3(a.sh.heads * (r.total_rows / CT + r.num_seqs)), dim3(2 * D), 0, s, a, r, a.work);
  hipLaunchKernelGGL(fn, dim3(a.sh.heads, r.num_seqs), dim3(2 * V + 64 * helpers<D, V>()), inside ? most : smem, s, a, r, a.work, inside);
  return hipGetLastError();
}
template <int D, bool CD> hipError_t launch_d(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s) {
  switch (a.sh.vdim) {
    case 64: return launch_one<D, 64, CD>(a, r, s);
    case 128: return launch_one<D, 128, CD>(a, r, s);
    case 256: return launch_one<D, 256, CD>(a, r, s);
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
  // rows of a sequence on average: up to 1, 2, 4 workgroups per compute unit, more
  static constexpr int FROM[2][3][4] = {{{9, 9, 20, 24}, {9, CT, CT, CT}, {9, 9, 9, 9}}, {{9, 36, 56, 96}, {9, 14, CT, CT}, {9, 10, 10, 10}}};
  const int64_t from = FROM[d / 128][v / 128][wgs <= cus ? 0 : wgs <= 2 * cus ? 1 : wgs <= 4 * cus ? 2 : 3];
  const int64_t all = v == 128 && wgs > 2 * cus ? 21 : from;
  if (rows >= all * num_seqs || (rows >= from * num_seqs && rows < (CT + 1) * num_seqs)) {
    a.cut = 0;
  } else if (rows >= from * num_seqs) {
    a.cut = 28;
    a.longest = (int)(rows * (int64_t)a.sh.heads / (2 * cus)) + 30;
  }
}

int64_t chunk_delta_work(GatedDeltaArgs a, int rows, int num_seqs) {
  chunk_delta_cut(a, rows, num_seqs);
  return a.cut <= rows ? (int64_t)(rows / CT + num_seqs) * a.sh.heads * WORK : 0;
}

hipError_t launch_chunk_delta(const GatedDeltaArgs& a, RaggedRows r, hipStream_t s) {
  switch (a.sh.dim) {
    case 64: return a.z != nullptr ? launch_d<64, true>(a, r, s) : launch_d<64, false>(a, r, s);
    case 128: return a.z != nullptr ? launch_d<128, true>(a, r, s) : launch_d<128, false>(a, r, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace die
