// The matrix recurrence S <- a_t S + b_t k_t v_t^T, o_t = S^T q_t of prompt portions in chunks of 32 tokens on the matrix
// cores (gfx950), for bf16 activations; state, decays and results are fp32 and keep their 24 bits.
//
// With A_i = a_1 .. a_i over a chunk and W_ij = b_j a_(j+1) .. a_i (i >= j):
//     o_i = sum_(j <= i) W_ij (q_i . k_j) v_j + A_i S^T q_i        S <- A_32 S + sum_j (W_32j k_j) v_j^T
// so a chunk is four products. One wave owns 32 columns of S for the whole step (in its accumulators), the waves of a
// workgroup share one (sequence, head) and its staged q, k, v rows; the normaliser n <- a n + b k is one more column block
// whose values are ones.
//
// Precision. q, k, v are bf16 and enter the products exactly. What is fp32 (W q.k, S, W v) is cut into three bf16 parts by
// truncation, 8 + 8 + 8 bits, which is exact, and takes three products with fp32 accumulators. Products of decays are
// multiplied up directly (no logarithms, no quotients: any a, zero and negative ones too), at most a few more roundings than
// the token-by-token form. Distance from a 64-bit evaluation, 16 x 1024 tokens of the state-space shape: 1.2e-7 (results) and
// 0.8e-7 (state), the token-by-token kernel 1.4e-7 and 1.1e-7.
//
// An infinite value or state makes the rows from its token on and the state NaN (a part of an infinity is NaN), where token by token some
// of them may stay infinite; earlier rows and other sequences are as they are.
//
// What bounds it: instruction issue. A wave takes some 950 vector and 62 matrix instructions per chunk at dim 128 (cutting fragments, weighing
// scores), a SIMD issues one per 4.5 - 5 cycles in all, and two waves per SIMD at 230 registers hide the rest. Against the token-by-token
// kernels (bf16, us, before -> after): 16 x 1024 tokens, 64 heads of 128 x 64 sharing q and k 794 -> 189 (2.4 TB/s of its inputs, results and
// states), 16 heads of 128 x 128 with SiLU 1050 -> 154; 16 x 1000, 32 heads of 64 x 128 with normaliser 589 -> 220; one sequence of 1024, 64
// heads 410 -> 102. Of these, decays chosen where they are used and not where they are loaded (which waited for all loads of the chunk), rows
// of whole chunks stored without a condition each, and parts cut beside the products before them: 197 -> 189, 200 -> 154, 121 -> 102. (Remainders by
// the dot product with -1, one instruction for two: no gain, with the normaliser 3 % slower.)
#include "common.h"
#include "lane_reduce.h"
#include "chunk_rec.h"

namespace die {

namespace {

typedef __attribute__((address_space(3))) short4_t lds_short4;
typedef __attribute__((ext_vector_type(8))) short short8_t;

constexpr int CT = 32;   // tokens of a chunk

__device__ __forceinline__ bf16x8_t frag(uint4 w) { return __builtin_bit_cast(bf16x8_t, w); }
__device__ __forceinline__ f32x16_t mm(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// the value of lane PERM[i] of the own quad
template <int PERM> __device__ __forceinline__ float quad(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), PERM, 0xf, 0xf, true));
}
// the value of the lane 4 or 8 places before (0x114, 0x118) or behind (0x104, 0x108) in the own row of 16 lanes, 1 outside it
template <int CTRL> __device__ __forceinline__ float row_shift(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0x3f800000, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_of(float x, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
}
constexpr int perm4(int a, int b, int c, int d) { return a | b << 2 | c << 4 | d << 6; }

// two floats -> the upper halves of their bit patterns as a bf16 pair (truncation)
__device__ __forceinline__ uint32_t top2(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float below(float x) { return x - __uint_as_float(__float_as_uint(x) & 0xffff0000u); }
// 8 floats -> three bf16 fragments that sum to them exactly
__device__ __forceinline__ void split3(const float* x, bf16x8_t* f) {
  uint4 w[3];
  float r[8];
#pragma unroll
  for (int p = 0; p < 3; ++p) {
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = p == 0 ? x[e] : below(r[e]);
    w[p] = make_uint4(top2(r[0], r[1]), top2(r[2], r[3]), top2(r[4], r[5]), top2(r[6], r[7]));
    f[p] = frag(w[p]);
  }
}

// base (the same for all lanes) + a lane's offset in bytes: one scalar and one 32-bit address register, where 64-bit lane addresses
// of all accumulator rows would take two registers each
template <typename T> __device__ __forceinline__ T* at_bytes(T* base, uint32_t off) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off);
}
template <typename T> __device__ __forceinline__ const T* at_bytes(const T* base, uint32_t off) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}

// bf16 silu(z) of 8 packed values, rounded to bf16 (to the same bits as with expf, for every bf16 z)
__device__ __forceinline__ uint4 silu8(uint4 w) {
  float f[8];
  unpack8(w, f);
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = f[e] / (1.0f + __expf(-f[e]));
  return pack8(f);
}

// 8 elements of an MFMA operand whose contraction index runs over a row of LDS: 4 at c, 4 at c + 8
__device__ __forceinline__ bf16x8_t row_frag(const bf16_t* p) {
  const uint2 a = *reinterpret_cast<const uint2*>(p), b = *reinterpret_cast<const uint2*>(p + 8);
  return frag(make_uint4(a.x, a.y, b.x, b.y));
}
// the same where it runs over rows (pitch in bytes) of the own column: transposed reads of rows r .. r + 3 and r + 8 .. r + 11
__device__ __forceinline__ bf16x8_t col_frag(const char* p, int pitch) {
  const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p));
  const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p + 8 * pitch));
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// One workgroup per (sequence, NW / NV neighbouring heads that share q and k): NW waves, one per 32 value columns, and with a
// normaliser (of one head) one more. Every operand whose
// contraction runs over 16 indices takes them in the order 4 hi + 0 .. 3, 8 + 4 hi + 0 .. 3 (hi = lane / 32): the order in which
// a 32 x 32 accumulator holds its rows, so that score and state accumulators are operands as they stand.
template <int ND, int NW, int NV, bool SILU>
__global__ void __launch_bounds__(64 * (NW + 1), 2) chunk_linear_kernel(ChunkLinearArgs a, RaggedRows r) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int D = 32 * ND, V = 32 * NV, VW = 32 * NW, KP = D + 8, VP = VW + 8, CH = D / 8, CHV = VW / 8;
  constexpr int BUF = CT * (2 * KP + VP);                        // elements of a staged chunk: q | k | v rows
  constexpr int RQ = 64 * NW / (2 * CH), PQ = CT / RQ;           // q and k rows per pass of the workgroup, passes
  constexpr int RV = 64 * NW / CHV, PV = CT / RV;                // v rows
  static_assert(RQ * 2 * CH == 64 * NW && RQ * PQ == CT && RV * PV == CT, "whole passes");
  bf16_t* buf = reinterpret_cast<bf16_t*>(smem);
  const int s = blockIdx.y, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31, hi = lane >> 5;
  float* tab = reinterpret_cast<float*>(smem + BUF * sizeof(bf16_t)) + wave * 4 * CT;   // the wave's own
  const int q0 = __builtin_amdgcn_readfirstlane(r.cu_q ? r.cu_q[s] : s);
  const int L = __builtin_amdgcn_readfirstlane(r.cu_q ? r.cu_q[s + 1] - q0 : 1);
  if (L <= 0 || L < a.cut) return;
  if (a.cut > 0 && !divided(r.cu_q, r.num_seqs, r.total_rows, a.cut, a.longest)) return;
  const bool fresh = r.positions[q0] <= 0;
  const int H = a.heads, h0 = blockIdx.x * (NW / NV), g = h0 / (H / a.groups);
  const bool ones = wave == NW;                                  // the normaliser's column block (stages nothing)
  const int h = ones ? h0 : h0 + wave / NV, col = 32 * (wave % NV);   // the wave's head and first column of its state
  const int64_t slot = (int64_t)__builtin_amdgcn_readfirstlane(r.state_slots[s]) * H + h;
  float* st = ones ? a.n_state + slot * D : a.state + slot * (int64_t)(D * V) + col;
  uint32_t scol = 4 * (ones ? 4 * hi : li + 4 * hi * V);

  const int rq = tid / (2 * CH), xq = tid % (2 * CH), rv = tid / CHV, xv = tid % CHV;
  const uint32_t cq = (xq < CH ? a.qoff + xq * 8 : a.koff + (xq - CH) * 8) + g * D, cv = a.voff + h0 * V + xv * 8;
  const int lq = (xq < CH ? 0 : CT * KP) + rq * KP + xq % CH * 8, lv = 2 * CT * KP + rv * VP + xv * 8;
  const uint32_t oq = 2 * (rq * (uint32_t)a.xstride + cq), ov = 2 * (rv * (uint32_t)a.xstride + cv);
  uint4 pf[PQ + PV];
  float pa, pb;
  auto fetch = [&](int t0) {
    const int last = L - t0 - 1;   // rows beyond the portion repeat its last one: their weights are zero
    const bf16_t* x = a.x + (int64_t)(q0 + t0) * a.xstride;
    if (ones) {
    } else if (last >= CT - 1) {
#pragma unroll
      for (int u = 0; u < PQ; ++u)
        pf[u] = *reinterpret_cast<const uint4*>(at_bytes(x + (int64_t)(u * RQ) * a.xstride, oq));
#pragma unroll
      for (int u = 0; u < PV; ++u)
        pf[PQ + u] = *reinterpret_cast<const uint4*>(at_bytes(x + (int64_t)(u * RV) * a.xstride, ov));
    } else {
#pragma unroll
      for (int u = 0; u < PQ; ++u)
        pf[u] = *reinterpret_cast<const uint4*>(at_bytes(x, 2 * (min(u * RQ + rq, last) * (uint32_t)a.xstride + cq)));
#pragma unroll
      for (int u = 0; u < PV; ++u)
        pf[PQ + u] = *reinterpret_cast<const uint4*>(at_bytes(x, 2 * (min(u * RV + rv, last) * (uint32_t)a.xstride + cv)));
    }
    const float* p = a.ab != nullptr ? a.ab + ((int64_t)(q0 + t0 + min(li, last)) * H + h) * a.abw : a.decay + h;
    pa = p[0], pb = p[a.ab != nullptr ? 1 : 0];   // (as they are: a choice here would wait for all of these loads)
  };
  auto stash = [&] {
    if (ones) return;
#pragma unroll
    for (int u = 0; u < PQ; ++u) *reinterpret_cast<uint4*>(buf + lq + u * RQ * KP) = SILU ? silu8(pf[u]) : pf[u];
#pragma unroll
    for (int u = 0; u < PV; ++u) *reinterpret_cast<uint4*>(buf + lv + u * RV * VP) = SILU ? silu8(pf[PQ + u]) : pf[PQ + u];
  };

  f32x16_t S[ND];
  fetch(0);
#pragma unroll
  for (int m = 0; m < ND; ++m)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = 32 * m + 8 * (e >> 2) + (e & 3);
      const float x = *at_bytes(st, scol + 4 * (ones ? row : row * V));
      S[m][e] = fresh ? 0.f : x;   // (a new sequence reads its slot but not its content)
    }
  stash();
  __syncthreads();

  const int trow = 4 * hi + (lane & 15) / 4, tcol = 16 * (lane >> 4 & 1) + 4 * (lane & 3);   // of the transposed reads
  for (int t0 = 0; t0 < L; t0 += CT) {
    const bf16_t* b = buf;
    const bool in = li < L - t0;
    const float av = in ? pa : 1.0f, bv = in ? (a.ab != nullptr ? pb : 1.0f) : 0.0f;
    int G = li >> 2, rr = li & 3;              // the own token's quad and place in it
    asm volatile("" : "+v"(G), "+v"(rr));      // (else some 80 masks are kept over the loop, in spilled scalar registers)
    const bool more = t0 + CT < L;
    if (more) fetch(t0 + CT);

    // ---- products of decays over quads of tokens, then over halves of the chunk, then over both
    const float a1 = quad<perm4(0, 0, 1, 2)>(av), a2 = quad<perm4(0, 1, 0, 1)>(av);   // of the token 1 and 2 places before
    // (every cross-lane move stands outside the conditionals: all lanes have to take part in it)
    float I4 = rr >= 1 ? av * a1 : av;                       // a over the quad up to the own token
    const float I2 = quad<perm4(0, 1, 0, 1)>(I4);
    I4 = rr >= 2 ? I4 * I2 : I4;
    const float an = quad<perm4(1, 2, 3, 3)>(av);
    float E4 = rr <= 2 ? av * an : av;                       // a over the quad from the own token on
    const float E2 = quad<perm4(2, 3, 2, 3)>(E4);
    E4 = rr <= 1 ? E4 * E2 : E4;
    const float En = quad<perm4(1, 2, 3, 3)>(E4), t4 = rr <= 2 ? En : 1.0f;   // a over the quad behind the own token
    // over the 4 quads of the own half: inclusive from the left and from the right, then the other half's total
    const float m0 = quad<perm4(3, 3, 3, 3)>(I4), m1 = row_shift<0x114>(m0), m2 = row_shift<0x118>(m0);   // own quad, 1 and 2 before
    float fwd = m0 * m1, bwd = m0 * row_shift<0x104>(m0);
    fwd *= row_shift<0x118>(fwd);
    bwd *= row_shift<0x108>(bwd);
    const float all0 = lane_of(fwd, 15), all1 = lane_of(fwd, 31), all = all0 * all1;
    const float sb = row_shift<0x104>(bwd);                                               // behind the own quad, in its half
    const float inner = row_shift<0x114>(fwd) * I4, outer = sb * t4;                      // up to / behind the own token, in its half
    const float before = li < 16 ? inner : inner * all0, behind = li < 16 ? outer * all1 : outer;
    // a between quad 2 x + hi of a half and the own token: of the own half (zero unless that quad is before), of the first half
    float same[2], other[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int k = (G & 3) - 2 * x - hi;
      same[x] = k <= 0 ? 0.f : k == 1 ? I4 : I4 * (k == 2 ? m1 : m1 * m2);
      const float s0 = lane_of(sb, 8 * x), s1 = lane_of(sb, 8 * x + 4);
      other[x] = inner * (hi ? s1 : s0);
    }
    const float cg[4] = {li < 16 ? same[0] : other[0], li < 16 ? same[1] : other[1], li < 16 ? 0.f : same[0], li < 16 ? 0.f : same[1]};
    // W inside the own quad: column e of row rr
    const float w2 = av * a1, a123 = w2 * a2;
    const float b0 = quad<perm4(0, 0, 0, 0)>(bv), b1 = quad<perm4(1, 1, 1, 1)>(bv), b2 = quad<perm4(2, 2, 2, 2)>(bv), b3 = quad<perm4(3, 3, 3, 3)>(bv);
    const float dw[4] = {b0 * (rr == 0 ? 1.0f : rr == 1 ? av : rr == 2 ? w2 : a123), b1 * (rr == 0 ? 0.f : rr == 1 ? 1.0f : rr == 2 ? av : w2),
                         b2 * (rr < 2 ? 0.f : rr == 2 ? 1.0f : av), b3 * (rr < 3 ? 0.f : 1.0f)};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    if (hi == 0) {
      tab[li] = t4 * bv;                   // factor of column j towards later quads
      tab[CT + li] = behind * bv;          // W_32j
      tab[2 * CT + li] = before;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();

    // ---- scores (transposed: row j, column i) and the state's part of the result
    f32x16_t sc = {}, o = {};
    const bf16_t* qr = b + li * KP + 4 * hi;
    const bf16_t* kr = b + CT * KP + li * KP + 4 * hi;
    // 16 channels at a time, the next ones' parts cut beside the products of the current ones: a wave's instructions issue in order
    bf16x8_t qf[2], kf1[2], sf[2][3];
    auto rows_of = [&](int t) { qf[t & 1] = row_frag(qr + 16 * t), kf1[t & 1] = row_frag(kr + 16 * t); };
    auto cut = [&](int t) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = S[t / 2][8 * (t & 1) + e];
      split3(x, sf[t & 1]);
    };
    rows_of(0);
    cut(0);
#pragma unroll
    for (int t = 0; t < 2 * ND; ++t) {
      __builtin_amdgcn_sched_barrier(0);
      if (t + 1 < 2 * ND) rows_of(t + 1), cut(t + 1);
      sc = mm(kf1[t & 1], qf[t & 1], sc);
#pragma unroll
      for (int p = 2; p >= 0; --p) o = mm(qf[t & 1], sf[t & 1][p], o);
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- weights, then P V
    const char* vb = reinterpret_cast<const char*>(b + 2 * CT * KP + 32 * (ones ? 0 : wave)) + trow * (2 * VP) + 2 * tcol;
    bf16x8_t vf[2];
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2) {
      vf[k2] = col_frag(vb + 16 * k2 * (2 * VP), 2 * VP);
      if (ones) vf[k2] = frag(make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
    }
    // zero weights times an infinite or NaN value would reach the rows before it: such values enter the products as zeros, and
    // the rows from their token on become NaN
    bf16x8_t vz[2] = {vf[0], vf[1]};
    uint32_t top = 0;
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2) {
      const uint4 w = __builtin_bit_cast(uint4, vf[k2]);
      top |= ((w.x & 0x7f807f80u) + 0x00800080u) | ((w.y & 0x7f807f80u) + 0x00800080u) | ((w.z & 0x7f807f80u) + 0x00800080u) |
             ((w.w & 0x7f807f80u) + 0x00800080u);
    }
    const bool odd = __ballot((top & 0x80008000u) != 0) != 0;
    int jodd = CT;
    if (odd) {
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        short8_t w = __builtin_bit_cast(short8_t, vf[k2]);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if ((w[e] & 0x7f80) == 0x7f80) jodd = min(jodd, 16 * k2 + (e & 4) * 2 + 4 * hi + (e & 3)), w[e] = 0;
        vz[k2] = __builtin_bit_cast(bf16x8_t, w);
      }
      jodd = min(jodd, __shfl_xor(jodd, 32, 64));
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float4 A4 = *reinterpret_cast<const float4*>(tab + 2 * CT + 8 * u + 4 * hi);
      o[4 * u] *= A4.x, o[4 * u + 1] *= A4.y, o[4 * u + 2] *= A4.z, o[4 * u + 3] *= A4.w;
    }
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2) {
      float x[8];
      bf16x8_t f[3];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int gq = 2 * k2 + u;
        const float4 t = *reinterpret_cast<const float4*>(tab + 8 * gq + 4 * hi);
        const float tt[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool own = 2 * gq + hi == G;
          const float w = own ? dw[e] : tt[e] * cg[gq];
          // (a later token contributes nothing, whatever its score, a and b are)
          x[4 * u + e] = (own && e <= rr) || 2 * gq + hi < G ? w * sc[8 * k2 + 4 * u + e] : 0.f;
        }
      }
      split3(x, f);
#pragma unroll
      for (int p = 2; p >= 0; --p) o = mm(f[p], vz[k2], o);
    }
    if (odd) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (8 * (e >> 2) + 4 * hi + (e & 3) >= jodd) o[e] = __builtin_nanf("");
    }
    // ---- results: row i in the registers, the wave's columns in its lanes
    const int nb = L - t0;
    const uint32_t hv = ones ? H : H * V;
    uint32_t at = 4 * (4 * hi * hv + (ones ? 0 : li));
    asm volatile("" : "+v"(at));   // (else the rows' offsets are kept over the loop, in registers that spill)
    float* op = ones ? a.nq + (int64_t)(q0 + t0) * H + h : a.out + ((int64_t)(q0 + t0) * H + h) * V + col;
    const bool mine = !ones || li == 0;
    if (nb >= CT && !ones) {   // (a condition per row costs as much as the row)
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) *at_bytes(op + (int64_t)(8 * u + e) * hv, at) = o[4 * u + e] * a.qscale;
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (mine && 8 * u + 4 * hi + e < nb) *at_bytes(op, at + 4 * (8 * u + e) * hv) = o[4 * u + e] * a.qscale;
    }
    // ---- the state: its scaling and the values' parts beside the products
    const char* kb = reinterpret_cast<const char*>(b + CT * KP) + trow * (2 * KP) + 2 * tcol;
    bf16x8_t wf[2][3], kf[2];
    auto weigh = [&](int k2) {
      const float4 ta = *reinterpret_cast<const float4*>(tab + CT + 16 * k2 + 4 * hi);
      const float4 tb = *reinterpret_cast<const float4*>(tab + CT + 16 * k2 + 8 + 4 * hi);
      const float tt[8] = {ta.x, ta.y, ta.z, ta.w, tb.x, tb.y, tb.z, tb.w};
      float x[8];
      unpack8(__builtin_bit_cast(uint4, vf[k2]), x);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] *= tt[e];
      split3(x, wf[k2]);
    };
    auto fade = [&](int m) {
#pragma unroll
      for (int e = 0; e < 16; ++e) S[m][e] *= all;
    };
    auto cols_of = [&](int t) { kf[t & 1] = col_frag(kb + 16 * (t / ND) * (2 * KP) + 64 * (t % ND), 2 * KP); };
    cols_of(0);
    weigh(0);
    fade(0);
#pragma unroll
    for (int t = 0; t < 2 * ND; ++t) {
      __builtin_amdgcn_sched_barrier(0);
      if (t + 1 < 2 * ND) cols_of(t + 1);
      if (t + 1 < ND) fade(t + 1);
      if (t == ND - 1) weigh(1);
#pragma unroll
      for (int p = 2; p >= 0; --p) S[t % ND] = mm(kf[t & 1], wf[t / ND][p], S[t % ND]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) {
      __syncthreads();   // every wave is done with this chunk
      stash();
      __syncthreads();
    }
  }
  asm volatile("" : "+v"(scol));   // the offsets of the loads are formed again, not kept through the loop
  if (!ones) {
#pragma unroll
    for (int m = 0; m < ND; ++m)
#pragma unroll
      for (int e = 0; e < 16; ++e) *at_bytes(st, scol + 4 * (32 * m + 8 * (e >> 2) + (e & 3)) * V) = S[m][e];
  } else if (li == 0) {
#pragma unroll
    for (int m = 0; m < ND; ++m)
#pragma unroll
      for (int e = 0; e < 16; ++e) *at_bytes(st, scol + 4 * (32 * m + 8 * (e >> 2) + (e & 3))) = S[m][e];
  }
}

template <int ND, int NW, int NV, bool SILU> hipError_t launch_one(const ChunkLinearArgs& a, RaggedRows r, hipStream_t s) {
  constexpr int KP = 32 * ND + 8, VP = 32 * NW + 8;
  const int waves = NW + (a.n_state != nullptr ? 1 : 0);
  const size_t smem = (size_t)CT * (2 * KP + VP) * sizeof(bf16_t) + (size_t)waves * 4 * CT * sizeof(float);
  hipLaunchKernelGGL((chunk_linear_kernel<ND, NW, NV, SILU>), dim3(a.heads * NV / NW, r.num_seqs), dim3(64 * waves), smem, s, a, r);
  return hipGetLastError();
}
// Four waves stage q and k with half or a quarter of the registers per thread that one or two take, which spill at dim 128, so
// narrow heads that share q and k go together (dim 128, vdim 64, 16 x 1024 tokens of 64 heads: two waves 244 us, two heads in
// four 196 us).
template <int ND, bool SILU> hipError_t launch_nd(const ChunkLinearArgs& a, RaggedRows r, hipStream_t s) {
  const int v = a.vdim / 32;
  if constexpr (!SILU) {   // (with SiLU every head has its own q and k)
    const int share = a.n_state != nullptr ? 1 : a.heads / a.groups;
    if (v == 1 && share % 4 == 0) return launch_one<ND, 4, 1, SILU>(a, r, s);
    if (v == 2 && share % 2 == 0) return launch_one<ND, 4, 2, SILU>(a, r, s);
  }
  if (v == 1) return launch_one<ND, 1, 1, SILU>(a, r, s);
  if (v == 2) return launch_one<ND, 2, 2, SILU>(a, r, s);
  return v == 4 ? launch_one<ND, 4, 4, SILU>(a, r, s) : hipErrorInvalidValue;
}
template <int ND> hipError_t launch_silu(const ChunkLinearArgs& a, RaggedRows r, hipStream_t s) {
  return a.silu ? launch_nd<ND, true>(a, r, s) : launch_nd<ND, false>(a, r, s);
}

}  // namespace

void chunk_linear_cut(ChunkLinearArgs& a, int rows, int num_seqs) {
  const bool sizes = (a.dim == 32 || a.dim == 64 || a.dim == 128) && (a.vdim == 32 || a.vdim == 64 || a.vdim == 128);
  const bool aligned = a.xstride % 8 == 0 && a.qoff % 8 == 0 && a.koff % 8 == 0 && a.voff % 8 == 0 &&
                       (reinterpret_cast<uintptr_t>(a.x) & 15) == 0 && a.xstride < (1 << 25);   // (a chunk's offsets in 32 bits)
  const int64_t n = num_seqs, wgs = a.heads * n, cus = num_cus();
  const bool norm = a.n_state != nullptr, many = wgs > 2 * cus;
  const bool one = a.vdim == 32 && (norm || a.heads / a.groups % 4 != 0);   // one wave stages q, k and v (launch_nd)
  const int64_t state = a.dim * a.vdim;
  a.cut = rows + 1;
  if (!sizes || !aligned || rows < 8 * n || (rows == 8 * n && (many || state < 128 * 128))) return;
  if (!a.silu && ((a.dim == 128 && one && rows < 24 * n) || (a.vdim == 4 * a.dim && many && rows < (norm ? 24 : 12) * n))) return;
  const int64_t load = wgs * state / (64 * 128);   // in states of 64 x 128
  a.cut = norm && state > 64 * 64 && load > 3 * cus && rows <= (load > 6 * cus ? 12 : 10) * n ? 13 : 0;
  a.longest = (int)(rows * (int64_t)a.heads * 5 / (8 * cus)) + 8;
}

hipError_t launch_chunk_linear(const ChunkLinearArgs& a, RaggedRows r, hipStream_t s) {
  switch (a.dim / 32) {
    case 1: return launch_silu<1>(a, r, s);
    case 2: return launch_silu<2>(a, r, s);
    case 4: return launch_silu<4>(a, r, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace die
