// Grouped-query softmax attention over a paged cache, for prompt portions and single decode tokens alike. A cache
// block holds block_size tokens head-major: [G][block_size][K: dim | V: vdim], so the keys and values that one
// key/value head reads from a block are one contiguous piece of memory. A query at position p of its sequence sees the cached positions j <= p
// with p - j < window (window 0: all of them) and, with seg > 0, floor(j / seg) = floor(p / seg) (positions attend
// within fixed segments counted from position 0); its score is (q . k_j) * scale + bias[min(p - j, bias_rows - 1), h]
// (bias optional); the softmax denominator holds one more per-head term exp(sink_h) that belongs to no position
// (the running maximum starts at the sink, the running sum at 1). Query and value widths may differ. With
// a.sigmoid there is no softmax: every visible key weighs sigmoid(score + head_bias[h]) by itself (template
// parameter SIG; no running maximum or sum, no sink, and partial sums of split keys simply add).
//
// Scores, softmax weights and the weighted sum are fp32; storage of q / cache / out is bf16 or fp32.
//
// FMA form (any shape, both storage types): a workgroup of 4 waves owns 4 * RPW rows (a row = one token and one
// of the H / G query heads of ONE key/value head), stages tiles of BK keys and values once in LDS as fp32 (odd row
// stride) and shares them between its rows. Lanes split (key, slice of dim) for the scores, value columns for the
// weighted sum. The matrix-core form for bf16 follows it below.
#include <algorithm>

#include "common.h"
#include "seq_launchers.h"

namespace die {

namespace {

constexpr int WAVES = 4;

template <bool F32> __device__ __forceinline__ float ldt(const void* p, int64_t i) {
  if constexpr (F32)
    return reinterpret_cast<const float*>(p)[i];
  else
    return bf2f(reinterpret_cast<const bf16_t*>(p)[i]);
}
template <bool F32> __device__ __forceinline__ void stt(void* p, int64_t i, float v) {
  if constexpr (F32)
    reinterpret_cast<float*>(p)[i] = v;
  else
    reinterpret_cast<bf16_t*>(p)[i] = f2bf(v);
}

// tanh through one v_exp_f32 and one reciprocal: 1 - 2 / (2^(2 x log2 e) + 1); exact limits at +-inf
__device__ __forceinline__ float fast_tanh(float x) {
  const float e = __builtin_amdgcn_exp2f(x * 2.885390081777927f);
  return 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
}

// the first key a query at position p sees
__device__ __forceinline__ int first_key(const SinkAttnArgs& a, int p) {
  int lo = a.window > 0 ? max(0, p - a.window + 1) : 0;
  if (a.seg > 0) lo = max(lo, p - p % a.seg);
  return lo;
}

template <int BK, int CC, int RPW, bool F32, bool SIG>
__global__ void __launch_bounds__(256) sink_attn_kernel(SinkAttnArgs a, int QS, int KS, int VS) {
  constexpr int RW = RPW * WAVES;
  extern __shared__ float smem[];
  float* qs = smem;                 // [RW][QS]
  float* ks = qs + RW * QS;         // [BK][KS]
  float* vs = ks + BK * KS;         // [BK][VS]
  float* ps = vs + BK * VS;         // [RW][BK]
  const int s = blockIdx.y, g = blockIdx.z, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int H = a.heads, G = a.kv_heads, QPG = H / G, D = a.dim, DV = a.vdim;
  const int roww = D + DV;
  const int q0 = a.cu_q ? a.cu_q[s] : s;
  const int nq = a.cu_q ? a.cu_q[s + 1] - q0 : 1;
  const int nrows = nq * QPG, row0 = blockIdx.x * RW;
  if (row0 >= nrows) return;
  const int ctx = a.ctx_lens[s];
  const int last_row = min(row0 + RW, nrows) - 1;
  const int p_first = (int)a.positions[q0 + row0 / QPG], p_last = (int)a.positions[q0 + last_row / QPG];
  const int jlo = first_key(a, p_first);
  const int jhi = min(p_last, ctx - 1);

  for (int r = wave; r < RW; r += WAVES) {
    const int row = row0 + r;
    const bool ok = row < nrows;
    const int64_t t = q0 + (ok ? row / QPG : 0);
    const int h = g * QPG + (ok ? row % QPG : 0);
    for (int d = lane; d < QS; d += 64) qs[r * QS + d] = (ok && d < D) ? ldt<F32>(a.q, (t * H + h) * D + d) : 0.f;
  }

  int prow[RPW], hrow[RPW], jrow[RPW];
  bool rok[RPW];
  float m[RPW], l[RPW], o[RPW][CC];
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const int row = row0 + wave * RPW + i;
    rok[i] = row < nrows;
    prow[i] = rok[i] ? (int)a.positions[q0 + row / QPG] : -1;
    jrow[i] = first_key(a, max(prow[i], 0));
    hrow[i] = g * QPG + (rok[i] ? row % QPG : 0);
    const bool has_sink = a.sink != nullptr && rok[i];
    m[i] = has_sink ? a.sink[hrow[i]] : -1e30f;
    l[i] = has_sink ? 1.0f : 0.0f;
#pragma unroll
    for (int c = 0; c < CC; ++c) o[i][c] = 0.f;
  }

  constexpr int NP = 64 / BK;
  const int key = lane % BK, part = lane / BK;
  const int dlen = (D + NP - 1) / NP, d0 = part * dlen, d1 = min(D, d0 + dlen);
  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;

  for (int j0 = jlo; j0 <= jhi; j0 += BK) {
    __syncthreads();
    for (int k = wave; k < BK; k += WAVES) {
      const int j = j0 + k;
      const bool in = j <= jhi;
      const int64_t rowp =
          in ? (((int64_t)bt[j / a.block_size] * G + g) * a.block_size + j % a.block_size) * roww : 0;
      for (int d = lane; d < D; d += 64) ks[k * KS + d] = in ? ldt<F32>(a.cache, rowp + d) : 0.f;
      for (int d = lane; d < DV; d += 64) vs[k * VS + d] = in ? ldt<F32>(a.cache, rowp + D + d) : 0.f;
    }
    __syncthreads();
    float acc[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) acc[i] = 0.f;
    for (int d = d0; d < d1; ++d) {
      const float kv = ks[key * KS + d];
#pragma unroll
      for (int i = 0; i < RPW; ++i) acc[i] += qs[(wave * RPW + i) * QS + d] * kv;
    }
    const int j = j0 + key;
    float alpha[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      float sc = acc[i];
#pragma unroll
      for (int off = BK; off < 64; off <<= 1) sc += __shfl_xor(sc, off, 64);
      const int n = prow[i] - j;
      const bool valid = rok[i] && j <= jhi && n >= 0 && j >= jrow[i];
      sc *= a.scale;
      if (a.softcap > 0.f) sc = a.softcap * tanhf(sc / a.softcap);
      if (valid && a.slopes != nullptr) sc -= a.slopes[hrow[i]] * (float)n;
      if (valid && a.bias != nullptr) sc += a.bias[(int64_t)min(n, a.bias_rows - 1) * H + hrow[i]];
      if constexpr (SIG) {
        if (a.head_bias != nullptr) sc += a.head_bias[hrow[i]];
        if (part == 0) ps[(wave * RPW + i) * BK + key] = valid ? 1.0f / (1.0f + expf(-sc)) : 0.f;
        continue;
      }
      sc = valid ? sc : -INFINITY;
      const float mn = fmaxf(m[i], wave_max(sc));
      const float pe = valid ? expf(sc - mn) : 0.f;
      const float psum = wave_sum(part == 0 ? pe : 0.f);
      alpha[i] = expf(m[i] - mn);
      l[i] = l[i] * alpha[i] + psum;
      m[i] = mn;
      if (part == 0) ps[(wave * RPW + i) * BK + key] = pe;
    }
    __syncthreads();
    if constexpr (!SIG) {
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
#pragma unroll
        for (int c = 0; c < CC; ++c) o[i][c] *= alpha[i];
      }
    }
    for (int k = 0; k < BK; ++k) {
      float vc[CC];
#pragma unroll
      for (int c = 0; c < CC; ++c) vc[c] = (lane + 64 * c < DV) ? vs[k * VS + lane + 64 * c] : 0.f;
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
        const float pk = ps[(wave * RPW + i) * BK + k];
#pragma unroll
        for (int c = 0; c < CC; ++c) o[i][c] += pk * vc[c];
      }
    }
  }

#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    if (!rok[i]) continue;
    const int row = row0 + wave * RPW + i;
    const int64_t t = q0 + row / QPG;
    const float inv = SIG ? 1.0f : (l[i] > 0.f ? 1.0f / l[i] : 0.f);
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      const int col = lane + 64 * c;
      if (col < DV) stt<F32>(a.out, (t * H + hrow[i]) * DV + col, o[i][c] * inv);
    }
  }
}

inline int odd(int x) { return x | 1; }

template <int BK, int CC, int RPW, bool F32> hipError_t launch_one(const SinkAttnArgs& a, hipStream_t s) {
  constexpr int RW = RPW * WAVES;
  const int QS = odd(a.dim), KS = odd(a.dim), VS = odd(a.vdim);
  const size_t lds = sizeof(float) * ((size_t)RW * QS + (size_t)BK * KS + (size_t)BK * VS + (size_t)RW * BK);
  if (lds > 150 * 1024) return hipErrorInvalidValue;
  auto kern = a.sigmoid ? sink_attn_kernel<BK, CC, RPW, F32, true> : sink_attn_kernel<BK, CC, RPW, F32, false>;
  if (lds > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds);
    if (e != hipSuccess) return e;
  }
  const int qpg = a.heads / a.kv_heads;
  const int tiles = (a.max_q * qpg + RW - 1) / RW;
  hipLaunchKernelGGL(kern, dim3(tiles, a.num_seqs, a.kv_heads), dim3(256), lds, s, a, QS, KS, VS);
  return hipGetLastError();
}

template <int BK, int RPW, bool F32> hipError_t launch_cc(const SinkAttnArgs& a, hipStream_t s) {
  if (a.vdim <= 64) return launch_one<BK, 1, RPW, F32>(a, s);
  if (a.vdim <= 128) return launch_one<BK, 2, RPW, F32>(a, s);
  if (a.vdim <= 256) return launch_one<BK, 4, RPW, F32>(a, s);
  return hipErrorInvalidValue;
}

template <bool F32> hipError_t launch_fma(const SinkAttnArgs& a, hipStream_t s) {
  const int qpg = a.heads / a.kv_heads;
  // few rows per (sequence, key/value head): one row per wave, smaller key tiles
  if (a.max_q * qpg <= 4) return launch_cc<32, 1, F32>(a, s);
  if (a.dim + a.vdim > 384) return launch_cc<32, 4, F32>(a, s);
  return launch_cc<64, 4, F32>(a, s);
}

// ---------------------------------------------------------------------------------------------------
// bf16 on the matrix cores (v_mfma_f32_32x32x16_bf16), for dim % 16 == 0, dim <= 256, vdim % 8 == 0, vdim <= 256 and pages of a
// power of two tokens (the
// value columns of a staged row are padded to a multiple of 32; what the padding holds only reaches output columns that
// do not exist).
// Workgroup = NW waves x 32 rows of one (sequence, key/value head); NW = 1 for steps of few rows (decode). Keys are staged
// in LDS as rows [K_g | V_g], STG at a time in two buffers in turn: one barrier per stage, the next stage's global loads in
// flight while this one is computed. Per tile of 32 keys:
//   S^T[key][q] = K Q^T        A = K rows from LDS, B = Q rows               (dim / 16 MFMAs; dim <= 128: Q in registers)
//   online softmax per query column (a lane pair owns a query), fp32 scores and weights in log2 units, the bias
//   per distance added before, the running max seeded with the sink; the max moves (and O is rescaled) only when a tile
//   exceeds it by 2^LAZY; P is rounded to bf16 only as MFMA operand
//   O^T[d][q] += V^T P^T      A = the value columns of the same tile read transposed (ds_read_tr16_b64),
//                              B = P^T straight from the score accumulator   (2 * vdim / 32 MFMAs)
// Split keys (decode over long contexts): split z takes keys [jlo + z * chunk, + chunk) and writes its
// unnormalised O, running max and sum to a workspace; sink_attn_merge_kernel combines them. The sink enters
// split 0 only.
constexpr int MKT = 32;
constexpr int BT_LDS_MAX = 2048;
constexpr float LAZY = 8.0f;
// Weights that enter the products in two bf16 parts are taken 1 + 2^-8 times, and the sums divided by that: the second part is then positive
// wherever the weight is (a rounding leaves up to 2^-9 of it, of either sign), so that an infinite value stays what it is: zero times it
// would be NaN, and a negative part of the other sign. (From weights of 2^-124 on; the part is no bf16 number below.)
constexpr float OVER = 1.0f + 0x1p-8f;
// second parts of the weights x, y, whose first ones are in b
__device__ __forceinline__ uint32_t rest2(float x, float y, uint32_t b) {
  return pack2(fmaf(x, OVER, -__uint_as_float(b << 16)), fmaf(y, OVER, -__uint_as_float(b & 0xffff0000u)));
}
// keys per stage; whether the queries live in registers (else in LDS)
template <int NW, int NKC> constexpr int stage_keys() { return NW == 4 && NKC <= 16 ? 64 : MKT; }
template <int NDB, int NW, int NKC> constexpr bool q_in_regs() { return NKC <= 16 && (NW == 4 || NDB <= 4); }
typedef __attribute__((address_space(3))) short4_t lds_short4;
typedef __attribute__((ext_vector_type(8))) short short8_t;

// FINE: the weights enter the products in two bf16 parts (SinkAttnArgs::fine)
template <int NDB, int NW, int NKC, bool SIG, bool FINE>
__global__ void __launch_bounds__(64 * NW, NW == 4 && NKC <= 16 && NDB <= 4 ? 2 : 1) sink_attn_mfma_kernel(SinkAttnArgs a, int KP, int QP, int QR, int BTC,
                                                                float* ws_o, float* ws_ml, int nsplit, int chunk) {
  constexpr int ROWS = 32 * NW, NT = 64 * NW, STG = stage_keys<NW, NKC>();
  constexpr bool QREG = q_in_regs<NDB, NW, NKC>();
  constexpr int NKK = QREG ? NKC / 2 : 1;                     // steps of 16 dims of a query held in registers
  constexpr int NPF = (STG * (4 * NDB + NKC) + NT - 1) / NT;  // 16-byte chunks of a stage per thread
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  // QR query rows are staged (none with QREG): all ROWS of a prompt-sized step; for steps of few rows (NW = 1) only the rows there
  // can be plus one zero row that every further query column reads, which keeps the workgroup's LDS small enough
  // for two waves per SIMD
  bf16_t* qs = reinterpret_cast<bf16_t*>(smem_raw);          // [QR][QP]
  bf16_t* ks = qs + QR * QP;                                  // two of [STG][KP] = [K_g | V_g]
  int bx = blockIdx.x, by = blockIdx.y;
  {
    // XCD k (workgroups are dealt round-robin by linear id) takes a contiguous eighth of the sequence-major tile
    // list, so one sequence's cache rows stay in one L2
    const unsigned total = gridDim.x * gridDim.y, lin = blockIdx.x + gridDim.x * blockIdx.y;
    if (total % 8 == 0) {
      const unsigned nl = (lin % 8) * (total / 8) + lin / 8;
      bx = (int)(nl % gridDim.x);
      by = (int)(nl / gridDim.x);
    }
    bx = gridDim.x - 1 - bx;   // a sequence's last rows see the most keys: they start first
  }
  const int H = a.heads, G = a.kv_heads, QPG = H / G, D = a.dim, DV = a.vdim;
  const int s = by, g = blockIdx.z % G, z = blockIdx.z / G;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tid = threadIdx.x;
  const int roww = D + DV;
  const int q0 = a.cu_q ? a.cu_q[s] : s;
  const int nq = a.cu_q ? a.cu_q[s + 1] - q0 : 1;
  const int nrows = nq * QPG, row0 = bx * ROWS;
  if (row0 >= nrows) return;
  const int ctx = a.ctx_lens[s];
  const int last_row = min(row0 + ROWS, nrows) - 1;
  const int p_first = (int)a.positions[q0 + row0 / QPG], p_last = (int)a.positions[q0 + last_row / QPG];
  int jlo = first_key(a, p_first);
  int jhi = min(p_last, ctx - 1);
  if (nsplit > 1) {
    jlo += z * chunk;
    jhi = min(jhi, jlo + chunk - 1);
  }
  const bf16_t* qg = reinterpret_cast<const bf16_t*>(a.q);
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  const int qcol = lane & 31, hh = lane >> 5;
  const int myrow = row0 + wave * 32 + qcol;
  const bool rok = myrow < nrows;
  const int myh = g * QPG + (rok ? myrow % QPG : 0);
  const int64_t orow = rok ? (int64_t)(q0 + myrow / QPG) * H + myh : 0;
  const int64_t wrows = (int64_t)a.total_q * H;
  if (jlo > jhi) {  // an empty split (uniform over the workgroup): it only reports that it holds nothing
    if (nsplit > 1 && rok && hh == 0) {
      ws_ml[((int64_t)z * wrows + orow) * 2] = -1e30f;
      ws_ml[((int64_t)z * wrows + orow) * 2 + 1] = 0.f;
    }
    return;
  }

  const int nkk = D / 16;
  bf16x8_t qf[NKK];
  if constexpr (QREG) {
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (rok && kk < nkk) v = *reinterpret_cast<const uint4*>(qg + orow * D + 16 * kk + 8 * hh);
      qf[kk] = __builtin_bit_cast(bf16x8_t, v);
    }
  } else {
    const int lch = D / 8;
    for (int idx = tid; idx < QR * lch; idx += NT) {
      const int r = idx / lch, c = idx % lch, row = row0 + r;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (row < nrows) {
        const int64_t t = q0 + row / QPG;
        v = *reinterpret_cast<const uint4*>(qg + (t * H + g * QPG + row % QPG) * D + 8 * c);
      }
      *reinterpret_cast<uint4*>(qs + r * QP + 8 * c) = v;
    }
  }

  const bool wave_live = row0 + wave * 32 < nrows;
  const int prow = rok ? (int)a.positions[q0 + myrow / QPG] : -1;
  const int jrow = first_key(a, max(prow, 0));
  const unsigned seen = rok ? max(min(prow, jhi) - jrow + 1, 0) : 0;   // this row sees keys jrow .. jrow + seen - 1
  constexpr float LOG2E = 1.4426950408889634f;
  const float sl2 = a.scale * LOG2E;
  const bool shaped = a.softcap > 0.f || a.slopes != nullptr;
  const bool plain = !shaped && a.bias == nullptr && sl2 > 0.f;
  const float capl2 = a.softcap * LOG2E, s_over_cap = a.softcap > 0.f ? a.scale / a.softcap : 0.f;
  const float cap_m2 = -2.0f * capl2, s2_over_cap = s_over_cap * 2.885390081777927f;
  const float slope2 = a.slopes != nullptr ? a.slopes[myh] * LOG2E : 0.f;
  const float hb2 = SIG && a.head_bias != nullptr ? a.head_bias[myh] * LOG2E : 0.f;
  const bool has_sink = a.sink != nullptr && rok && z == 0;
  float m = has_sink ? a.sink[myh] * LOG2E : -1e30f;
  float l = has_sink ? 1.0f : 0.0f;
  f32x16_t o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;

  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
  const int kch = (D + DV) / 8;
  bf16_t* spare = ks + 2 * STG * KP;   // [KP]: takes a stage's surplus chunks
  int* btl = reinterpret_cast<int*>(spare + KP);
  const int b_lo = jlo / a.block_size, nbt = jhi / a.block_size - b_lo + 1;
  const bool bt_lds = nbt <= BTC;
  if (bt_lds)
    for (int u = tid; u < nbt; u += NT) btl[u] = bt[b_lo + u];
  u32x4_t pf[NPF];   // (native vectors: arrays of uint4 structs go through scratch)
  // chunk idx = tid + u * NT of a tile is (key k, 16-byte piece c) = (idx / kch, idx % kch): one division per
  // thread, then steps of (NT / kch, NT % kch); a block size that is a power of two divides by shifting
  const int k_first = tid / kch, c_first = tid - k_first * kch, k_step = NT / kch, c_step = NT - k_step * kch;
  const int bs_shift = __builtin_ctz(a.block_size);   // a power of two (mfma_ok)
  const uint32_t rowb = 2 * roww, blkb = (uint32_t)G * a.block_size * rowb;
  const char* cg = reinterpret_cast<const char*>(cache) + (int64_t)g * a.block_size * rowb;
  // all block ids first, then all loads: no load waits for another's block id. Keys beyond the last re-read it: their
  // scores are masked
  auto fetch = [&](int j0, bool lds) {
    int jj[NPF], cc[NPF];
    uint32_t blk[NPF];
    int k = k_first, c = c_first;
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      jj[u] = min(j0 + min(k, STG - 1), jhi);
      cc[u] = c;
      k += k_step;
      c += c_step;
      if (c >= kch) {
        c -= kch;
        ++k;
      }
    }
    if (lds) {
#pragma unroll
      for (int u = 0; u < NPF; ++u) blk[u] = btl[(jj[u] >> bs_shift) - b_lo];
    } else {
#pragma unroll
      for (int u = 0; u < NPF; ++u) blk[u] = bt[jj[u] >> bs_shift];
    }
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      const uint32_t in = (uint32_t)(jj[u] & (a.block_size - 1)) * rowb + 16 * cc[u];
      pf[u] = *reinterpret_cast<const u32x4_t*>(cg + (uint64_t)blk[u] * blkb + in);
    }
  };
  fetch(jlo, false);
  const int pitchB = KP * 2;
  const int g16 = lane >> 4, i16 = lane & 15;
  const int voff = (4 * hh + (i16 >> 2)) * pitchB + (D + 16 * (g16 & 1) + 4 * (i16 & 3)) * 2;
  const float* bias = a.bias ? a.bias + myh : nullptr;
  // distances from bias_rows - 1 on share the table's last row: a lane whose 16 keys of a tile all lie that far
  // back adds that one value without looking anything up
  const float bias_far = bias ? bias[(int64_t)(a.bias_rows - 1) * H] * LOG2E : 0.f;
  // a tile is interior for a wave when every one of its 32 x 32 (key, row) pairs is visible: no masking then
  const int wrow_first = row0 + wave * 32, wrow_last = wrow_first + 31;
  const bool wave_full = wrow_last < nrows;
  const int pw_first = wave_live ? (int)a.positions[q0 + wrow_first / QPG] : 0;
  const int pw_last = wave_live ? (int)a.positions[q0 + min(wrow_last, nrows - 1) / QPG] : 0;
  const int jw_first = first_key(a, pw_first), jw_last = first_key(a, pw_last);
  int buf = 0;
  for (int js = jlo; js <= jhi; js += STG, buf ^= 1) {
    bf16_t* kst = ks + buf * STG * KP;   // last read two stages ago: every wave has passed a barrier since
    {
      int k = k_first, c = c_first;
#pragma unroll
      for (int u = 0; u < NPF; ++u) {
        *reinterpret_cast<u32x4_t*>((k < STG ? kst + k * KP : spare) + 8 * c) = pf[u];
        k += k_step;
        c += c_step;
        if (c >= kch) {
          c -= kch;
          ++k;
        }
      }
    }
    __syncthreads();
    if (js + STG <= jhi) fetch(js + STG, bt_lds);  // in flight while this stage is computed
    for (int j0 = js; j0 < js + STG && j0 <= jhi; j0 += MKT) {
      if (!wave_live || j0 > pw_last || j0 + MKT <= jw_first) continue;   // nothing of this tile is visible to the wave
      const bf16_t* kt = kst + (j0 - js) * KP;
      const char* vbase = reinterpret_cast<const char*>(kt) + voff;
      f32x16_t sc;
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[r] = 0.f;
      const bf16_t* ka = kt + qcol * KP + 8 * hh;
      if constexpr (QREG) {
        // all NKK steps without a branch between them, so that their LDS reads are in flight together: beyond dim the
        // query's fragments are zero, and the key's first columns stand in
        bf16x8_t kf[NKK];
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk)
          kf[kk] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(ka + (kk < nkk ? 16 * kk : 0)));
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kk], qf[kk], sc, 0, 0, 0);
      } else {
        const bf16_t* qb = qs + min(wave * 32 + qcol, QR - 1) * QP + 8 * hh;
#pragma unroll 4
        for (int kk = 0; kk < nkk; ++kk) {
          const bf16x8_t af = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(ka + 16 * kk));
          const bf16x8_t bfr = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(qb + 16 * kk));
          sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bfr, sc, 0, 0, 0);
        }
      }
      float mx = -INFINITY, mul = 1.0f;   // sc * mul: scores in log2 units
      const bool interior = wave_full && j0 + MKT - 1 <= min(pw_first, jhi) && j0 >= jw_last;
      if (plain) {
        mul = sl2;
        if (!interior) {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            sc[r] = (unsigned)(j0 + (r & 3) + 8 * (r >> 2) + 4 * hh - jrow) < seen ? sc[r] : -INFINITY;
        }
        if constexpr (!SIG) {
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[r]);
          mx *= sl2;
        }
      } else if (shaped) {
        // capped scores and / or a linear distance penalty: cap * tanh(s * scale / cap) - slope * n, in log2 units.
        // tanh = 1 - 2 / (2^(2 x log2 e) + 1), so the capped score is one multiply-add of the reciprocal; the
        // distance of score r is that of score 0 minus a constant
        const float nf0 = (float)(prow - j0 - 4 * hh);
        if (interior && bias == nullptr) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float nf = nf0 - (float)((r & 3) + 8 * (r >> 2));
            float v;
            if (a.softcap > 0.f)
              v = fmaf(cap_m2, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(sc[r] * s2_over_cap) + 1.0f), capl2);
            else
              v = sc[r] * sl2;
            v = fmaf(-slope2, nf, v);
            sc[r] = v;
            mx = fmaxf(mx, v);
          }
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int j = j0 + (r & 3) + 8 * (r >> 2) + 4 * hh;
            const int n = prow - j;
            const bool valid = interior || (rok && j <= jhi && n >= 0 && j >= jrow);
            float v = a.softcap > 0.f ? capl2 * fast_tanh(sc[r] * s_over_cap) : sc[r] * sl2;
            v -= slope2 * (float)n;
            if (bias != nullptr && valid) v += bias[(int64_t)min(n, a.bias_rows - 1) * H] * LOG2E;
            v = valid ? v : -INFINITY;
            sc[r] = v;
            mx = fmaxf(mx, v);
          }
        }
      } else if (interior) {
        const bool far = bias == nullptr || prow - (j0 + 27 + 4 * hh) >= a.bias_rows - 1;
        if (far) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float v = sc[r] * sl2 + bias_far;
            sc[r] = v;
            mx = fmaxf(mx, v);
          }
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int n = prow - (j0 + (r & 3) + 8 * (r >> 2) + 4 * hh);
            const float v = sc[r] * sl2 + bias[(int64_t)min(n, a.bias_rows - 1) * H] * LOG2E;
            sc[r] = v;
            mx = fmaxf(mx, v);
          }
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = j0 + (r & 3) + 8 * (r >> 2) + 4 * hh;
          const int n = prow - j;
          const bool valid = rok && j <= jhi && n >= 0 && j >= jrow;
          float v = sc[r] * sl2;
          if (bias != nullptr && valid) v += bias[(int64_t)min(n, a.bias_rows - 1) * H] * LOG2E;
          v = valid ? v : -INFINITY;
          sc[r] = v;
          mx = fmaxf(mx, v);
        }
      }
      float alpha = 1.0f;
      if constexpr (SIG) {
        // sigmoid: 1 / (1 + 2^-(v + bias)); a masked score is -inf and weighs 0
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(fmaf(-sc[r], mul, -hb2)));
      } else {
        mx = xor32_max(mx);
        const float mn = mx > m + LAZY ? mx : m;
        alpha = __builtin_amdgcn_exp2f(m - mn);   // v_exp_f32: arguments are <= 0 or -inf here
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float pe = __builtin_amdgcn_exp2f(fmaf(sc[r], mul, -mn));
          sc[r] = pe;
          sum += pe;
        }
        sum = xor32_sum(sum);
        l = l * alpha + sum;
        m = mn;
      }
      bf16x8_t pfr[2], plr[2];
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        uint4 w;
        w.x = pack2(sc[8 * s2 + 0], sc[8 * s2 + 1]);
        w.y = pack2(sc[8 * s2 + 2], sc[8 * s2 + 3]);
        w.z = pack2(sc[8 * s2 + 4], sc[8 * s2 + 5]);
        w.w = pack2(sc[8 * s2 + 6], sc[8 * s2 + 7]);
        pfr[s2] = __builtin_bit_cast(bf16x8_t, w);
        if constexpr (FINE) {
          auto rest = [&](int r, uint32_t b) { return rest2(sc[8 * s2 + r], sc[8 * s2 + r + 1], b); };
          plr[s2] = __builtin_bit_cast(bf16x8_t, make_uint4(rest(0, w.x), rest(2, w.y), rest(4, w.z), rest(6, w.w)));
        }
      }
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        if (!SIG && alpha != 1.0f) {
#pragma unroll
          for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
        }
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const char* a0 = vbase + (16 * s2) * pitchB + 64 * db;
          const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(a0));
          const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(a0 + 8 * pitchB));
          const short8_t a8 = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a8), pfr[s2], o[db], 0, 0, 0);
          if constexpr (FINE) o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a8), plr[s2], o[db], 0, 0, 0);
        }
      }
    }
  }
  if constexpr (FINE) l *= OVER;
  if (NW > 1 && nsplit <= 1) {
    // whole rows of 16-byte pieces through LDS: straight from the accumulators every store would touch 32 rows
    const float inv = SIG ? 1.0f : (l > 0.f ? 1.0f / l : 0.f);
    const int OP = 2 * (DV + 8);
    char* ob = smem_raw + wave * 32 * OP;
    __syncthreads();   // every wave is done with the keys
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        if (32 * db + 8 * q4 >= DV) continue;
        uint2 w;
        w.x = pack2(o[db][4 * q4 + 0] * inv, o[db][4 * q4 + 1] * inv);
        w.y = pack2(o[db][4 * q4 + 2] * inv, o[db][4 * q4 + 3] * inv);
        *reinterpret_cast<uint2*>(ob + qcol * OP + 2 * (32 * db + 8 * q4 + 4 * hh)) = w;
      }
    }
    __syncthreads();
    const int nch = DV / 8;
    bf16_t* og = reinterpret_cast<bf16_t*>(a.out);
    for (int idx = lane; idx < 32 * nch; idx += 64) {
      const int r = idx / nch, c = idx - r * nch, row = row0 + wave * 32 + r;
      if (row >= nrows) break;
      const int t = row / QPG;
      const uint4 w = *reinterpret_cast<const uint4*>(ob + r * OP + 16 * c);
      *reinterpret_cast<uint4*>(og + ((int64_t)(q0 + t) * H + g * QPG + (row - t * QPG)) * DV + 8 * c) = w;
    }
    return;
  }
  if (!rok) return;
  if (nsplit > 1) {
    float* wo = ws_o + ((int64_t)z * wrows + orow) * DV;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        if (32 * db + 8 * q4 < DV)
          *reinterpret_cast<float4*>(wo + 32 * db + 8 * q4 + 4 * hh) =
              make_float4(o[db][4 * q4], o[db][4 * q4 + 1], o[db][4 * q4 + 2], o[db][4 * q4 + 3]);
    if (hh == 0) {
      ws_ml[((int64_t)z * wrows + orow) * 2] = SIG ? 0.f : m;
      ws_ml[((int64_t)z * wrows + orow) * 2 + 1] = SIG ? 1.0f : l;
    }
    return;
  }
  const float inv = SIG ? 1.0f : (l > 0.f ? 1.0f / l : 0.f);
  bf16_t* op = reinterpret_cast<bf16_t*>(a.out) + orow * DV;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      if (32 * db + 8 * q4 >= DV) continue;
      uint2 w;
      w.x = pack2(o[db][4 * q4 + 0] * inv, o[db][4 * q4 + 1] * inv);
      w.y = pack2(o[db][4 * q4 + 2] * inv, o[db][4 * q4 + 3] * inv);
      *reinterpret_cast<uint2*>(op + 32 * db + 8 * q4 + 4 * hh) = w;
    }
  }
}


// The row tile, sequence and key/value head of a workgroup, of a grid (tiles, sequences, heads). A pair of sequence and head has its own
// cache rows. Workgroups go to the 8 XCDs, which have an L2 each, in turn: pair u is XCD u % 8's, so that its cache rows are in one L2
// and long and short sequences are spread (an eighth of the list for each XCD left it with neighbours of a sorted batch: 16 sequences of 519 -
// 1000 tokens behind 150 - 300, 4 heads: 165 us, now 131). Pairs that are no multiple of 8 are dealt tile by tile. Last tiles see the most keys
// and start first, those of all pairs together.
__device__ __forceinline__ void tile_of(int G, int& bx, int& s, int& g) {
  const unsigned nx = gridDim.x, pairs = gridDim.y * gridDim.z, lin = blockIdx.x + nx * (blockIdx.y + gridDim.y * blockIdx.z);
  unsigned u, t;
  if (pairs % 8 == 0) {
    const unsigned own = pairs / 8, j = lin / 8;
    t = j / own;
    u = lin % 8 + 8 * (j % own);
  } else {
    t = lin / pairs;
    u = lin % pairs;
  }
  bx = (int)(nx - 1 - t);
  s = (int)(u / (unsigned)G);
  g = (int)(u % (unsigned)G);
}

// Prompt-sized steps at the common widths (dim 64 or 128, vdim 64, 128 or 256), keys not split: the same algorithm with 16 rows per
// wave and 16x16x32 products, so that the sums and queries take 32 + 16 registers at 128 + 128 and 4 waves share a SIMD: one's
// softmax and waits run beside the others' products. A workgroup of 4 waves takes 64 rows; key tiles [K_g | V_g] come by DMA into two
// buffers, one barrier per tile. A tile of 32 rows by KCH 16-byte pieces lies in LDS without gaps; the pieces of a row are exchanged
// (XOR) so that 16 consecutive rows' reads of one piece fall on all banks, and the transposed reads of 8 rows by two pieces (a rotated row number:
// by the plain one pairs of rows shared banks).
// Bound by the issue of vector instructions (110 per wave and tile beside 16 products). 16 ragged sequences of up to 1024 rows, 16 heads
// in 4 groups of 128 + 128, a window of 512: 32 rows per wave (above), two waves per SIMD and tiles through registers took 110 us,
// this takes 82 (99 before tile_of and the two waits named below); 16 sequences of 500, vdim 256: 222 -> 90. Long sequences whose keys are all seen (the other kernel reads LDS half as
// often there): 4 x 1500 rows of 32 heads 161 -> 149, 4 x 4096 of 16 558 -> 475, 1 x 16384 2582 -> 2501. With a bias per distance
// (130 distances, a window of 1024) 16 x 1024 rows 160 -> 141, 4 x 4096 240 -> 228 (where every score looks its distance up: 182, 297).
template <int NK, int NV> struct RowTile {
  static constexpr int KCH = 4 * NK + 2 * NV, NPF = MKT * KCH / 256, BYTES = MKT * KCH * 16;
  static constexpr int X = KCH % 16 == 0 ? 16 : 8;   // rows r and r + 16 / X share banks
  static __device__ __forceinline__ int swz(int row) {
    const int i = row / (16 / X) % X;
    return (2 * i & (X - 1)) | i / (X / 2);
  }
  static constexpr int OP = 32 * NV + 16;            // pitch of a result row in LDS
  static constexpr int TABLE = 1024;                 // key rows in LDS
  static constexpr int LDS = 2 * BYTES + 4 * TABLE > 64 * OP ? 2 * BYTES + 4 * TABLE : 64 * OP;
};
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void global_cvoid;

template <int NK, int NV, bool SIG, bool FINE>
__global__ void __launch_bounds__(256, NV <= 8 ? 4 : 3) sink_attn_rows_kernel(SinkAttnArgs a) {
  using Z = RowTile<NK, NV>;
  constexpr int KCH = Z::KCH, D = 32 * NK, DV = 16 * NV, roww = D + DV;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];   // two tiles, key rows; at the end the results
  const int H = a.heads, G = a.kv_heads, QPG = H / G;
  int bx, s, g;
  tile_of(G, bx, s, g);
  const int lane = threadIdx.x & 63, tid = threadIdx.x, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q0 = a.cu_q ? a.cu_q[s] : s;
  const int nq = a.cu_q ? a.cu_q[s + 1] - q0 : 1;
  const int nrows = nq * QPG, row0 = bx * 64;
  if (row0 >= nrows) return;
  const int last_row = min(row0 + 64, nrows) - 1;
  const int p_first = (int)a.positions[q0 + row0 / QPG], p_last = (int)a.positions[q0 + last_row / QPG];
  const int jlo = first_key(a, p_first), jhi = min(p_last, a.ctx_lens[s] - 1);
  const int nt = jhi < jlo ? 0 : (jhi - jlo) / MKT + 1;

  // cache rows of the workgroup's keys in LDS, TABLE keys at a time
  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
  int* rows = reinterpret_cast<int*>(smem_raw + 2 * Z::BYTES);
  const int bs_shift = __builtin_ctz(a.block_size);   // a power of two (mfma_ok)
  int jt = jlo;
  auto stage_rows = [&]() {
    for (int u = tid; u < Z::TABLE && jt + u <= jhi; u += 256)
      rows[u] = ((bt[(jt + u) >> bs_shift] * G + g) << bs_shift) + ((jt + u) & (a.block_size - 1));
    __syncthreads();
  };
  stage_rows();
  // piece u of this thread: 16 bytes of key krow + u * 256 / KCH of the tile, or of the next one where a row ends
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  int krow[Z::NPF], pcol[Z::NPF];
#pragma unroll
  for (int u = 0; u < Z::NPF; ++u) {
    const int idx = tid + 256 * u;
    krow[u] = idx / KCH;
    pcol[u] = 8 * ((idx % KCH) ^ Z::swz(krow[u]));
  }
  auto fetch = [&](int j0, int buf) {   // (keys beyond the last repeat it)
    if (min(j0 + MKT - 1, jhi) - jt >= Z::TABLE) {
      __syncthreads();
      jt = j0;
      stage_rows();
    }
    const int at = j0 - jt, end = jhi - jt;
    int row[Z::NPF];
#pragma unroll
    for (int u = 0; u < Z::NPF; ++u) row[u] = rows[min(at + krow[u], end)];
    __builtin_amdgcn_sched_barrier(0);   // (all lookups, then the loads: they would go in turns, each waited for)
#pragma unroll
    for (int u = 0; u < Z::NPF; ++u) {
      char* to = smem_raw + buf * Z::BYTES + (256 * u + 64 * wave) * 16;
      __builtin_amdgcn_global_load_lds((global_cvoid*)(cache + ((uint64_t)(uint32_t)row[u] * roww + pcol[u])), (lds_void*)to, 16, 0, 0);
    }
  };
  if (nt > 0) fetch(jlo, 0);

  const int wrow = row0 + wave * 16, myrow = wrow + li;
  const bool rok = myrow < nrows, wave_live = wrow < nrows, wave_full = wrow + 15 < nrows;
  const int tq = q0 + (rok ? myrow / QPG : 0), myh = g * QPG + (rok ? myrow % QPG : 0);   // (rows beyond the last repeat the first)
  const int64_t orow = (int64_t)tq * H + myh;
  bf16x8_t qf[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k)
    qf[k] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(a.q) + orow * D + 32 * k + 8 * lg));
  const int prow = rok ? (int)a.positions[tq] : -1;
  const int jrow = first_key(a, max(prow, 0));
  const unsigned seen = rok ? max(min(prow, jhi) - jrow + 1, 0) : 0;   // this row sees keys jrow .. jrow + seen - 1
  // a tile is interior for a wave when every one of its 32 x 16 (key, row) pairs is visible: no masking then
  const int pw_first = wave_live ? (int)a.positions[q0 + wrow / QPG] : 0;
  const int pw_last = wave_live ? (int)a.positions[q0 + min(wrow + 15, nrows - 1) / QPG] : 0;
  const int jw_first = first_key(a, pw_first), jw_last = first_key(a, pw_last);
  constexpr float LOG2E = 1.4426950408889634f;
  const float sl2 = a.scale * LOG2E;
  const bool shaped = a.softcap > 0.f || a.slopes != nullptr;
  const bool plain = !shaped && a.bias == nullptr && sl2 > 0.f;
  const float capl2 = a.softcap * LOG2E, s2_over_cap = a.softcap > 0.f ? a.scale / a.softcap * 2.885390081777927f : 0.f;
  const float slope2 = a.slopes != nullptr ? a.slopes[myh] * LOG2E : 0.f;
  const float hb2 = SIG && a.head_bias != nullptr ? a.head_bias[myh] * LOG2E : 0.f;
  const float* bias = a.bias ? a.bias + myh : nullptr;
  const float bias_far = bias ? bias[(int64_t)(a.bias_rows - 1) * H] * LOG2E : 0.f;
  const bool has_sink = !SIG && a.sink != nullptr && rok;
  float m = has_sink ? a.sink[myh] * LOG2E : -1e30f;
  float l = has_sink && lg == 0 ? 1.0f : 0.0f;   // (the sum of this lane's keys)
  f32x4_t o[NV];
#pragma unroll
  for (int db = 0; db < NV; ++db) o[db] = f32x4_t{};
  // K fragments: key li of 16, piece 4 k + lg; V fragments: keys 4 lg .. of either 16 (the order in which the weights lie in
  // registers), columns 16 db ..
  const int ksw = Z::swz(li), vrow = 4 * lg + (li >> 2), vsw = Z::swz(vrow);
  const int kat = 16 * li * KCH, vat = 16 * vrow * KCH + 8 * (li & 1), vpc = 4 * NK + (li >> 1 & 1);
  // The queries are here. (Without this the compiler waits for them in the loop, behind the next tile's DMA and so for that too.)
  __builtin_amdgcn_s_waitcnt(15 << 8 | 7 << 4);
  for (int i = 0; i < nt; ++i) {
    const int j0 = jlo + i * MKT;
    // tile i is in LDS for every wave, and every wave has left the other buffer
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(7 << 4);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (i + 1 < nt) fetch(j0 + MKT, (i + 1) & 1);
    if (!wave_live || j0 > pw_last || j0 + MKT <= jw_first) continue;   // nothing of this tile is visible to the wave
    const char* ks = smem_raw + (i & 1) * Z::BYTES;
    f32x4_t sc[2] = {};
#pragma unroll
    for (int k = 0; k < NK; ++k)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint4 w = *reinterpret_cast<const uint4*>(ks + kat + 256 * KCH * t + 16 * ((4 * k + lg) ^ ksw));
        sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w), qf[k], sc[t], 0, 0, 0);
      }
    const bool interior = wave_full && j0 + MKT - 1 <= min(pw_first, jhi) && j0 >= jw_last;
    float mul = 1.0f;   // sc * mul: scores in log2 units
    if (plain) {
      mul = sl2;
    } else {
      // capped scores: cap * tanh(s * scale / cap) = cap - 2 cap / (2^(2 x log2 e) + 1), one multiply-add of the reciprocal
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = prow - (j0 + 16 * t + 4 * lg + e);
          float v = sc[t][e];
          if (a.softcap > 0.f)
            v = fmaf(-2.0f * capl2, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(v * s2_over_cap) + 1.0f), capl2);
          else
            v *= sl2;
          sc[t][e] = fmaf(-slope2, (float)n, v);
        }
      if (bias != nullptr) {
        // distances from bias_rows - 1 on share the table's last row: a lane whose keys all lie that far back looks nothing up
        const int n0 = prow - (j0 + 4 * lg);   // of the lane's first key; the others are 1 .. 3 and 16 .. 19 nearer
        if (n0 - 19 >= a.bias_rows - 1) {
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) sc[t][e] += bias_far;
        } else {
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              sc[t][e] += bias[(int64_t)min(max(n0 - 16 * t - e, 0), a.bias_rows - 1) * H] * LOG2E;
        }
      }
    }
    if (!interior) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[t][e] = (unsigned)(j0 + 16 * t + 4 * lg + e - jrow) < seen ? sc[t][e] : -INFINITY;
    }
    float alpha = 1.0f;
    if constexpr (SIG) {   // 1 / (1 + 2^-(v + bias)); a masked score is -inf and weighs 0
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[t][e] = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(fmaf(-sc[t][e], mul, -hb2)));
    } else {
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, sc[t][e]);
      mx = xor16_max(xor32_max(mx * mul));
      const float mn = mx > m + LAZY ? mx : m;
      alpha = __builtin_amdgcn_exp2f(m - mn);   // v_exp_f32: arguments are <= 0 or -inf here
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sc[t][e] = __builtin_amdgcn_exp2f(fmaf(sc[t][e], mul, -mn));
          sum += sc[t][e];
        }
      l = l * alpha + sum;
      m = mn;
    }
    const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, make_uint4(pack2(sc[0][0], sc[0][1]), pack2(sc[0][2], sc[0][3]),
                                                                pack2(sc[1][0], sc[1][1]), pack2(sc[1][2], sc[1][3])));
    bf16x8_t pl = {};   // what the rounding left, and 2^-8 of the weight (OVER)
    if constexpr (FINE) {
      const uint4 h = __builtin_bit_cast(uint4, pf);
      pl = __builtin_bit_cast(bf16x8_t, make_uint4(rest2(sc[0][0], sc[0][1], h.x), rest2(sc[0][2], sc[0][3], h.y), rest2(sc[1][0], sc[1][1], h.z),
                                                   rest2(sc[1][2], sc[1][3], h.w)));
    }
    if (!SIG && __builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {   // wave-uniform
      asm volatile("" : "+v"(alpha));                                // (not multiplied ahead of the condition)
#pragma unroll
      for (int db = 0; db < NV; ++db)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[db][e] *= alpha;
    }
#pragma unroll
    for (int db = 0; db < NV; ++db) {
      const char* at = ks + vat + 16 * ((2 * db + vpc) ^ vsw);   // (rows r and r + 16 are exchanged alike)
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)at);
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at + 256 * KCH));
      const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, o[db], 0, 0, 0);
      if constexpr (FINE) o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl, o[db], 0, 0, 0);
    }
  }
  // results through LDS (tiles and table are done with), so that whole rows are written 16 bytes a lane
  __syncthreads();
  l = xor16_sum(xor32_sum(l));
  if constexpr (FINE) l *= OVER;
  const float inv = SIG ? (FINE ? 1.0f / OVER : 1.0f) : (l > 0.f ? 1.0f / l : 0.f);
  char* os = smem_raw + wave * 16 * Z::OP;
#pragma unroll
  for (int db = 0; db < NV; ++db)
    *reinterpret_cast<uint2*>(os + li * Z::OP + 32 * db + 8 * lg) = make_uint2(pack2(o[db][0] * inv, o[db][1] * inv), pack2(o[db][2] * inv, o[db][3] * inv));
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  constexpr int PR = DV / 8, RPI = 64 / PR;   // pieces of a row, rows of an instruction
#pragma unroll
  for (int u = 0; u < 16 / RPI; ++u) {
    const int row = RPI * u + lane / PR;
    const int64_t to = (int64_t)__shfl((int)orow, row, 64) * DV + 8 * (lane % PR);
    const uint4 w = *reinterpret_cast<const uint4*>(os + row * Z::OP + 16 * (lane % PR));
    if (wrow + row < nrows) *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(a.out) + to) = w;
  }
}


// The same with 32 rows per wave and 32x32x16 products, for steps of many rows: a fragment of keys or values that is read from LDS
// serves 32 rows, and a lane holds one row's scores of half the tile, so that maxima and sums cross lanes once. 4 waves take 128 rows,
// two workgroups share a CU. Key tiles of 64 (vdim 256: 32). Pieces of a row are exchanged (XOR) by the row's low bits, rotated: 16
// consecutive rows' reads of one piece, and the transposed reads of 4 rows by four neighbouring pieces, fall on all banks.
// Plain scores of a positive scale only (wide_takes). Bound by vector and matrix instructions of two waves per SIMD, which run in turns
// more than side by side (30 % and 42 % of the cycles): figures at wide_takes.
template <int NK, int NVB> struct WideTile {
  static constexpr int KT = NVB > 4 ? 32 : 64;                    // keys of a tile
  static constexpr int KCH = 4 * NK + 4 * NVB, NPF = KT * KCH / 256, BYTES = KT * KCH * 16;
  static constexpr int X = KCH % 16 == 0 && NVB <= 4 ? 16 : 8;    // pieces that change places
  static __device__ __forceinline__ int swz(int row) { 
    return X == 16 ? (row & 3) << 2 | (row >> 2 & 3) : KCH % 16 == 8 ? (row >> 1 & 1) << 2 | (row >> 2 & 3) : (row & 3) << 1 | (row >> 2 & 1);
  }
  static constexpr int TABLE = 1024;                              // key rows in LDS
  static constexpr int LDS = 2 * BYTES + 4 * TABLE;
};

template <int NK, int NVB, bool SIG>
__global__ void __launch_bounds__(256, 2) sink_attn_wide_kernel(SinkAttnArgs a) {
  using Z = WideTile<NK, NVB>;
  constexpr int KCH = Z::KCH, KT = Z::KT, NT = KT / 32, D = 32 * NK, DV = 32 * NVB, roww = D + DV;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];   // two tiles, key rows
  const int H = a.heads, G = a.kv_heads, QPG = H / G;
  int bx, s, g;
  tile_of(G, bx, s, g);
  const int lane = threadIdx.x & 63, tid = threadIdx.x, li = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q0 = a.cu_q ? a.cu_q[s] : s;
  const int nq = a.cu_q ? a.cu_q[s + 1] - q0 : 1;
  const int nrows = nq * QPG, row0 = bx * 128;
  if (row0 >= nrows) return;
  const int last_row = min(row0 + 128, nrows) - 1;
  const int p_first = (int)a.positions[q0 + row0 / QPG], p_last = (int)a.positions[q0 + last_row / QPG];
  const int jlo = first_key(a, p_first), jhi = min(p_last, a.ctx_lens[s] - 1);
  const int nt = jhi < jlo ? 0 : (jhi - jlo) / KT + 1;

  // cache rows of the workgroup's keys in LDS, TABLE keys at a time
  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
  int* rows = reinterpret_cast<int*>(smem_raw + 2 * Z::BYTES);
  const int bs_shift = __builtin_ctz(a.block_size);   // a power of two (mfma_ok)
  int jt = jlo;
  auto stage_rows = [&]() {
    for (int u = tid; u < Z::TABLE && jt + u <= jhi; u += 256)
      rows[u] = ((bt[(jt + u) >> bs_shift] * G + g) << bs_shift) + ((jt + u) & (a.block_size - 1));
    __syncthreads();
  };
  stage_rows();
  // piece u of this thread: 16 bytes of key krow[u] of the tile
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  int krow[Z::NPF], pcol[Z::NPF];
#pragma unroll
  for (int u = 0; u < Z::NPF; ++u) {
    const int idx = tid + 256 * u;
    krow[u] = idx / KCH;
    pcol[u] = 8 * ((idx % KCH) ^ Z::swz(krow[u]));
  }
  auto fetch = [&](int j0, int buf) {   // (keys beyond the last repeat it)
    if (min(j0 + KT - 1, jhi) - jt >= Z::TABLE) {
      __syncthreads();
      jt = j0;
      stage_rows();
    }
    const int at = j0 - jt, end = jhi - jt;
    int row[Z::NPF];
#pragma unroll
    for (int u = 0; u < Z::NPF; ++u) row[u] = rows[min(at + krow[u], end)];
    __builtin_amdgcn_sched_barrier(0);   // (all lookups, then the loads)
#pragma unroll
    for (int u = 0; u < Z::NPF; ++u) {
      char* to = smem_raw + buf * Z::BYTES + (256 * u + 64 * wave) * 16;
      __builtin_amdgcn_global_load_lds((global_cvoid*)(cache + ((uint64_t)(uint32_t)row[u] * roww + pcol[u])), (lds_void*)to, 16, 0, 0);
    }
  };
  if (nt > 0) fetch(jlo, 0);

  const int wrow = row0 + wave * 32, myrow = wrow + li;
  const bool rok = myrow < nrows, wave_live = wrow < nrows, wave_full = wrow + 31 < nrows;
  const int tq = q0 + (rok ? myrow / QPG : 0), myh = g * QPG + (rok ? myrow % QPG : 0);   // (rows beyond the last repeat the first)
  const int64_t orow = (int64_t)tq * H + myh;
  bf16x8_t qf[2 * NK];
#pragma unroll
  for (int k = 0; k < 2 * NK; ++k)
    qf[k] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(a.q) + orow * D + 16 * k + 8 * hi));
  const int prow = rok ? (int)a.positions[tq] : -1;
  const int jrow = first_key(a, max(prow, 0));
  const unsigned seen = rok ? max(min(prow, jhi) - jrow + 1, 0) : 0;   // this row sees keys jrow .. jrow + seen - 1
  // a tile is interior for a wave when every one of its (key, row) pairs is visible: no masking then
  const int pw_first = wave_live ? (int)a.positions[q0 + wrow / QPG] : 0;
  const int pw_last = wave_live ? (int)a.positions[q0 + min(wrow + 31, nrows - 1) / QPG] : 0;
  const int jw_first = first_key(a, pw_first), jw_last = first_key(a, pw_last);
  constexpr float LOG2E = 1.4426950408889634f;
  const float sl2 = a.scale * LOG2E;
  const float hb2 = SIG && a.head_bias != nullptr ? a.head_bias[myh] * LOG2E : 0.f;
  const bool has_sink = !SIG && a.sink != nullptr && rok;
  float m = has_sink ? a.sink[myh] * LOG2E : -1e30f;
  float l = has_sink && hi == 0 ? 1.0f : 0.0f;   // (the sum of this lane's keys)
  f32x16_t o[NVB];
#pragma unroll
  for (int db = 0; db < NVB; ++db) o[db] = f32x16_t{};
  // K fragments: key li of 32, piece 2 k + hi; V fragments: keys 4 hi .. and 8 + 4 hi .. of 16 (the order in which the weights lie
  // in registers), columns 32 db ..
  const int ksw = Z::swz(li), vrow = 4 * hi + (lane & 15) / 4, vsw = Z::swz(vrow), vsw8 = Z::swz(vrow + 8);
  const int kat = 16 * li * KCH, vat = 16 * vrow * KCH + 8 * (lane & 1), vpc = 4 * NK + 2 * (lane >> 4 & 1) + (lane >> 1 & 1);
  __builtin_amdgcn_s_waitcnt(15 << 8 | 7 << 4);
  for (int i = 0; i < nt; ++i) {
    const int j0 = jlo + i * KT;
    // tile i is in LDS for every wave, and every wave has left the other buffer
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(7 << 4);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (i + 1 < nt) fetch(j0 + KT, (i + 1) & 1);
    if (!wave_live || j0 > pw_last || j0 + KT <= jw_first) continue;   // nothing of this tile is visible to the wave
    const char* ks = smem_raw + (i & 1) * Z::BYTES;
    f32x16_t sc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) sc[t] = f32x16_t{};
    // fragments of NT x KG products ahead
    constexpr int KG = 2, NG = 2 * NK / KG;
    bf16x8_t kf[2][KG][NT];
    auto read_k = [&](int gk) {
#pragma unroll
      for (int k = 0; k < KG; ++k)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          kf[gk & 1][k][t] = __builtin_bit_cast(
              bf16x8_t, *reinterpret_cast<const uint4*>(ks + kat + 512 * KCH * t + 16 * ((2 * (KG * gk + k) + hi) ^ ksw)));
    };
    read_k(0);
#pragma unroll
    for (int gk = 0; gk < NG; ++gk) {
      if (gk + 1 < NG) read_k(gk + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < KG; ++k)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          sc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[gk & 1][k][t], qf[KG * gk + k], sc[t], 0, 0, 0);
    }
    // score e of block t: key j0 + 32 t + 8 (e / 4) + 4 hi + e % 4
    const bool interior = wave_full && j0 + KT - 1 <= min(pw_first, jhi) && j0 >= jw_last;
    if (!interior) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          sc[t][e] = (unsigned)(j0 + 32 * t + 8 * (e / 4) + 4 * hi + e % 4 - jrow) < seen ? sc[t][e] : -INFINITY;
    }
    if constexpr (SIG) {   // 1 / (1 + 2^-(v + bias)); a masked score is -inf and weighs 0
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[t][e] = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(fmaf(-sc[t][e], sl2, -hb2)));
    } else {
      float mx = sc[0][0];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sc[t][e]);
      mx = xor32_max(mx * sl2);
      const float mn = mx > m + LAZY ? mx : m;
      if (__builtin_amdgcn_ballot_w64(mn != m) != 0) {   // wave-uniform
        const float alpha = __builtin_amdgcn_exp2f(m - mn);
        l *= alpha;
#pragma unroll
        for (int db = 0; db < NVB; ++db)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[db][e] *= alpha;
        m = mn;
      }
      float sum[2] = {};
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          sc[t][e] = __builtin_amdgcn_exp2f(fmaf(sc[t][e], sl2, -m));   // v_exp_f32: arguments are at most LAZY, or -inf
          sum[e & 1] += sc[t][e];
        }
      l += sum[0] + sum[1];
    }
#pragma unroll
    for (int u = 0; u < 2 * NT; ++u) {   // 16 keys each
      const f32x16_t& c = sc[u / 2];
      const int e = 8 * (u & 1);
      const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, make_uint4(pack2(c[e], c[e + 1]), pack2(c[e + 2], c[e + 3]), pack2(c[e + 4], c[e + 5]),
                                                                  pack2(c[e + 6], c[e + 7])));
#pragma unroll
      for (int db = 0; db < NVB; ++db) {
        const char* at = ks + vat + 256 * KCH * u;
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at + 16 * ((4 * db + vpc) ^ vsw)));
        const short4_t up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at + 128 * KCH + 16 * ((4 * db + vpc) ^ vsw8)));
        const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7));
        o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, o[db], 0, 0, 0);
      }
    }
  }
  // results: a row's columns 32 db + 8 q + 4 hi .. in the registers; lanes 32 apart exchange halves, so that each stores 8 columns
  l = xor32_sum(l);
  const float inv = SIG ? 1.0f : (l > 0.f ? 1.0f / l : 0.f);
  bf16_t* op = reinterpret_cast<bf16_t*>(a.out) + orow * DV + 8 * hi;
#pragma unroll
  for (int db = 0; db < NVB; ++db)
#pragma unroll
    for (int q = 0; q < 16; q += 8) {
      const auto x = __builtin_amdgcn_permlane32_swap(pack2(o[db][q] * inv, o[db][q + 1] * inv), pack2(o[db][q + 4] * inv, o[db][q + 5] * inv), false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(pack2(o[db][q + 2] * inv, o[db][q + 3] * inv), pack2(o[db][q + 6] * inv, o[db][q + 7] * inv), false, false);
      if (rok) *reinterpret_cast<uint4*>(op + 32 * db + 2 * q) = make_uint4(x[0], y[0], x[1], y[1]);
    }
}

// column c of an output row (token t, head h) after the optional turn and gate, from the row's raw columns o(c)
template <typename F>
__device__ __forceinline__ float gated_out(const SinkAttnArgs& a, int64_t t, int h, int c, F&& o) {
  float v = o(c);
  if (a.gate == nullptr) return v;
  if (a.out_inv_freq != nullptr) {
    const int half = a.vdim / 2, i = c < half ? c : c - half;
    float sn, cs;
    sincosf((float)a.positions[t] * a.out_inv_freq[i], &sn, &cs);
    v = c < half ? v * cs + o(c + half) * sn : v * cs - o(c - half) * sn;
  }
  return v * a.gate_mult / (1.0f + expf(-bf2f(reinterpret_cast<const bf16_t*>(a.gate)[t * a.gstride + h])));
}

// ---------------------------------------------------------------------------------------------------
// Decode steps (one query token per sequence) in bf16, dim % 8 == 0 <= 256, vdim % 8 == 0 <= 256, at most 8 query
// heads per key/value head. A workgroup of 4 waves owns one (sequence, key/value head, split of the keys); a wave walks its keys
// 16 KT at a time on its own (no barrier until the end) and always has the next keys' and values' loads in flight:
//   scores   16x16x32 matrix products of 16 keys (rows, read straight into the operand: 4 lanes share a key) and the query
//            heads (columns), fp32; lane (head, 4 keys) turns them into weights: running maximum over the head's 4 lanes,
//            running sum per lane (log2 units, the sink seeds split 0); with SIG sigmoids
//   values   VL lanes share a value row; weights come back through LDS as fp32; each thread keeps R x 8 output columns of its
//            64 / VL keys of a pass
// The waves' sums meet in LDS, rescaled to one maximum. Bound by the loads in flight: 16 KB per wave, 3 waves per SIMD where 168
// registers hold them (values are read after the keys' products free registers). Keys 128 at a time per workgroup, with barriers
// between scores, softmax and values and shuffles for every sum, took 62 us of 73 (1.6 TB/s) where this takes 24 of 33: 32 sequences
// of about 1500 keys, 16 heads in 4 groups, dim = vdim = 128 (4.1 TB/s; in 16 splits of 128 keys, one trip each, 28 of 39); 64 sequences with 32
// heads 194 -> 91.
// Splits write unnormalised sums + (max, sum) to the workspace and
// sink_attn_merge_kernel combines them.
template <int R, int NKC, int VL, int KT, bool SIG>
__global__ void __launch_bounds__(256, R < 8 && R * NKC * VL < 512 && NKC * VL < 256 ? 3 : 2) sink_attn_decode_kernel(SinkAttnArgs a, float* ws_o, float* ws_ml, int nsplit) {
  constexpr int KPT = 16 * KT, NV = 64 / VL, NPV = KPT / NV, WK = KPT + 1;
  extern __shared__ __attribute__((aligned(16))) float dsm[];
  const int z = blockIdx.x, s = blockIdx.y, g = blockIdx.z, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* pw = dsm + wave * WK * R;       // [KPT][R] weights of the wave's keys, then the rescale of its sums
  float* ml = dsm + 4 * WK * R;          // [4][R][2]: maximum, sum of every wave
  float* red = ml + 8 * R;               // [4][R][DV]
  const int H = a.heads, G = a.kv_heads, QPG = H / G, D = a.dim, DV = a.vdim, roww = D + DV;
  const int p = (int)a.positions[s];
  const int ctx = a.ctx_lens[s];
  // wave w of all splits takes trips w, w + waves, ..: each has its share of the keys that are there, however many the table has room for
  const int jlo = first_key(a, p), jhi = min(p, ctx - 1), step = 4 * KPT * nsplit;
  const int64_t wrows = (int64_t)a.total_q * H;
  if (jlo + 4 * KPT * z > jhi && nsplit > 1) {   // an empty split: it only reports that it holds nothing
    if (tid < QPG) {
      const int64_t orow = (int64_t)s * H + g * QPG + tid;
      ws_ml[((int64_t)z * wrows + orow) * 2] = -1e30f;
      ws_ml[((int64_t)z * wrows + orow) * 2 + 1] = 0.f;
    }
    return;
  }
  constexpr float LOG2E = 1.4426950408889634f;
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
  const int li = lane & 15, lg = lane >> 4;    // scores: my query head (keys: my row), my 4 keys (my 8 dims) of 16 (32)
  const int vl = lane % VL, vg = lane / VL;    // values: my 8 columns, my key of NV
  const int bs_shift = (a.block_size & (a.block_size - 1)) == 0 ? __builtin_ctz(a.block_size) : -1;
  // Every load is unconditional, so that all of them are in flight together: keys beyond the last repeat it (their weights are
  // zero), lanes beyond a row's width repeat its start (the query is zero there, the output columns are not used)
  int64_t rows[KT];    // cache row of key li of each 16 (narrow rows: a cache of 2^32 of them fits the memory)
  int blk[KT];         // its block, asked for a trip ahead
  auto block_of = [&](int j) { return bs_shift >= 0 ? j >> bs_shift : j / a.block_size; };
  auto ask = [&](int j0) {
#pragma unroll
    for (int t = 0; t < KT; ++t) blk[t] = bt[block_of(min(j0 + 16 * t + li, jhi))];
  };
  auto find = [&](int j0) {
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      const int j = min(j0 + 16 * t + li, jhi);
      rows[t] = ((int64_t)blk[t] * G + g) * a.block_size + (j - block_of(j) * a.block_size);
    }
  };
  bf16x8_t kq[KT][NKC];
  uint4 vq[NPV];
  auto load_keys = [&]() {
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      const bf16_t* row = cache + rows[t] * roww;
#pragma unroll
      for (int c = 0; c < NKC; ++c) {
        const int d = 32 * c + 8 * lg;
        kq[t][c] = *reinterpret_cast<const bf16x8_t*>(row + (d < D ? d : 0));
      }
    }
  };
  auto load_values = [&]() {
#pragma unroll
    for (int u = 0; u < NPV; ++u) {
      const int64_t row = __shfl((long long)rows[u * NV / 16], u * NV % 16 + vg, 64);
      vq[u] = *reinterpret_cast<const uint4*>(cache + row * roww + D + (8 * vl < DV ? 8 * vl : 0));
    }
  };
  int j0 = jlo + KPT * (4 * z + wave);
  if (j0 <= jhi) {
    ask(j0);
    find(j0);
    load_keys();
    load_values();
    ask(j0 + step);
  }
  bf16x8_t qf[NKC];
  const bool mine = li < QPG;
  const int h = g * QPG + (mine ? li : 0);
#pragma unroll
  for (int c = 0; c < NKC; ++c) {
    const int d = 32 * c + 8 * lg;
    const uint4 w = *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(a.q) + ((int64_t)s * H + h) * D + (d < D ? d : 0));
    qf[c] = __builtin_bit_cast(bf16x8_t, mine && d < D ? w : make_uint4(0, 0, 0, 0));
  }
  const float slope = a.slopes != nullptr ? a.slopes[h] * LOG2E : 0.f;
  const float hb = SIG && a.head_bias != nullptr ? a.head_bias[h] * LOG2E : 0.f;
  const bool has_sink = !SIG && a.sink != nullptr && z == 0 && wave == 0;
  float m = SIG ? 0.f : has_sink ? a.sink[h] * LOG2E : -1e30f, l = SIG || (has_sink && lg == 0) ? 1.0f : 0.0f;
  float acc[R][8];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[r][e] = 0.f;
  const float qk_scale = a.softcap > 0.f ? a.scale / a.softcap : a.scale * LOG2E;

  for (; j0 <= jhi; j0 += step) {
    f32x4_t d[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      d[t] = f32x4_t{};
#pragma unroll
      for (int c = 0; c < NKC; ++c) d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kq[t][c], qf[c], d[t], 0, 0, 0);
    }
    const bool more = j0 + step <= jhi;
    if (more) {
      find(j0 + step);
      load_keys();
      ask(j0 + 2 * step);
    }
    float top = -INFINITY;
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = j0 + 16 * t + 4 * lg + e, n = p - j;
        float x = d[t][e] * qk_scale;
        if (a.softcap > 0.f) x = a.softcap * LOG2E * fast_tanh(x);
        if (a.slopes != nullptr) x -= slope * (float)n;
        if (a.bias != nullptr) x += a.bias[(int64_t)min(max(n, 0), a.bias_rows - 1) * H + h] * LOG2E;
        if constexpr (SIG) {
          x += hb;
          x = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x));
          d[t][e] = j <= jhi ? x : 0.f;
        } else {
          x = j <= jhi ? x : -INFINITY;
          top = fmaxf(top, x);
          d[t][e] = x;
        }
      }
    if constexpr (!SIG) {
      const float mn = fmaxf(m, xor16_max(xor32_max(top)));
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      l *= alpha;
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          d[t][e] = __builtin_amdgcn_exp2f(d[t][e] - mn);
          l += d[t][e];
        }
      if (lane < R) pw[KPT * R + lane] = alpha;
      m = mn;
    }
    if (li < R) {
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) pw[(16 * t + 4 * lg + e) * R + li] = d[t][e];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if constexpr (!SIG) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float alpha = pw[KPT * R + r];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r][e] *= alpha;
      }
    }
#pragma unroll
    for (int u = 0; u < NPV; ++u) {
      float f[8];
      unpack8(vq[u], f);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float w = pw[(u * NV + vg) * R + r];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r][e] = fmaf(w, f[e], acc[r][e]);
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(acc[r][e]));   // (summed before the next values' loads need registers)
    if (more) load_values();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the weights are read before the next ones replace them
    __builtin_amdgcn_wave_barrier();
  }
  // one maximum for the waves, then the sum of their and their key groups' results
  if constexpr (!SIG) {
    l = xor16_sum(xor32_sum(l));
    if (lane < R) {
      ml[(wave * R + lane) * 2] = m;
      ml[(wave * R + lane) * 2 + 1] = l;
    }
    __syncthreads();
  }
  float mt[R], lt[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    mt[r] = 0.f;
    lt[r] = 1.0f;
    float f = 1.0f;
    if constexpr (!SIG) {
      mt[r] = fmaxf(fmaxf(ml[r * 2], ml[(R + r) * 2]), fmaxf(ml[(2 * R + r) * 2], ml[(3 * R + r) * 2]));
      lt[r] = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) lt[r] += ml[(w * R + r) * 2 + 1] * __builtin_amdgcn_exp2f(ml[(w * R + r) * 2] - mt[r]);
      f = __builtin_amdgcn_exp2f(ml[(wave * R + r) * 2] - mt[r]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float x = xor32_sum(acc[r][e] * f);
      if constexpr (VL == 16) x = xor16_sum(x);
      acc[r][e] = x;
    }
    if (vg == 0 && 8 * vl < DV) {
      float* dst = red + (wave * R + r) * DV + 8 * vl;
      *reinterpret_cast<float4*>(dst) = make_float4(acc[r][0], acc[r][1], acc[r][2], acc[r][3]);
      *reinterpret_cast<float4*>(dst + 4) = make_float4(acc[r][4], acc[r][5], acc[r][6], acc[r][7]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= QPG) break;
    const int64_t orow = (int64_t)s * H + g * QPG + r;
    const int c = tid;
    if (c >= DV) break;
    auto column = [&](int col) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) v += red[(w * R + r) * DV + col];
      return v;
    };
    if (nsplit > 1) {
      ws_o[((int64_t)z * wrows + orow) * DV + c] = column(c);
      if (c == 0) {
        ws_ml[((int64_t)z * wrows + orow) * 2] = mt[r];
        ws_ml[((int64_t)z * wrows + orow) * 2 + 1] = lt[r];
      }
    } else {
      const float inv = lt[r] > 0.f ? 1.0f / lt[r] : 0.f;
      reinterpret_cast<bf16_t*>(a.out)[(int64_t)s * a.ostride + (g * QPG + r) * DV + c] =
          f2bf(gated_out(a, s, g * QPG + r, c, [&](int col) { return column(col) * inv; }));
    }
  }
}

// out[row] = sum_z O_z 2^(m_z - m*) / sum_z l_z 2^(m_z - m*), m* = max_z m_z (running maxima in log2 units; sigmoid
// weights: the plain sum of the splits that hold keys, l_z > 0), then the optional turn and gate. One workgroup per
// (token, head).
__global__ void __launch_bounds__(128) sink_attn_merge_kernel(SinkAttnArgs a) {
  __shared__ float wz[128];   // a split's weight 2^(m_z - m*) / sum (nsplit <= 128)
  __shared__ int id[128], count[2];
  __shared__ float orow[256];
  const int64_t row = blockIdx.x, rows = (int64_t)a.heads * a.total_q;
  const int64_t t = row / a.heads;
  const int h = (int)(row - t * a.heads), DV = a.vdim, nsplit = a.nsplit;
  const int z = threadIdx.x;
  const float mz = z < nsplit ? a.ws_ml[((int64_t)z * rows + row) * 2] : -1e30f;
  const float lz = z < nsplit ? a.ws_ml[((int64_t)z * rows + row) * 2 + 1] : 0.f;
  float mstar = wave_max(mz);
  __shared__ float red2[4];
  if ((threadIdx.x & 63) == 0) red2[threadIdx.x >> 6] = mstar;
  __syncthreads();
  mstar = fmaxf(red2[0], red2[1]);
  const float w = lz > 0.f ? exp2f(mz - mstar) : 0.f;
  float lsum = wave_sum(lz * w);
  const bool holds = a.sigmoid ? lz > 0.f : w != 0.f;
  const unsigned long long in = __ballot(holds);
  if ((threadIdx.x & 63) == 0) {
    red2[2 + (threadIdx.x >> 6)] = lsum;
    count[threadIdx.x >> 6] = __popcll(in);
  }
  __syncthreads();
  lsum = red2[2] + red2[3];
  // the splits that hold keys, in order
  const int n = a.sigmoid || lsum > 0.f ? count[0] + count[1] : 0;
  if (holds) {
    const int at = (z < 64 ? 0 : count[0]) + __popcll(in & ((1ull << (z & 63)) - 1));
    wz[at] = a.sigmoid ? 1.0f : w / lsum;
    id[at] = z;
  }
  __syncthreads();
  for (int c = threadIdx.x; c < DV; c += 128) {
    float acc = 0.f;
    int k0 = 0;
    auto add = [&](auto count) {   // loads in flight together: 7.6 -> 4.4 us for 16 splits of 512 rows
      constexpr int N = decltype(count)::value;
      float x[N];
#pragma unroll
      for (int k = 0; k < N; ++k) x[k] = a.ws_o[((int64_t)id[k0 + k] * rows + row) * DV + c];
#pragma unroll
      for (int k = 0; k < N; ++k) acc += x[k] * wz[k0 + k];
      k0 += N;
    };
    while (k0 + 8 <= n) add(IntC<8>{});
    if (n & 4) add(IntC<4>{});
    if (n & 2) add(IntC<2>{});
    if (n & 1) add(IntC<1>{});
    orow[c] = acc;
  }
  if (a.out_inv_freq != nullptr) __syncthreads();   // (else every thread reads its own columns)
  bf16_t* out = reinterpret_cast<bf16_t*>(a.out) + t * a.ostride + h * DV;
  for (int c = threadIdx.x; c < DV; c += 128) out[c] = f2bf(gated_out(a, t, h, c, [&](int col) { return orow[col]; }));
}

template <int NDB, int NW, int NKC, bool SIG> hipError_t launch_mfma(const SinkAttnArgs& a, hipStream_t s) {
  auto* fn = sink_attn_mfma_kernel<NDB, NW, NKC, SIG, false>;
  if constexpr (!SIG && NW == 4 && NKC <= 16 && (NDB == 2 || NDB == 4 || NDB == 8))
    if (a.fine) fn = sink_attn_mfma_kernel<NDB, NW, NKC, SIG, true>;
  const int kp = a.dim + 32 * NDB + 8, qp = a.dim + 8;
  const int qpg0 = a.heads / a.kv_heads;
  const int qr = q_in_regs<NDB, NW, NKC>() ? 0 : (NW == 1 ? min(32, a.max_q * qpg0 + 1) : 32 * NW);
  const int nsp = a.ws_o != nullptr ? max(1, a.nsplit) : 1;
  // block-table entries staged per workgroup: its key range's (else they are read from global memory)
  const int btc = min(BT_LDS_MAX, (nsp > 1 ? a.chunk / a.block_size + 2 : a.bt_stride) + 1);
  const size_t lds = sizeof(bf16_t) * ((size_t)qr * qp + (size_t)(2 * stage_keys<NW, NKC>() + 1) * kp) + sizeof(int) * btc;
  if (lds > 150 * 1024) return hipErrorInvalidValue;
  if (lds > 48 * 1024) {  // only then: the limit is raised per function, and a raised limit is not free
    static size_t raised[2] = {};
    size_t& own = raised[fn != sink_attn_mfma_kernel<NDB, NW, NKC, SIG, false>];
    if (lds > own) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)lds);
      if (e != hipSuccess) return e;
      own = lds;
    }
  }
  const int qpg = a.heads / a.kv_heads;
  const int nsplit = a.ws_o != nullptr ? max(1, a.nsplit) : 1;
  const dim3 grid((unsigned)(((int64_t)a.max_q * qpg + 32 * NW - 1) / (32 * NW)), (unsigned)a.num_seqs,
                  (unsigned)(a.kv_heads * nsplit));
  hipLaunchKernelGGL(fn, grid, dim3(64 * NW), lds, s, a, kp, qp, qr, btc, a.ws_o, a.ws_ml, nsplit, a.chunk);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || nsplit <= 1) return e;
  hipLaunchKernelGGL(sink_attn_merge_kernel, dim3((unsigned)((int64_t)a.heads * a.total_q)), dim3(128), 0, s, a);
  return hipGetLastError();
}

template <int NW, int NKC, bool SIG> hipError_t launch_mfma_ndb(const SinkAttnArgs& a, hipStream_t s) {
  switch ((a.vdim + 31) / 32) {
    case 1: return launch_mfma<1, NW, NKC, SIG>(a, s);
    case 2: return launch_mfma<2, NW, NKC, SIG>(a, s);
    case 3: return launch_mfma<3, NW, NKC, SIG>(a, s);
    case 4: return launch_mfma<4, NW, NKC, SIG>(a, s);
  }
  if constexpr (NKC >= 16) {
    switch ((a.vdim + 31) / 32) {
      case 5: return launch_mfma<5, NW, NKC, SIG>(a, s);
      case 6: return launch_mfma<6, NW, NKC, SIG>(a, s);
      case 7: return launch_mfma<7, NW, NKC, SIG>(a, s);
      case 8: return launch_mfma<8, NW, NKC, SIG>(a, s);
    }
  }
  return hipErrorInvalidValue;
}

template <int NW, bool SIG> hipError_t launch_mfma_sig(const SinkAttnArgs& a, hipStream_t s) {
  if (a.dim <= 64 && a.vdim <= 128) return launch_mfma_ndb<NW, 8, SIG>(a, s);
  return a.dim <= 128 ? launch_mfma_ndb<NW, 16, SIG>(a, s) : launch_mfma_ndb<NW, 32, SIG>(a, s);
}
template <int NW> hipError_t launch_mfma_nw(const SinkAttnArgs& a, hipStream_t s) {
  return a.sigmoid ? launch_mfma_sig<NW, true>(a, s) : launch_mfma_sig<NW, false>(a, s);
}

template <int R, int NKC, int VL, bool SIG> hipError_t launch_decode_one(const SinkAttnArgs& a, hipStream_t s) {
  constexpr int KT = NKC <= 4 && VL == 16 ? 2 : 1;   // (wider rows: half the keys, to hold as many bytes)
  auto* fn = sink_attn_decode_kernel<R, NKC, VL, KT, SIG>;
  const size_t lds = sizeof(float) * ((size_t)4 * (16 * KT + 1) * R + 8 * R + (size_t)4 * R * a.vdim);   // at most 37 KB
  const int nsplit = a.ws_o != nullptr ? max(1, a.nsplit) : 1;
  hipLaunchKernelGGL(fn, dim3(nsplit, a.num_seqs, a.kv_heads), dim3(256), lds, s, a, a.ws_o, a.ws_ml, nsplit);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || nsplit <= 1) return e;
  hipLaunchKernelGGL(sink_attn_merge_kernel, dim3((unsigned)((int64_t)a.heads * a.total_q)), dim3(128), 0, s, a);
  return hipGetLastError();
}

template <int NKC, int VL, bool SIG> hipError_t launch_decode_sig(const SinkAttnArgs& a, hipStream_t s) {
  const int qpg = a.heads / a.kv_heads;
  if (qpg <= 1) return launch_decode_one<1, NKC, VL, SIG>(a, s);
  if (qpg <= 2) return launch_decode_one<2, NKC, VL, SIG>(a, s);
  if (qpg <= 4) return launch_decode_one<4, NKC, VL, SIG>(a, s);
  return launch_decode_one<8, NKC, VL, SIG>(a, s);
}
template <int NKC, int VL> hipError_t launch_decode_r(const SinkAttnArgs& a, hipStream_t s) {
  return a.sigmoid ? launch_decode_sig<NKC, VL, true>(a, s) : launch_decode_sig<NKC, VL, false>(a, s);
}

template <int NKC> hipError_t launch_decode_v(const SinkAttnArgs& a, hipStream_t s) {
  return a.vdim <= 128 ? launch_decode_r<NKC, 16>(a, s) : launch_decode_r<NKC, 32>(a, s);
}

// cached keys of a sequence that a step can see
inline int64_t keys_of(const SinkAttnArgs& a) {
  int64_t keys = (int64_t)a.bt_cols * a.block_size;
  if (a.window > 0) keys = std::min<int64_t>(keys, (int64_t)a.window + a.max_q);
  return a.seg > 0 ? std::min<int64_t>(keys, (int64_t)a.seg + a.max_q) : keys;
}
// FINE: the weights enter the products in two bf16 parts, for steps of up to four row tiles of 128 per CU over more than one of 64 keys. The
// kernel with split keys, which ran them before, rounds relative to every split's own largest weight, which is then exact: whole
// keys with rounded weights are up to 6 % further from 64 bits (5 x 77 rows behind 300: 2.18e-3, whole 2.31e-3, in two parts 1.66e-3).
inline int64_t wide_tiles(const SinkAttnArgs& a) { return ((int64_t)a.max_q * (a.heads / a.kv_heads) + 127) / 128 * a.num_seqs * a.kv_heads; }
inline bool fine_takes(const SinkAttnArgs& a) { return wide_tiles(a) <= 4 * (int64_t)num_cus() && keys_of(a) > 64; }
template <int NK, int NV> hipError_t launch_rows(const SinkAttnArgs& a, hipStream_t s) {
  const int64_t rows = (int64_t)a.max_q * (a.heads / a.kv_heads);
  const bool fine = fine_takes(a);
  const dim3 grid((unsigned)((rows + 63) / 64), (unsigned)a.num_seqs, (unsigned)a.kv_heads);
  auto* fn = a.sigmoid ? (fine ? sink_attn_rows_kernel<NK, NV, true, true> : sink_attn_rows_kernel<NK, NV, true, false>)
                       : (fine ? sink_attn_rows_kernel<NK, NV, false, true> : sink_attn_rows_kernel<NK, NV, false, false>);
  hipLaunchKernelGGL(fn, grid, dim3(256), (RowTile<NK, NV>::LDS), s, a);
  return hipGetLastError();
}
template <int NK, int NVB> hipError_t launch_wide(const SinkAttnArgs& a, hipStream_t s) {
  using Z = WideTile<NK, NVB>;
  const int64_t rows = (int64_t)a.max_q * (a.heads / a.kv_heads);
  const dim3 grid((unsigned)((rows + 127) / 128), (unsigned)a.num_seqs, (unsigned)a.kv_heads);
  auto* fn = a.sigmoid ? sink_attn_wide_kernel<NK, NVB, true> : sink_attn_wide_kernel<NK, NVB, false>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, Z::LDS);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, grid, dim3(256), Z::LDS, s, a);
  return hipGetLastError();
}
template <int NK> hipError_t launch_wide_v(const SinkAttnArgs& a, hipStream_t s) {
  if (a.vdim == 64) return launch_wide<NK, 2>(a, s);
  return a.vdim == 128 ? launch_wide<NK, 4>(a, s) : launch_wide<NK, 8>(a, s);
}
template <int NK> hipError_t launch_rows_v(const SinkAttnArgs& a, hipStream_t s) {
  if (a.vdim == 64) return launch_rows<NK, 4>(a, s);
  return a.vdim == 128 ? launch_rows<NK, 8>(a, s) : launch_rows<NK, 16>(a, s);
}
// prompt-sized steps at the widths of sink_attn_rows_kernel
inline bool rows_fits(const SinkAttnArgs& a) {
  return a.max_q * (a.heads / a.kv_heads) > 32 && (a.dim == 64 || a.dim == 128) && (a.vdim == 64 || a.vdim == 128 || a.vdim == 256) &&
         (int64_t)a.total_q * a.heads < (1ll << 31);
}
// and keys not split
inline bool rows_takes(const SinkAttnArgs& a) { return (a.ws_o == nullptr || a.nsplit <= 1) && rows_fits(a); }

// Of these, those that go 128 rows per workgroup: more than four tiles per CU and long keys (a workgroup's start is the same for 64 rows). Fewer tiles
// keep 64 rows also where 128 are faster: their keys were split before, and their weights go in two bf16 parts (fine_takes), which the wide
// kernel has no registers for. Scores with caps, slopes or a bias are bound by vector instructions, of which four waves per SIMD
// issue more than two. 64 / 128 rows, us: 16 x 1000 behind 300, 16 heads 132 / 110, vdim 256 187 / 160, window of 512 89 / 80; 4 x 1000 of 32
// heads (4 tiles per CU) 57 / 54; 2 x 1000 37 / 38; 16 x 250 23.0 / 24.3; capped 16 x 500 of 32 heads 121 / 135.
inline bool wide_takes(const SinkAttnArgs& a) {
  return a.softcap <= 0.f && a.slopes == nullptr && a.bias == nullptr && a.scale > 0.f && wide_tiles(a) > 4 * (int64_t)num_cus() && keys_of(a) >= 512;
}

inline bool decode_ok(const SinkAttnArgs& a) {
  return !a.f32 && a.cu_q == nullptr && a.max_q == 1 && a.heads / a.kv_heads <= 8 && a.dim % 8 == 0 && a.dim <= 256 &&
         a.vdim % 8 == 0 && a.vdim <= 256 && (reinterpret_cast<uintptr_t>(a.q) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(a.cache) & 15) == 0 && (a.nsplit <= 1 || a.nsplit <= 128);
}

inline bool mfma_ok(const SinkAttnArgs& a) {
  return !a.f32 && (a.block_size & (a.block_size - 1)) == 0 && a.dim % 16 == 0 && a.dim <= 256 && a.vdim % 8 == 0 && a.vdim <= 256 &&
         (reinterpret_cast<uintptr_t>(a.q) & 15) == 0 && (reinterpret_cast<uintptr_t>(a.cache) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(a.out) & 15) == 0 &&
         (int64_t)a.kv_heads * a.block_size * (a.dim + a.vdim) * 2 < (1ll << 32);
}

}  // namespace

bool sink_attn_uses_mfma(const SinkAttnArgs& a) { return a.impl != 1 && mfma_ok(a); }
bool sink_attn_fits_rows(const SinkAttnArgs& a) { return sink_attn_uses_mfma(a) && rows_fits(a); }
bool sink_attn_uses_decode(const SinkAttnArgs& a) { return a.impl == 0 && decode_ok(a); }
bool sink_attn_fuses_gate(const SinkAttnArgs& a) {
  return sink_attn_uses_decode(a) || (sink_attn_uses_mfma(a) && a.ws_o != nullptr && a.nsplit > 1);
}

const char* sink_attn_form(const SinkAttnArgs& a) {
  if (sink_attn_uses_decode(a)) return "decode";
  if (!sink_attn_uses_mfma(a)) return "fma";
  return rows_takes(a) ? "rows" : a.ws_o != nullptr && a.nsplit > 1 ? "split" : "tiles";
}

const char* sink_attn_kernel(const SinkAttnArgs& a) {
  if (sink_attn_uses_decode(a) || !sink_attn_uses_mfma(a)) return sink_attn_form(a);
  if (rows_takes(a)) return wide_takes(a) ? "wide" : fine_takes(a) ? "fine rows" : "rows";
  return a.ws_o != nullptr && a.nsplit > 1 && a.fine && !a.sigmoid ? "fine split" : sink_attn_form(a);
}

hipError_t launch_sink_attn(const SinkAttnArgs& a, hipStream_t s) {
  if (a.num_seqs == 0 || a.total_q == 0) return hipSuccess;
  if (a.heads < 1 || a.kv_heads < 1 || a.heads % a.kv_heads != 0 || a.dim < 1 || a.dim > 512 || a.vdim < 1 ||
      a.vdim > 256 || a.block_size < 1 || a.max_q < 1 || a.window < 0 || a.seg < 0 || (a.gate != nullptr && !sink_attn_fuses_gate(a)) ||
      (a.out_inv_freq != nullptr && (a.vdim & 1)) || (a.bias != nullptr && a.bias_rows < 1) ||
      (a.sigmoid ? a.sink != nullptr : a.head_bias != nullptr))
    return hipErrorInvalidValue;
  if (sink_attn_uses_decode(a)) {
    if (a.dim <= 64) return launch_decode_v<2>(a, s);
    return a.dim <= 128 ? launch_decode_v<4>(a, s) : launch_decode_v<8>(a, s);
  }
  if (sink_attn_uses_mfma(a)) {
    const int qpg = a.heads / a.kv_heads;
    if (rows_takes(a) && wide_takes(a)) return a.dim == 64 ? launch_wide_v<2>(a, s) : launch_wide_v<4>(a, s);
    if (rows_takes(a)) return a.dim == 64 ? launch_rows_v<2>(a, s) : launch_rows_v<4>(a, s);
    return a.max_q * qpg <= 32 ? launch_mfma_nw<1>(a, s) : launch_mfma_nw<4>(a, s);
  }
  if (a.impl == 2) return hipErrorInvalidValue;
  return a.f32 ? launch_fma<true>(a, s) : launch_fma<false>(a, s);
}

}  // namespace die
