// Latent (compressed-KV) attention over the paged latent cache, in its absorbed form: every head's query
// is first projected into the latent space (q_lat = W_uk^T q_nope, a batched GEMM outside this file), so
// all heads of a token score against the SAME cached row [latent | rotated shared key part] and the output
// is the weighted sum of the latent rows (W_uv is applied afterwards). One kernel serves prompt chunks and
// single decode tokens: a row is a (token, head) pair, its keys are the cache positions j <= p inside the
// sliding window, and the softmax denominator may hold a per-head sink term exp(sink_h) attached to no position
// (running max starts at the sink, running sum at 1).
//
// Scores, softmax weights and the weighted sum are fp32 (FMA); storage of q / cache / out is bf16 or fp32.
// Workgroup = 4 waves x 4 rows. A tile of BK keys is staged once in LDS as fp32 (row stride odd: a lane per
// key reads conflict-free; a lane per column too) and shared by the 16 rows. Lanes split (key, part of the
// score dimension); the rotary part of q is rotated while it is loaded.
#include "common.h"
#include "mix_launchers.h"

namespace die {

namespace {

constexpr int RPW = 4, WAVES = 4, RW = RPW * WAVES;

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

template <int BK, int CC, bool F32>
__global__ void __launch_bounds__(256) latent_attn_kernel(LatentAttnArgs a, int QS, int KS) {
  extern __shared__ float smem[];
  float* qs = smem;                 // [RW][QS]
  float* ks = qs + RW * QS;         // [BK][KS]
  float* ps = ks + BK * KS;         // [WAVES][RPW][BK]
  const int s = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int H = a.heads, R = a.sh.rank, Dk = a.sh.rank + a.sh.rot_dim;
  const int q0 = a.cu_q ? a.cu_q[s] : s;
  const int nq = a.cu_q ? a.cu_q[s + 1] - q0 : 1;
  const int nrows = nq * H, row0 = blockIdx.x * RW;
  if (row0 >= nrows) return;
  const int ctx = a.ctx_lens[s];
  const int last_row = min(row0 + RW, nrows) - 1;
  const int p_first = (int)a.positions[q0 + row0 / H], p_last = (int)a.positions[q0 + last_row / H];
  const int jlo = a.window > 0 ? max(0, p_first - a.window + 1) : 0;
  const int jhi = min(p_last, ctx - 1);

  // queries -> LDS (fp32), the rotary part rotated by the row's position
  for (int r = wave; r < RW; r += WAVES) {
    const int row = row0 + r;
    const bool ok = row < nrows;
    const int tl = ok ? row / H : 0, h = ok ? row % H : 0;
    const int64_t t = q0 + tl;
    const float p = ok ? (float)a.positions[t] : 0.f;
    const int64_t ql = ((int64_t)h * a.total_q + t) * R;
    const int64_t qr = t * a.q_stride + (int64_t)h * a.q_hstride;
    for (int d = lane; d < QS; d += 64) {
      float v = 0.f;
      if (ok && d < R) {
        v = ldt<F32>(a.q_lat, ql + d);
      } else if (ok && d < Dk) {
        const int dd = d - R, i = dd >> 1;
        if (i < a.sh.rot_pairs) {
          const float u = ldt<F32>(a.q_rot, qr + 2 * i), w = ldt<F32>(a.q_rot, qr + 2 * i + 1);
          float sn, cs;
          sincosf(p * a.sh.inv_freq[i], &sn, &cs);
          v = (dd & 1) ? w * cs + u * sn : u * cs - w * sn;
        } else {
          v = ldt<F32>(a.q_rot, qr + dd);
        }
      }
      qs[r * QS + d] = v;
    }
  }

  int prow[RPW];
  bool rok[RPW];
  float m[RPW], l[RPW], o[RPW][CC];
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const int row = row0 + wave * RPW + i;
    rok[i] = row < nrows;
    prow[i] = rok[i] ? (int)a.positions[q0 + row / H] : -1;
    const bool has_sink = a.sink != nullptr && rok[i];
    m[i] = has_sink ? a.sink[row % H] : -1e30f;
    l[i] = has_sink ? 1.0f : 0.0f;
#pragma unroll
    for (int c = 0; c < CC; ++c) o[i][c] = 0.f;
  }

  constexpr int NP = 64 / BK;
  const int key = lane % BK, part = lane / BK;
  const int dlen = (Dk + NP - 1) / NP, d0 = part * dlen, d1 = min(Dk, d0 + dlen);
  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;

  for (int j0 = jlo; j0 <= jhi; j0 += BK) {
    __syncthreads();  // the previous tile (and, first, the queries) are no longer / now in LDS
    for (int k = wave; k < BK; k += WAVES) {
      const int j = j0 + k;
      const bool in = j <= jhi;
      const int64_t rowp = in ? ((int64_t)bt[j / a.block_size] * a.block_size + j % a.block_size) * Dk : 0;
      for (int d = lane; d < Dk; d += 64) ks[k * KS + d] = in ? ldt<F32>(a.cache, rowp + d) : 0.f;
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
      const bool valid = rok[i] && j <= jhi && j <= prow[i] && (a.window <= 0 || prow[i] - j < a.window);
      sc = valid ? sc * a.scale : -INFINITY;
      const float mn = fmaxf(m[i], wave_max(sc));
      const float pe = valid ? expf(sc - mn) : 0.f;
      const float psum = wave_sum(part == 0 ? pe : 0.f);
      alpha[i] = expf(m[i] - mn);
      l[i] = l[i] * alpha[i] + psum;
      m[i] = mn;
      if (part == 0) ps[(wave * RPW + i) * BK + key] = pe;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
#pragma unroll
      for (int c = 0; c < CC; ++c) o[i][c] *= alpha[i];
    }
    for (int k = 0; k < BK; ++k) {
      float kvc[CC];
#pragma unroll
      for (int c = 0; c < CC; ++c) kvc[c] = (lane + 64 * c < R) ? ks[k * KS + lane + 64 * c] : 0.f;
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
        const float pk = ps[(wave * RPW + i) * BK + k];
#pragma unroll
        for (int c = 0; c < CC; ++c) o[i][c] += pk * kvc[c];
      }
    }
  }

#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    if (!rok[i]) continue;
    const int row = row0 + wave * RPW + i;
    const int64_t t = q0 + row / H;
    const int h = row % H;
    const float inv = l[i] > 0.f ? 1.0f / l[i] : 0.f;
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      const int col = lane + 64 * c;
      if (col < R) stt<F32>(a.out, ((int64_t)h * a.total_q + t) * R + col, o[i][c] * inv);
    }
  }
}

// ---------------------------------------------------------------------------------------------------
// bf16 on the matrix cores (v_mfma_f32_32x32x16_bf16), for rank % 32 == 0, rank <= 256, rot_dim % 16 == 0,
// rot_dim <= 128. Workgroup = NW waves x 32 rows (NW = 1 for steps of few rows per sequence: decode). Per
// tile of 32 keys, staged once in LDS row-major ([key][Dk], the next tile's global loads in flight meanwhile):
//   S^T[key][q] = K Q^T        A = K rows from LDS, B = Q rows from LDS      (Dk / 16 MFMAs)
//   online softmax per query column (one lane pair owns a query: no cross-lane traffic beyond xor 32),
//   fp32 scores and weights, running max seeded with the sink; P is rounded to bf16 only as the MFMA operand
//   O^T[d][q] += V^T P^T      A = the latent columns of the same tile, read transposed (ds_read_tr16_b64),
//                              B = P^T straight from the score accumulator  (2 * rank / 32 MFMAs)
// Split keys (grid.z = nsplit > 1; decode over long contexts): split z takes keys [jlo + z * chunk, + chunk),
// writes its unnormalised O, running max and sum to a workspace, and latent_attn_merge_kernel combines them;
// the sink enters split 0 only.
constexpr int MKT = 32;
constexpr int BT_LDS_MAX = 2048;  // block-table entries staged per workgroup (else read from global memory)
typedef __attribute__((address_space(3))) short4_t lds_short4;
typedef __attribute__((ext_vector_type(8))) short short8_t;
// What the rounding of the weights x, y to b left. (Zero and negative as well: an infinite latent column makes its key's score infinite or NaN,
// and so its weight 0 or NaN, before any of it counts.)
__device__ __forceinline__ uint32_t rest2(float x, float y, uint32_t b) {
  return pack2(x - __uint_as_float(b << 16), y - __uint_as_float(b & 0xffff0000u));
}

// FINE: the weights enter the products in two bf16 parts (LatentAttnArgs::fine)
template <int NDB, int NW, bool FINE>
__global__ void __launch_bounds__(64 * NW) latent_attn_mfma_kernel(LatentAttnArgs a, int KP) {
  constexpr int ROWS = 32 * NW, NT = 64 * NW;
  constexpr int NPF = (MKT * (4 * NDB + 16) + NT - 1) / NT;  // 16-byte chunks of a key tile per thread (rot_dim <= 128)
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  bf16_t* qs = reinterpret_cast<bf16_t*>(smem_raw);          // [ROWS][KP]
  bf16_t* ks = qs + ROWS * KP;                                // [MKT][KP]
  // unsplit steps: XCD k (workgroups are dealt round-robin by linear id) takes a contiguous eighth of the
  // sequence-major tile list, so one sequence's cache rows stay in one L2
  int bx = blockIdx.x, by = blockIdx.y;
  if (gridDim.z == 1) {
    const unsigned total = gridDim.x * gridDim.y, lin = blockIdx.x + gridDim.x * blockIdx.y;
    if (total % 8 == 0) {
      const unsigned nl = (lin % 8) * (total / 8) + lin / 8;
      bx = (int)(nl % gridDim.x);
      by = (int)(nl / gridDim.x);
    }
  }
  const int s = by, z = blockIdx.z, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tid = threadIdx.x;
  const int H = a.heads, R = a.sh.rank, Dk = a.sh.rank + a.sh.rot_dim;
  const int q0 = a.cu_q ? a.cu_q[s] : s;
  const int nq = a.cu_q ? a.cu_q[s + 1] - q0 : 1;
  const int nrows = nq * H, row0 = bx * ROWS;
  if (row0 >= nrows) return;
  const int ctx = a.ctx_lens[s];
  const int last_row = min(row0 + ROWS, nrows) - 1;
  const int p_first = (int)a.positions[q0 + row0 / H], p_last = (int)a.positions[q0 + last_row / H];
  int jlo = a.window > 0 ? max(0, p_first - a.window + 1) : 0;
  int jhi = min(p_last, ctx - 1);
  if (a.nsplit > 1) {
    jlo += z * a.chunk;
    jhi = min(jhi, jlo + a.chunk - 1);
  }
  const bf16_t* qlat = reinterpret_cast<const bf16_t*>(a.q_lat);
  const bf16_t* qrot = reinterpret_cast<const bf16_t*>(a.q_rot);
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  const int qcol = lane & 31, hh = lane >> 5;
  const int myrow = row0 + wave * 32 + qcol;
  const bool rok = myrow < nrows;
  const int64_t orow = rok ? (int64_t)(myrow % H) * a.total_q + (q0 + myrow / H) : 0;
  if (jlo > jhi) {  // an empty split (uniform over the workgroup): it only reports that it holds nothing
    if (a.nsplit > 1 && rok && hh == 0) {
      a.ws_ml[((int64_t)z * a.heads * a.total_q + orow) * 2] = -1e30f;
      a.ws_ml[((int64_t)z * a.heads * a.total_q + orow) * 2 + 1] = 0.f;
    }
    return;
  }

  // queries -> LDS: the latent part as 16-byte copies, the rotary part rotated in fp32
  const int lch = R / 8;
  for (int idx = tid; idx < ROWS * lch; idx += NT) {
    const int r = idx / lch, c = idx % lch, row = row0 + r;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (row < nrows) {
      const int64_t t = q0 + row / H;
      v = *reinterpret_cast<const uint4*>(qlat + ((int64_t)(row % H) * a.total_q + t) * R + 8 * c);
    }
    *reinterpret_cast<uint4*>(qs + r * KP + 8 * c) = v;
  }
  // one thread per interleaved pair (an odd last element passes unchanged); bf16 operands: the fast sin / cos
  const int npair = (a.sh.rot_dim + 1) / 2;
  for (int idx = tid; idx < ROWS * npair; idx += NT) {
    const int r = idx / npair, i = idx % npair, row = row0 + r;
    const bool two = 2 * i + 1 < a.sh.rot_dim;
    float v0 = 0.f, v1 = 0.f;
    if (row < nrows) {
      const int64_t t = q0 + row / H;
      const int64_t qr = t * a.q_stride + (int64_t)(row % H) * a.q_hstride;
      const float u = bf2f(qrot[qr + 2 * i]), w = two ? bf2f(qrot[qr + 2 * i + 1]) : 0.f;
      v0 = u;
      v1 = w;
      if (i < a.sh.rot_pairs) {
        float sn, cs;
        __sincosf((float)a.positions[t] * a.sh.inv_freq[i], &sn, &cs);
        v0 = u * cs - w * sn;
        v1 = w * cs + u * sn;
      }
    }
    qs[r * KP + R + 2 * i] = f2bf(v0);
    if (two) qs[r * KP + R + 2 * i + 1] = f2bf(v1);
  }

  const bool wave_live = row0 + wave * 32 < nrows;
  const int prow = rok ? (int)a.positions[q0 + myrow / H] : -1;
  constexpr float LOG2E = 1.4426950408889634f;
  const float sl2 = a.scale * LOG2E;
  const bool has_sink = a.sink != nullptr && rok && z == 0;
  float m = has_sink ? a.sink[myrow % H] * LOG2E : -1e30f;
  float l = has_sink ? 1.0f : 0.0f;
  f32x16_t o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;

  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
  const int kch = Dk / 8, nkk = Dk / 16, nchunks = MKT * kch;
  // block-table entries of this workgroup's key range in LDS (visible after the loop's first barrier; the first
  // tile's loads read the table from global memory)
  int* btl = reinterpret_cast<int*>(ks + MKT * KP);
  const int b_lo = jlo / a.block_size, nbt = jhi / a.block_size - b_lo + 1;
  const bool bt_lds = nbt <= BT_LDS_MAX;
  if (bt_lds)
    for (int u = tid; u < nbt; u += NT) btl[u] = bt[b_lo + u];
  uint4 pf[NPF];
  auto fetch = [&](int j0, bool lds) {
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      const int idx = tid + u * NT;
      const int k = idx / kch, c = idx % kch, j = j0 + k;
      pf[u] = make_uint4(0, 0, 0, 0);
      if (idx < nchunks && j <= jhi) {
        const int jb = j / a.block_size;
        const int64_t blk = lds ? btl[jb - b_lo] : bt[jb];
        pf[u] = *reinterpret_cast<const uint4*>(cache + (blk * a.block_size + (j - jb * a.block_size)) * Dk + 8 * c);
      }
    }
  };
  fetch(jlo, false);
  const int pitchB = KP * 2;
  const int g16 = lane >> 4, i16 = lane & 15;
  const char* vbase = reinterpret_cast<const char*>(ks) + (4 * hh + (i16 >> 2)) * pitchB +
                      (16 * (g16 & 1) + 4 * (i16 & 3)) * 2;
  for (int j0 = jlo; j0 <= jhi; j0 += MKT) {
    __syncthreads();  // every wave is done with the previous tile (first: the queries are being written)
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      const int idx = tid + u * NT;
      if (idx < nchunks) *reinterpret_cast<uint4*>(ks + (idx / kch) * KP + 8 * (idx % kch)) = pf[u];
    }
    __syncthreads();
    if (j0 + MKT <= jhi) fetch(j0 + MKT, bt_lds);  // in flight while this tile is computed
    if (!wave_live) continue;
    f32x16_t sc;
#pragma unroll
    for (int r = 0; r < 16; ++r) sc[r] = 0.f;
    const bf16_t* ka = ks + qcol * KP + 8 * hh;
    const bf16_t* qb = qs + (wave * 32 + qcol) * KP + 8 * hh;
    for (int kk = 0; kk < nkk; ++kk) {
      const bf16x8_t af = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(ka + 16 * kk));
      const bf16x8_t bfr = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(qb + 16 * kk));
      sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bfr, sc, 0, 0, 0);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int j = j0 + (r & 3) + 8 * (r >> 2) + 4 * hh;
      const bool valid = rok && j <= jhi && j <= prow && (a.window <= 0 || prow - j < a.window);
      const float v = valid ? sc[r] * sl2 : -INFINITY;
      sc[r] = v;
      mx = fmaxf(mx, v);
    }
    mx = xor32_max(mx);
    const float mn = fmaxf(m, mx);
    const float alpha = exp2f(m - mn);
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float pe = exp2f(sc[r] - mn);
      sc[r] = pe;
      sum += pe;
    }
    sum = xor32_sum(sum);
    l = l * alpha + sum;
    m = mn;
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
      if (alpha != 1.0f) {
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
  if (!rok) return;
  if (a.nsplit > 1) {
    float* wo = a.ws_o + ((int64_t)z * a.heads * a.total_q + orow) * R;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(wo + 32 * db + 8 * g + 4 * hh) =
            make_float4(o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]);
    if (hh == 0) {
      a.ws_ml[((int64_t)z * a.heads * a.total_q + orow) * 2] = m;
      a.ws_ml[((int64_t)z * a.heads * a.total_q + orow) * 2 + 1] = l;
    }
    return;
  }
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  bf16_t* op = reinterpret_cast<bf16_t*>(a.out) + orow * R;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      uint2 w;
      w.x = pack2(o[db][4 * g + 0] * inv, o[db][4 * g + 1] * inv);
      w.y = pack2(o[db][4 * g + 2] * inv, o[db][4 * g + 3] * inv);
      *reinterpret_cast<uint2*>(op + 32 * db + 8 * g + 4 * hh) = w;
    }
  }
}

// out[row] = sum_z O_z 2^(m_z - m*) / sum_z l_z 2^(m_z - m*), m* = max_z m_z (running maxima in log2 units). One wave per row, 4 columns per
// lane and pass; the weights of 64 splits at a time on its lanes, so that the splits' rows are loaded together (with one after the other
// behind its weight 16 splits of 512 rows took 10.6 us).
__global__ void __launch_bounds__(256) latent_attn_merge_kernel(bf16_t* out, const float* ws_o, const float* ws_ml,
                                                                int nsplit, int64_t rows, int R) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  float mstar = -1e30f;
  for (int z = lane; z < nsplit; z += 64) mstar = fmaxf(mstar, ws_ml[((int64_t)z * rows + row) * 2]);
  mstar = wave_max(mstar);
  float lsum = 0.f;
  for (int z0 = 0; z0 < nsplit; z0 += 64) {
    const int z = min(z0 + lane, nsplit - 1);
    const float2 ml = *reinterpret_cast<const float2*>(ws_ml + ((int64_t)z * rows + row) * 2);
    lsum += z0 + lane < nsplit && ml.y > 0.f ? ml.y * exp2f(ml.x - mstar) : 0.f;
  }
  lsum = wave_sum(lsum);
  const float inv = lsum > 0.f ? 1.0f / lsum : 0.f;
  for (int c0 = 0; c0 < R; c0 += 256) {
    const int c = c0 + 4 * lane;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int z0 = 0; z0 < nsplit; z0 += 64) {
      const int zl = min(z0 + lane, nsplit - 1);
      const float2 ml = *reinterpret_cast<const float2*>(ws_ml + ((int64_t)zl * rows + row) * 2);
      const float wl = z0 + lane < nsplit && ml.y > 0.f ? exp2f(ml.x - mstar) : 0.f;
      const uint64_t full = __ballot(wl != 0.f);
      if (full == 0) continue;
      const int some = __builtin_ctzll(full), n = 64 - __builtin_clzll(full);
      if (c < R) {
#pragma unroll 8
        for (int z = 0; z < n; ++z) {   // (an empty split's row is not written: another's is read, and counts nothing)
          const float w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wl), z));
          const float4 o = *reinterpret_cast<const float4*>(ws_o + ((int64_t)(z0 + (w != 0.f ? z : some)) * rows + row) * R + c);
          acc.x = fmaf(o.x, w, acc.x), acc.y = fmaf(o.y, w, acc.y), acc.z = fmaf(o.z, w, acc.z), acc.w = fmaf(o.w, w, acc.w);
        }
      }
    }
    if (c < R) *reinterpret_cast<uint2*>(out + row * R + c) = make_uint2(pack2(acc.x * inv, acc.y * inv), pack2(acc.z * inv, acc.w * inv));
  }
}
inline hipError_t launch_merge(const LatentAttnArgs& a, hipStream_t s) {
  const int64_t rows = (int64_t)a.heads * a.total_q;
  hipLaunchKernelGGL(latent_attn_merge_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, reinterpret_cast<bf16_t*>(a.out), a.ws_o, a.ws_ml,
                     a.nsplit, rows, a.sh.rank);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// Decode steps (one row per sequence): 16 heads of a sequence per workgroup, keys in tiles of 32 over its waves and, with nsplit > 1, over
// several workgroups: wave w of all of them takes tiles w, w + waves, .., so that every wave has work whatever the sequence's length. A wave
// loads a tile's rows straight into operands of the scores (key = lane % 16, all loads in flight together, the table's entries a tile
// ahead), writes their latent columns to LDS for the weighted sum's transposed reads, and has the next tile's rows loaded during softmax and
// sum. Waves share no barrier before the end, where their sums are brought to one maximum and added. Against one wave per workgroup that staged
// tiles in LDS for both products, by divisions at run time (rank 256 + 32, main kernel + merge, us): 32 sequences of 750 - 1500 keys, 16 heads
// 36 + 10 -> 12 + 4.7 (21 MB of rows: 4 at the copy rate, latency of three tiles), 64 of 1000 - 2000, 32 heads 87 + 9 -> 24 + 4 (4.0 TB/s with L2), 3 of
// 600 24 + 8 -> 9 + 4, 58 of 10 17 -> 8.
// FINE: the weights enter the products in two bf16 parts (more than 32 heads: launch_decode).
template <int NDB, int NROT> struct DecodeTile {
  static constexpr int R = 32 * NDB, NK = NDB + (NROT + 1) / 2, DK = R + 16 * NROT;   // latent columns, 32-wide steps of a row, its width
  static constexpr int PB = 2 * R + 32;                                               // pitch in LDS, bytes: 4 rows on different banks
  static constexpr int OP = R + 4;                                                    // pitch of a head's sums (floats)
  static constexpr int wave = 32 * PB > 64 * OP ? 32 * PB : 64 * OP;
  static constexpr int total = 4 * wave + 4 * 16 * 2 * 4;
};
template <int NDB, int NROT, bool FINE>
__global__ void __launch_bounds__(256, 2) latent_attn_decode_kernel(LatentAttnArgs a, int hblocks) {
  using Z = DecodeTile<NDB, NROT>;
  constexpr int R = Z::R, NK = Z::NK, ND = R / 16;
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lg = lane >> 4;
  // a sequence's blocks of heads read the same rows: they go to one XCD (workgroups are dealt to the 8 XCDs in turn), one after the other
  const int ns = max(1, a.nsplit), u = blockIdx.x / (8 * hblocks) * 8 + blockIdx.x % 8, hb = blockIdx.x / 8 % hblocks;
  if (u >= a.num_seqs * ns) return;
  const int s = u / ns, z = u % ns, H = a.heads, T = a.total_q;
  const int h0 = 16 * hb, h = min(h0 + li, H - 1);
  const int p = (int)a.positions[s], ctx = a.ctx_lens[s];
  const int jlo = a.window > 0 ? max(0, p - a.window + 1) : 0, jhi = min(p, ctx - 1);
  float* const ml = reinterpret_cast<float*>(dsm + 4 * Z::wave);   // [4][16][2]: maximum, sum of every wave
  const int64_t rows_all = (int64_t)H * T;
  if (jlo + 128 * z > jhi) {   // an empty split: it only reports that it holds nothing
    if (ns > 1 && tid < min(16, H - h0)) {
      float* w = a.ws_ml + ((int64_t)z * rows_all + (int64_t)(h0 + tid) * T + s) * 2;
      w[0] = -1e30f, w[1] = 0.f;
    }
    if (ns > 1) return;
  }
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
  const int bs_shift = (a.block_size & (a.block_size - 1)) == 0 ? __builtin_ctz(a.block_size) : -1;
  auto block_of = [&](int j) { return bs_shift >= 0 ? j >> bs_shift : j / a.block_size; };
  int blk[2];          // block of key 16 t + li of the tile that is loaded next
  bf16x8_t kf[2][NK];
  auto ask = [&](int j0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) blk[t] = bt[block_of(min(j0 + 16 * t + li, jhi))];   // (keys beyond the last repeat it: their weights are zero)
  };
  auto load = [&](int j0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int j = min(j0 + 16 * t + li, jhi);
      const bf16_t* row = cache + ((int64_t)blk[t] * a.block_size + (j - block_of(j) * a.block_size)) * Z::DK + 8 * lg;
#pragma unroll
      for (int c = 0; c < NK; ++c)
        kf[t][c] = *reinterpret_cast<const bf16x8_t*>(row + (NROT == 1 && c == NDB && lg >= 2 ? 0 : 32 * c));
    }
  };
  const int step = 128 * ns;
  int j0 = jlo + 32 * (4 * z + wave);
  const bool any = j0 <= jhi;
  if (any) {
    ask(j0);
    load(j0);
    ask(j0 + step);
  }
  // queries: the latent part as it lies, the rotary part turned in fp32
  bf16x8_t qf[NK];
  const bool mine = h0 + li < H;
  {
    const bf16_t* ql = reinterpret_cast<const bf16_t*>(a.q_lat) + ((int64_t)h * T + s) * R + 8 * lg;
#pragma unroll
    for (int c = 0; c < NDB; ++c) {
      const uint4 w = *reinterpret_cast<const uint4*>(ql + 32 * c);
      qf[c] = __builtin_bit_cast(bf16x8_t, mine ? w : make_uint4(0, 0, 0, 0));
    }
    const bf16_t* qr = reinterpret_cast<const bf16_t*>(a.q_rot) + (int64_t)s * a.q_stride + (int64_t)h * a.q_hstride;
#pragma unroll
    for (int c = NDB; c < NK; ++c) {
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * (c - NDB) + 4 * lg + e;   // pair of dims 2 i, 2 i + 1
        const bool in = mine && 2 * i < a.sh.rot_dim;
        const float x = in ? bf2f(qr[2 * i]) : 0.f, y = in ? bf2f(qr[2 * i + 1]) : 0.f;
        float sn = 0.f, cs = 1.0f;
        if (in && i < a.sh.rot_pairs) __sincosf((float)p * a.sh.inv_freq[i], &sn, &cs);
        w[e] = pack2(x * cs - y * sn, y * cs + x * sn);
      }
      qf[c] = __builtin_bit_cast(bf16x8_t, make_uint4(w[0], w[1], w[2], w[3]));
    }
  }
  constexpr float LOG2E = 1.4426950408889634f;
  const float sl2 = a.scale * LOG2E;
  const bool has_sink = a.sink != nullptr && z == 0 && wave == 0;
  float m = has_sink ? a.sink[h] * LOG2E : -1e30f, l = has_sink && lg == 0 ? 1.0f : 0.0f;
  f32x4_t o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) o[d] = f32x4_t{};
  char* const mem = dsm + wave * Z::wave;
  char* const wr = mem + li * Z::PB + 16 * lg;
  const char* const rd = mem + (4 * lg + (li >> 2)) * Z::PB + 8 * (li & 3);
  for (; j0 <= jhi; j0 += step) {
    f32x4_t sc[2] = {};
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < NK; ++c) {
        bf16x8_t k = kf[t][c];
        if (NROT == 1 && c == NDB && lg >= 2) k = bf16x8_t{};
        sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[c], sc[t], 0, 0, 0);
      }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < NDB; ++c) *reinterpret_cast<bf16x8_t*>(wr + 16 * t * Z::PB + 64 * c) = kf[t][c];
    if (j0 + step <= jhi) {
      load(j0 + step);
      ask(j0 + 2 * step);
    }
    float top = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = j0 + 16 * t + 4 * lg + e <= jhi ? sc[t][e] * sl2 : -INFINITY;
        sc[t][e] = x;
        top = fmaxf(top, x);
      }
    const float mn = fmaxf(m, xor16_max(xor32_max(top)));
    const float alpha = exp2f(m - mn);
    l *= alpha;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sc[t][e] = exp2f(sc[t][e] - mn);
        l += sc[t][e];
      }
    m = mn;
    const uint4 hp = make_uint4(pack2(sc[0][0], sc[0][1]), pack2(sc[0][2], sc[0][3]), pack2(sc[1][0], sc[1][1]), pack2(sc[1][2], sc[1][3]));
    const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, hp);
    bf16x8_t pl;
    if constexpr (FINE)
      pl = __builtin_bit_cast(bf16x8_t, make_uint4(rest2(sc[0][0], sc[0][1], hp.x), rest2(sc[0][2], sc[0][3], hp.y), rest2(sc[1][0], sc[1][1], hp.z),
                                                   rest2(sc[1][2], sc[1][3], hp.w)));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (__ballot(alpha != 1.0f) != 0) {
#pragma unroll
      for (int d = 0; d < ND; ++d) o[d] *= alpha;
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(rd + 32 * d));
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(rd + 16 * Z::PB + 32 * d));
      const short8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      if constexpr (FINE) o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, v), pl, o[d], 0, 0, 0);
      o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, v), pf, o[d], 0, 0, 0);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the tile is read before the next one replaces it
    __builtin_amdgcn_wave_barrier();
  }
  // one maximum for the waves, then the sum of their results
  l = xor16_sum(xor32_sum(l));
  if (lane < 16) ml[(wave * 16 + lane) * 2] = m, ml[(wave * 16 + lane) * 2 + 1] = l;
  __syncthreads();
  float mt = ml[2 * li];
#pragma unroll
  for (int w = 1; w < 4; ++w) mt = fmaxf(mt, ml[(16 * w + li) * 2]);
  const float f = exp2f(m - mt);
  float* const mo = reinterpret_cast<float*>(mem) + li * Z::OP + 4 * lg;   // (the wave's own part: its tiles are done)
#pragma unroll
  for (int d = 0; d < ND; ++d) *reinterpret_cast<f32x4_t*>(mo + 16 * d) = o[d] * f;
  __syncthreads();
  for (int e = tid; e < 16 * R / 4; e += 256) {
    const int hd = e / (R / 4), c = 4 * (e % (R / 4));
    if (h0 + hd >= H) break;
    f32x4_t v = {};
    float mx = ml[2 * hd], lt = 0.f;
#pragma unroll
    for (int w = 1; w < 4; ++w) mx = fmaxf(mx, ml[(16 * w + hd) * 2]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      v += *reinterpret_cast<const f32x4_t*>(dsm + w * Z::wave + 4 * (hd * Z::OP + c));
      lt += ml[(16 * w + hd) * 2 + 1] * exp2f(ml[(16 * w + hd) * 2] - mx);
    }
    const int64_t row = (int64_t)(h0 + hd) * T + s;
    if (ns > 1) {
      *reinterpret_cast<f32x4_t*>(a.ws_o + ((int64_t)z * rows_all + row) * R + c) = v;
      if (c == 0) *reinterpret_cast<float2*>(a.ws_ml + ((int64_t)z * rows_all + row) * 2) = make_float2(mx, lt);
    } else {
      const float inv = lt > 0.f ? 1.0f / lt : 0.f;
      *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(a.out) + row * R + c) = make_uint2(pack2(v[0] * inv, v[1] * inv), pack2(v[2] * inv, v[3] * inv));
    }
  }
}

inline size_t mfma_lds_bytes(int kp, int nw) {
  return sizeof(bf16_t) * (size_t)(32 * nw + MKT) * kp + sizeof(int) * BT_LDS_MAX;
}

template <int NDB, int NW> hipError_t launch_mfma(const LatentAttnArgs& a, hipStream_t s) {
  static bool attr_set[2] = {};
  auto* fn = latent_attn_mfma_kernel<NDB, NW, false>;
  if constexpr (NW == 4 && (NDB == 2 || NDB == 4 || NDB == 8))
    if (a.fine) fn = latent_attn_mfma_kernel<NDB, NW, true>;
  const int kp = a.sh.rank + a.sh.rot_dim + 8;
  bool& set = attr_set[fn != latent_attn_mfma_kernel<NDB, NW, false>];
  if (!set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       144 * 1024);
    if (e != hipSuccess) return e;
    set = true;
  }
  const dim3 grid((unsigned)(((int64_t)a.max_q * a.heads + 32 * NW - 1) / (32 * NW)), (unsigned)a.num_seqs,
                  (unsigned)max(1, a.nsplit));
  hipLaunchKernelGGL(fn, grid, dim3(64 * NW), mfma_lds_bytes(kp, NW), s, a, kp);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.nsplit <= 1) return e;
  return launch_merge(a, s);
}

inline bool mfma_ok(const LatentAttnArgs& a) {
  const int r = a.sh.rank;
  return !a.f32 && r % 32 == 0 && r <= 256 && a.sh.rot_dim % 16 == 0 && a.sh.rot_dim <= 128 &&
         (reinterpret_cast<uintptr_t>(a.q_lat) & 15) == 0 && (reinterpret_cast<uintptr_t>(a.cache) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(a.out) & 7) == 0;
}

// decode steps of the usual row widths
inline bool decode_fits(const LatentAttnArgs& a) {
  const int r = a.sh.rank, d = a.sh.rot_dim;
  return a.impl == 0 && a.cu_q == nullptr && a.max_q == 1 && mfma_ok(a) && (r == 64 || r == 128 || r == 256) && (d == 0 || d == 16 || d == 32 || d == 64);
}
// Two bf16 parts of the weights for more than 32 heads: such steps went through latent_attn_wide_kernel or FINE splits, which have them, and in one
// part were up to 10 % further from 64 bits (in two, 40, 64 and 128 heads, 1.0001 of those kernels; 2 - 8 % of the time). Up to 32 heads the
// kernels before had one part, and more splits: 0.988 of their distance in one. Workgroups of 16 heads read the same rows each, where
// latent_attn_wide_kernel read a tile once for 64 rows, and are faster all the same (rank 256 + 32, with the merge, kernels before / this, us):
// 64 heads 1 x 500 keys 29.0 / 16.2, 1 x 32000 257 / 47, 32 x 500 29.9 / 19.7, 32 x 2000 65 / 32, 64 x 4000 183 / 64; 128 heads 29.2 / 15.9, 262 / 48,
// 29.9 / 18.7, 79 / 42, 212 / 99.
template <int NDB, int NROT> hipError_t launch_decode(const LatentAttnArgs& a, hipStream_t s) {
  const auto fn = a.heads > 32 ? latent_attn_decode_kernel<NDB, NROT, true> : latent_attn_decode_kernel<NDB, NROT, false>;
  constexpr int smem = DecodeTile<NDB, NROT>::total;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  if (e != hipSuccess) return e;
  const int hb = (a.heads + 15) / 16;
  const int64_t units = (int64_t)a.num_seqs * max(1, a.nsplit);
  hipLaunchKernelGGL(fn, dim3((unsigned)((units + 7) / 8 * 8 * hb)), dim3(256), smem, s, a, hb);
  if (a.nsplit <= 1) return hipGetLastError();
  const hipError_t e2 = hipGetLastError();
  return e2 != hipSuccess ? e2 : launch_merge(a, s);
}
template <int NDB> hipError_t launch_decode_rot(const LatentAttnArgs& a, hipStream_t s) {
  if (a.sh.rot_dim == 0) return launch_decode<NDB, 0>(a, s);
  return a.sh.rot_dim == 16 ? launch_decode<NDB, 1>(a, s) : a.sh.rot_dim == 32 ? launch_decode<NDB, 2>(a, s) : launch_decode<NDB, 4>(a, s);
}
hipError_t launch_decode_any(const LatentAttnArgs& a, hipStream_t s) {
  return a.sh.rank == 64 ? launch_decode_rot<2>(a, s) : a.sh.rank == 128 ? launch_decode_rot<4>(a, s) : launch_decode_rot<8>(a, s);
}

template <int NW> hipError_t launch_mfma_ndb(const LatentAttnArgs& a, hipStream_t s) {
  switch (a.sh.rank / 32) {
    case 1: return launch_mfma<1, NW>(a, s);
    case 2: return launch_mfma<2, NW>(a, s);
    case 3: return launch_mfma<3, NW>(a, s);
    case 4: return launch_mfma<4, NW>(a, s);
    case 5: return launch_mfma<5, NW>(a, s);
    case 6: return launch_mfma<6, NW>(a, s);
    case 7: return launch_mfma<7, NW>(a, s);
    case 8: return launch_mfma<8, NW>(a, s);
  }
  return hipErrorInvalidValue;
}

// The first row and the sequence of a workgroup, of a grid (tiles of ROWS rows, sequences); false where the sequence has no such tile. A sequence's
// last tiles see the most keys and start first. Workgroups go to the 8 XCDs, which have an L2 each, in turn. Numbers of
// sequences that are multiples of 8: sequence s is XCD s % 8's, one after the other, so that its cache rows are in one L2 (all
// sequences' last tiles first, and so more sequences in an L2 at a time: 32 of 250 ragged rows, 32 heads 76 -> 90 us; 16 of 1024
// 203 -> 230). Other numbers share every L2 anyhow: there the last tiles of all sequences start first, which leaves the short ones for
// the end and gives each CU one of every kind (one sequence after the other, equal lengths, 16 heads: 12 of 500 73 -> 55, 7 of
// 1000 129 -> 105, 12 of 182 22.9 -> 22.1). So do up to 3 sequences of unequal lengths per XCD, each of them over all XCDs: an XCD's own would
// hold 1.3 - 1.5 times the mean work (24 of 101 - 200 rows, 16 heads 47.7 -> 38.7, 16 of 251 - 500, 32 heads 151 -> 120, 8 of 351 - 700 80 -> 73).
template <int ROWS> __device__ __forceinline__ bool tile_of(const LatentAttnArgs& a, int& s, int& row0) {
  const unsigned nx = gridDim.x, n = gridDim.y, lin = blockIdx.x + nx * blockIdx.y;
  unsigned t;   // from the sequence's last tile
  if (n % 8 == 0 && (n >= 32 || a.total_q == (int64_t)a.max_q * n)) {
    t = lin / 8 % nx;
    s = (int)(lin % 8 + 8 * (lin / 8 / nx));
  } else {
    t = lin / n;
    s = (int)(n % 8 == 0 ? (lin % n + t) % n : lin % n);
  }
  const int rows = (a.cu_q ? a.cu_q[s + 1] - a.cu_q[s] : 1) * a.heads;
  row0 = ((rows + ROWS - 1) / ROWS - 1 - (int)t) * ROWS;
  return row0 >= 0;
}

// Prompt-sized steps at the common rotary widths (rot_dim = 16 * NROT, NROT = 0: no rotary part): the same algorithm with every
// wave's query fragments in registers (loaded straight from global memory, the rotary part rotated on the way). A wave owns 16
// rows: sums and queries take 64 + 36 registers at rank 256, so that 3 waves share a SIMD and one's softmax runs beside the others'
// products. Key tiles come by DMA into two buffers of a workgroup of 4 waves, one barrier per tile. A tile of 32 rows by KCH 16-byte
// pieces lies in LDS as the DMA writes it, without gaps; the pieces of a row are exchanged (XOR) so that 16 consecutive rows' reads
// of one piece fall on all banks, and so do the transposed reads of 8 rows by two pieces (the number is rotated for those: by the plain
// row number pairs of rows shared banks, a quarter of the kernel's cycles).
// Bound by the latency of its LDS reads (see latent_attn_two_kernel, which takes larger steps). 16 sequences of 1024 rows, 16 heads,
// rank 256 + 32: 32 rows per wave, one wave per SIMD, tiles through registers, looked up piece by piece behind divisions: 518 us;
// the same with DMA and the next tile's scores under the softmax 370; this 246 (250 with the queries
// loaded behind the first tile, where 24 - 100 rows of 20 and more sequences took 3 % longer too).
template <int NDB, int NROT> struct RqTile {
  static constexpr int KCH = 4 * NDB + 2 * NROT, NPF = (MKT * KCH + 255) / 256, BYTES = NPF * 4096;
  static constexpr int G = KCH % 16 == 0 ? 16 : KCH % 8 == 0 ? 8 : KCH % 4 == 0 ? 4 : 2;   // rows r and r + 16 / G share banks
  static __device__ __forceinline__ int swz(int row) {
    const int i = row / (16 / G) % G;
    return (2 * i & (G - 1)) | i / (G / 2);
  }
  static constexpr int OP = 64 * NDB + 16;   // pitch of a result row in LDS
  static constexpr int TABLE = 1024;         // block-table entries in LDS
  static constexpr int LDS = 2 * BYTES + 4 * TABLE > 64 * OP ? 2 * BYTES + 4 * TABLE : 64 * OP;
};
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void global_cvoid;

template <int NDB, int NROT>
__global__ void __launch_bounds__(256, 3) latent_attn_mfma_rq_kernel(LatentAttnArgs a, uint32_t bs_mul, int bs_shift) {
  using Z = RqTile<NDB, NROT>;
  constexpr int KCH = Z::KCH, NPF = Z::NPF, NLAT = NDB, NK = NDB + NROT / 2;   // 32-wide steps of a row: latent, in all
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];   // two tiles, block-table entries; at the end the results
  int s, row0;
  if (!tile_of<64>(a, s, row0)) return;
  const int lane = threadIdx.x & 63, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.heads;
  constexpr int R = 32 * NDB, Dk = R + 16 * NROT;
  const int q0 = a.cu_q ? a.cu_q[s] : s;
  const int nq = a.cu_q ? a.cu_q[s + 1] - q0 : 1;
  const int nrows = nq * H;
  const int ctx = a.ctx_lens[s];
  const int last_row = min(row0 + 64, nrows) - 1;
  const int p_first = (int)a.positions[q0 + row0 / H], p_last = (int)a.positions[q0 + last_row / H];
  const int jlo = a.window > 0 ? max(0, p_first - a.window + 1) : 0;
  const int jhi = min(p_last, ctx - 1);
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  const int li = lane & 15, lg = lane >> 4;

  const int wrow = row0 + wave * 16, myrow = wrow + li;
  const bool rok = myrow < nrows, wave_live = wrow < nrows, all_rows = wrow + 15 < nrows;
  const int64_t tq = rok ? q0 + myrow / H : q0;
  const int hq = rok ? myrow % H : 0;
  const int64_t orow = (int64_t)hq * a.total_q + tq;
  const int prow = rok ? (int)a.positions[tq] : -1;
  const int pw_min = wave_live ? (int)a.positions[q0 + wrow / H] : 0;
  const int pw_max = wave_live ? (int)a.positions[q0 + min(wrow + 15, nrows - 1) / H] : 0;
  // this lane's query fragments: qf[k] = Q[row][32 k + 8 lg .. + 8]; an odd NROT leaves 16 columns, of which the lane has 4. (Rows
  // beyond the last repeat the first; every load is unconditional, so that all are in flight together, and beside the table's.)
  bf16x8_t qf[NK > 0 ? NK : 1];
  short4_t qt = {};
  const bf16_t* qlat = reinterpret_cast<const bf16_t*>(a.q_lat) + orow * R;
#pragma unroll
  for (int k = 0; k < NLAT; ++k) qf[k] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(qlat + 32 * k + 8 * lg));
  constexpr int E = NROT % 2 == 0 ? 8 : 4, NS = (NROT + 1) / 2;
  bf16_t qr[NS > 0 ? NS : 1][E];
  float fr[NS > 0 ? NS : 1][E / 2];
  if constexpr (NROT > 0) {
    const bf16_t* qp = reinterpret_cast<const bf16_t*>(a.q_rot) + tq * a.q_stride + (int64_t)hq * a.q_hstride + E * lg;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
#pragma unroll
      for (int e = 0; e < E; ++e) qr[k][e] = qp[32 * k + e];
#pragma unroll
      for (int i = 0; i < E / 2; ++i)
        fr[k][i] = a.sh.rot_pairs > 0 ? a.sh.inv_freq[min(16 * k + E / 2 * lg + i, a.sh.rot_pairs - 1)] : 0.f;
    }
  }

  // Block-table entries of the workgroup's keys in LDS (TABLE at a time), so that a tile's loads depend on LDS reads alone
  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
  int* btl = reinterpret_cast<int*>(smem_raw + 2 * Z::BYTES);
  auto block_of = [&](int j) { return a.block_size == 1 ? j : (int)(__umulhi((uint32_t)j, bs_mul) >> bs_shift); };
  const int b_hi = block_of(max(jhi, 0));
  int b_lo = block_of(jlo);
  auto stage_table = [&]() {
    for (int u = tid; u < Z::TABLE && b_lo + u <= b_hi; u += 256) btl[u] = bt[b_lo + u];
    __syncthreads();
  };
  stage_table();
  // tile rows by DMA: piece u of this thread is 16 bytes of key krow[u] (beyond the tile: of key 31, into the slack)
  int krow[NPF], pcol[NPF];
#pragma unroll
  for (int u = 0; u < NPF; ++u) {
    const int idx = tid + 256 * u, row = min(idx / KCH, MKT - 1);
    krow[u] = row;
    pcol[u] = 8 * (idx < MKT * KCH ? (idx - row * KCH) ^ Z::swz(row) : 0);
  }
  auto fetch = [&](int j0, int buf) {   // (keys beyond the last repeat it)
    if (block_of(min(j0 + MKT - 1, jhi)) >= b_lo + Z::TABLE) {
      __syncthreads();
      b_lo = block_of(j0);
      stage_table();
    }
    uint32_t row[NPF];   // (as many cache rows as a device holds)
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      const int j = min(j0 + krow[u], jhi), jb = block_of(j);
      row[u] = (uint32_t)btl[jb - b_lo] * (uint32_t)a.block_size + (uint32_t)(j - jb * a.block_size);
    }
    __builtin_amdgcn_sched_barrier(0);   // (all lookups, then the loads: they would go in turns, each waited for)
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      char* to = smem_raw + buf * Z::BYTES + (256 * u + 64 * wave) * 16;
      __builtin_amdgcn_global_load_lds((global_cvoid*)(cache + ((uint64_t)row[u] * Dk + pcol[u])), (lds_void*)to, 16, 0, 0);
    }
  };
  const int nt = jhi < jlo ? 0 : (jhi - jlo) / MKT + 1;
  if (nt > 0) fetch(jlo, 0);

  if constexpr (NROT > 0) {
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      float f[8] = {};
#pragma unroll
      for (int i = 0; i < E / 2; ++i) {
        const float u = bf2f(qr[k][2 * i]), w = bf2f(qr[k][2 * i + 1]);
        float sn, cs;
        __sincosf((float)prow * fr[k][i], &sn, &cs);
        const bool turned = 16 * k + E / 2 * lg + i < a.sh.rot_pairs;
        f[2 * i] = turned ? u * cs - w * sn : u;
        f[2 * i + 1] = turned ? w * cs + u * sn : w;
      }
      const uint4 w = pack8(f);
      if constexpr (E == 8)
        qf[NLAT + k] = __builtin_bit_cast(bf16x8_t, w);
      else
        qt = __builtin_bit_cast(short4_t, make_uint2(w.x, w.y));
    }
  }

  constexpr float LOG2E = 1.4426950408889634f;
  const float sl2 = a.scale * LOG2E;
  const bool has_sink = a.sink != nullptr && rok;
  float m = has_sink ? a.sink[hq] * LOG2E : -1e30f;
  float l = has_sink && lg == 0 ? 1.0f : 0.0f;   // (the sum of this lane's keys)
  f32x4_t o[2 * NDB];
#pragma unroll
  for (int db = 0; db < 2 * NDB; ++db) o[db] = f32x4_t{};
  // K fragments: key li of 16, piece 4 k + lg; V fragments: keys 4 lg .. of either 16 (the order in which the weights lie in
  // registers), columns 16 db ..
  const int ksw = Z::swz(li), vrow = 4 * lg + (li >> 2), vsw = Z::swz(vrow);
  const int kat = 16 * li * KCH, vat = 16 * vrow * KCH + 8 * (li & 1);
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
    if (!wave_live) continue;
    const char* ks = smem_raw + (i & 1) * Z::BYTES;
    f32x4_t sc[2] = {};
#pragma unroll
    for (int k = 0; k < NK; ++k)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint4 w = *reinterpret_cast<const uint4*>(ks + kat + 256 * KCH * t + 16 * ((4 * k + lg) ^ ksw));
        sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w), qf[k], sc[t], 0, 0, 0);
      }
    if constexpr (NROT % 2 != 0)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint2 w = *reinterpret_cast<const uint2*>(ks + kat + 256 * KCH * t + 16 * ((4 * NK + (lg >> 1)) ^ ksw) + 8 * (lg & 1));
        sc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(short4_t, w), qt, sc[t], 0, 0, 0);
      }
    // interior tiles (every key visible to every row of the wave) skip the per-score mask
    float mx = -INFINITY;
    const bool inner = all_rows && j0 + MKT - 1 <= min(pw_min, jhi) && (a.window <= 0 || pw_max - j0 < a.window);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) sc[t][e] *= sl2;
    if (!inner) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = j0 + 16 * t + 4 * lg + e;
          const bool valid = rok && j <= jhi && j <= prow && (a.window <= 0 || prow - j < a.window);
          sc[t][e] = valid ? sc[t][e] : -INFINITY;
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, sc[t][e]);
    mx = xor16_max(xor32_max(mx));
    const float mn = fmaxf(m, mx);
    float alpha = __builtin_amdgcn_exp2f(m - mn);
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sc[t][e] = __builtin_amdgcn_exp2f(sc[t][e] - mn);
        sum += sc[t][e];
      }
    l = l * alpha + sum;
    m = mn;
    const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, make_uint4(pack2(sc[0][0], sc[0][1]), pack2(sc[0][2], sc[0][3]),
                                                                pack2(sc[1][0], sc[1][1]), pack2(sc[1][2], sc[1][3])));
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {   // wave-uniform
      asm volatile("" : "+v"(alpha));                        // (not multiplied ahead of the condition)
#pragma unroll
      for (int db = 0; db < 2 * NDB; ++db)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[db][e] *= alpha;
    }
#pragma unroll
    for (int db = 0; db < 2 * NDB; ++db) {
      const char* at = ks + vat + 16 * ((2 * db + (li >> 1 & 1)) ^ vsw);   // (rows r and r + 16 are exchanged alike)
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)at);
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at + 256 * KCH));
      const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, o[db], 0, 0, 0);
    }
  }
  // results through LDS (tiles and table are done with), so that whole rows are written 16 bytes a lane
  __syncthreads();
  l = xor16_sum(xor32_sum(l));
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  char* os = smem_raw + wave * 16 * Z::OP;
#pragma unroll
  for (int db = 0; db < 2 * NDB; ++db)
    *reinterpret_cast<uint2*>(os + li * Z::OP + 32 * db + 8 * lg) = make_uint2(pack2(o[db][0] * inv, o[db][1] * inv), pack2(o[db][2] * inv, o[db][3] * inv));
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  constexpr int PR = R / 8, RPI = 64 / PR;   // pieces of a row, rows of an instruction
#pragma unroll
  for (int u = 0; u < 16 / RPI; ++u) {
    const int row = RPI * u + lane / PR;
    const int64_t to = (int64_t)__shfl((int)orow, row, 64) * R + 8 * (lane % PR);
    const uint4 w = *reinterpret_cast<const uint4*>(os + row * Z::OP + 16 * (lane % PR));
    if (wrow + row < nrows) *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(a.out) + to) = w;
  }
}

// The same with two groups of 16 rows per wave, each fragment that is read from LDS serving both, and the next ones read ahead of a step's products (with
// one group and three waves per SIMD there are no registers for that, and every pair of products waited for its reads: a wave and tile took 6300
// cycles for 410 instructions). Sums take 128 registers at rank 256; of the queries' 72 the first NQL steps' lie in LDS, so that two waves fit on a SIMD and two workgroups
// of 128 rows on a CU. The scale enters with the exponential's argument (a positive one). What bounds it: vector instructions, 49 % of the cycles (80 to 210 of a wave and
// tile rescale and exponentiate), beside products, 32 %, and LDS reads that the two waves of a SIMD don't hide; 16 sequences of 1024 rows, 16 heads, rank 256 + 32:
// 243 -> 193 us in the step (by the profiler, median of 12 passes, 272 -> 214). (The next tile's fetch kept apart from the transposed reads, which the compiler has wait for it, or waves in products first: 1 - 3 % slower.)
template <int NDB, int NROT> struct TwoTile : RqTile<NDB, NROT> {
  static_assert(NDB == 8, "below rank 256 three waves of one group are faster");
  using Z = RqTile<NDB, NROT>;
  static constexpr int ROWS = 128, NK = NDB + NROT / 2;         // rows of a workgroup; 32-wide steps of a row
  static constexpr int NQL = NROT == 0 ? 5 : 4, QB = 2048 * NQL;   // steps whose query fragments lie in LDS, a wave's bytes of them
  static constexpr int ALL = 2 * Z::BYTES + 4 * QB + 4 * Z::TABLE, LDS = ALL > 64 * Z::OP ? ALL : 64 * Z::OP;
  static_assert(2 * LDS <= 160 * 1024, "two workgroups per compute unit");
};
template <int NDB, int NROT>
__global__ void __launch_bounds__(256, 2) latent_attn_two_kernel(LatentAttnArgs a, uint32_t bs_mul, int bs_shift) {
  using Z = TwoTile<NDB, NROT>;
  constexpr int KCH = Z::KCH, NPF = Z::NPF, NLAT = NDB, NK = Z::NK, NQL = Z::NQL;   // 32-wide steps of a row: latent, in all
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];   // two tiles, query fragments, block-table entries; at the end the results
  int s, row0;
  if (!tile_of<Z::ROWS>(a, s, row0)) return;
  const int lane = threadIdx.x & 63, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.heads;
  constexpr int R = 32 * NDB, Dk = R + 16 * NROT;
  const int q0 = a.cu_q ? a.cu_q[s] : s;
  const int nq = a.cu_q ? a.cu_q[s + 1] - q0 : 1;
  const int nrows = nq * H;
  const int ctx = a.ctx_lens[s];
  const int last_row = min(row0 + Z::ROWS, nrows) - 1;
  const int p_first = (int)a.positions[q0 + row0 / H], p_last = (int)a.positions[q0 + last_row / H];
  const int jlo = a.window > 0 ? max(0, p_first - a.window + 1) : 0;
  const int jhi = min(p_last, ctx - 1);
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  const int li = lane & 15, lg = lane >> 4;

  const int wrow = row0 + wave * 32;
  const bool wave_live = wrow < nrows, all_rows = wrow + 31 < nrows;
  const int pw_min = wave_live ? (int)a.positions[q0 + wrow / H] : 0;
  const int pw_max = wave_live ? (int)a.positions[q0 + min(wrow + 31, nrows - 1) / H] : 0;
  // this lane's query fragments of either group: 32-wide step k of row li, columns 32 k + 8 lg .. + 8; an odd NROT leaves 16 columns, of which the lane
  // has 4. The first NQL steps go to LDS. (Rows beyond the last repeat the first; every load is unconditional, so that all are in flight together, and
  // beside the table's.)
  int prow[2];
  uint32_t orow[2];
  float sink[2];
  bf16x8_t qf[2][NK > 0 ? NK : 1];
  short4_t qt[2] = {};
  constexpr int E = NROT % 2 == 0 ? 8 : 4, NS = (NROT + 1) / 2;
  bf16_t qr[2][NS > 0 ? NS : 1][E];
  float fr[NS > 0 ? NS : 1][E / 2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int myrow = wrow + 16 * g + li;
    const bool rok = myrow < nrows;
    const int64_t tq = rok ? q0 + myrow / H : q0;
    const int hq = rok ? myrow % H : 0;
    orow[g] = (uint32_t)((int64_t)hq * a.total_q + tq);
    prow[g] = rok ? (int)a.positions[tq] : -1;
    sink[g] = a.sink != nullptr ? a.sink[hq] : 0.f;
    const bf16_t* qlat = reinterpret_cast<const bf16_t*>(a.q_lat) + (int64_t)orow[g] * R;
#pragma unroll
    for (int k = 0; k < NLAT; ++k) qf[g][k] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(qlat + 32 * k + 8 * lg));
    if constexpr (NROT > 0) {
      const bf16_t* qp = reinterpret_cast<const bf16_t*>(a.q_rot) + tq * a.q_stride + (int64_t)hq * a.q_hstride + E * lg;
#pragma unroll
      for (int k = 0; k < NS; ++k)
#pragma unroll
        for (int e = 0; e < E; ++e) qr[g][k][e] = qp[32 * k + e];
    }
  }
  if constexpr (NROT > 0) {
#pragma unroll
    for (int k = 0; k < NS; ++k)
#pragma unroll
      for (int i = 0; i < E / 2; ++i)
        fr[k][i] = a.sh.rot_pairs > 0 ? a.sh.inv_freq[min(16 * k + E / 2 * lg + i, a.sh.rot_pairs - 1)] : 0.f;
  }

  // Block-table entries of the workgroup's keys in LDS (TABLE at a time), so that a tile's loads depend on LDS reads alone
  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
  int* btl = reinterpret_cast<int*>(smem_raw + 2 * Z::BYTES + 4 * Z::QB);
  char* const ql = smem_raw + 2 * Z::BYTES + wave * Z::QB + 16 * lane;   // the wave's query fragments
  auto block_of = [&](int j) { return a.block_size == 1 ? j : (int)(__umulhi((uint32_t)j, bs_mul) >> bs_shift); };
  const int b_hi = block_of(max(jhi, 0));
  int b_lo = block_of(jlo);
  auto stage_table = [&]() {
    for (int u = tid; u < Z::TABLE && b_lo + u <= b_hi; u += 256) btl[u] = bt[b_lo + u];
    __syncthreads();
  };
  stage_table();
  // tile rows by DMA: piece u of this thread is 16 bytes of key krow[u] (beyond the tile: of key 31, into the slack)
  int krow[NPF], pcol[NPF];
#pragma unroll
  for (int u = 0; u < NPF; ++u) {
    const int idx = tid + 256 * u, row = min(idx / KCH, MKT - 1);
    krow[u] = row;
    pcol[u] = 8 * (idx < MKT * KCH ? (idx - row * KCH) ^ Z::swz(row) : 0);
  }
  auto fetch = [&](const bf16_t* src, char* to, int j0) __attribute__((always_inline)) {   // (keys beyond the last repeat it)
    if (block_of(min(j0 + MKT - 1, jhi)) >= b_lo + Z::TABLE) {
      __syncthreads();
      b_lo = block_of(j0);
      stage_table();
    }
    uint32_t row[NPF];   // (as many cache rows as a device holds)
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      const int j = min(j0 + krow[u], jhi), jb = block_of(j);
      row[u] = (uint32_t)btl[jb - b_lo] * (uint32_t)a.block_size + (uint32_t)(j - jb * a.block_size);
    }
    __builtin_amdgcn_sched_barrier(0);   // (all lookups, then the loads: they would go in turns, each waited for)
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      __builtin_amdgcn_global_load_lds((global_cvoid*)(src + ((uint64_t)row[u] * Dk + pcol[u])), (lds_void*)(to + (256 * u + 64 * wave) * 16), 16, 0, 0);
    }
  };
  const int nt = jhi < jlo ? 0 : (jhi - jlo) / MKT + 1;
  if (nt > 0) fetch(cache, smem_raw, jlo);

#pragma unroll
  for (int g = 0; g < 2; ++g) {
    if constexpr (NROT > 0) {
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        float f[8] = {};
#pragma unroll
        for (int i = 0; i < E / 2; ++i) {
          const float u = bf2f(qr[g][k][2 * i]), w = bf2f(qr[g][k][2 * i + 1]);
          float sn, cs;
          __sincosf((float)prow[g] * fr[k][i], &sn, &cs);
          const bool turned = 16 * k + E / 2 * lg + i < a.sh.rot_pairs;
          f[2 * i] = turned ? u * cs - w * sn : u;
          f[2 * i + 1] = turned ? w * cs + u * sn : w;
        }
        const uint4 w = pack8(f);
        if constexpr (E == 8)
          qf[g][NLAT + k] = __builtin_bit_cast(bf16x8_t, w);
        else
          qt[g] = __builtin_bit_cast(short4_t, make_uint2(w.x, w.y));
      }
    }
#pragma unroll
    for (int k = 0; k < NQL; ++k) *reinterpret_cast<uint4*>(ql + 1024 * (2 * k + g)) = __builtin_bit_cast(uint4, qf[g][k]);
  }
  // (a wave reads the fragments that it wrote)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();

  constexpr float LOG2E = 1.4426950408889634f;
  const float sl2 = a.scale * LOG2E;
  float m[2], l[2];   // (l: the sum of this lane's keys)
  f32x4_t o[2][2 * NDB];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const bool has_sink = a.sink != nullptr && wrow + 16 * g + li < nrows;
    m[g] = has_sink ? sink[g] * LOG2E : -1e30f;
    l[g] = has_sink && lg == 0 ? 1.0f : 0.0f;
#pragma unroll
    for (int db = 0; db < 2 * NDB; ++db) o[g][db] = f32x4_t{};
  }
  // K fragments: key li of 16, piece 4 k + lg; V fragments: keys 4 lg .. of either 16 (the order in which the weights lie in
  // registers), columns 16 db ..
  // (the number that is XOR-ed is below G: a piece G and more on is an offset)
  constexpr int KB = Z::G < 4 ? 1 : Z::G / 4, VB = Z::G / 2;
  const int ksw = Z::swz(li), vrow = 4 * lg + (li >> 2), vsw = Z::swz(vrow);
  uint32_t kat[KB], vat[VB];
#pragma unroll
  for (int u = 0; u < KB; ++u) kat[u] = 16 * li * KCH + 16 * ((4 * u + lg) ^ ksw);
#pragma unroll
  for (int u = 0; u < VB; ++u) vat[u] = 16 * vrow * KCH + 8 * (li & 1) + 16 * ((2 * u + (li >> 1 & 1)) ^ vsw);   // (rows r and r + 16 are exchanged alike)
  // The queries are here. (Without this the compiler waits for them in the loop, behind the next tile's DMA and so for that too.)
  __builtin_amdgcn_s_waitcnt(15 << 8 | 7 << 4);
  // Tile i at `ks`, the next one's fetch to `to`
  auto tile = [&](const bf16_t* src, char* to, const char* ks, int i) __attribute__((always_inline)) {
    const int j0 = jlo + i * MKT;
    // tile i is in LDS for every wave, and every wave has left the other buffer
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(7 << 4);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (i + 1 < nt) fetch(src, to, j0 + MKT);
    if (!wave_live) return;
    f32x4_t sc[2][2] = {};   // [group][16 keys]
    // fragments of the next step of the row ahead of a step's products; each serves both groups
    bf16x8_t kf[2][2], qs[2][2];
    auto read_k = [&](int k) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
        kf[k & 1][t] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(ks + kat[k % KB] + 256 * KCH * t + 64 * (k - k % KB)));
      if (k < NQL) {
#pragma unroll
        for (int g = 0; g < 2; ++g) qs[k & 1][g] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(ql + 1024 * (2 * k + g)));
      }
    };
    read_k(0);
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      if (k + 1 < NK) read_k(k + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int g = 0; g < 2; ++g)
          sc[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[k & 1][t], k < NQL ? qs[k & 1][g] : qf[g][k], sc[g][t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (NROT % 2 != 0)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint2 w = *reinterpret_cast<const uint2*>(ks + 16 * li * KCH + 256 * KCH * t + 16 * ((4 * NK + (lg >> 1)) ^ ksw) + 8 * (lg & 1));
#pragma unroll
        for (int g = 0; g < 2; ++g) sc[g][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(short4_t, w), qt[g], sc[g][t], 0, 0, 0);
      }
    // V fragments VG column blocks ahead, the first ones beside the softmax
    constexpr int VG = 2, NV = 2 * NDB / VG;
    bf16x8_t vf[2][VG];
    auto read_v = [&](int g) __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < VG; ++d) {
        const int db = VG * g + d;
        const char* at = ks + vat[db % VB] + 32 * (db - db % VB);
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)at);
        const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at + 256 * KCH));
        vf[g & 1][d] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    read_v(0);
    __builtin_amdgcn_sched_barrier(0);
    // interior tiles (every key visible to every row of the wave) skip the per-score mask
    const bool inner = all_rows && j0 + MKT - 1 <= min(pw_min, jhi) && (a.window <= 0 || pw_max - j0 < a.window);
    if (!inner) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = j0 + 16 * t + 4 * lg + e;   // (rows beyond the last: position -1)
            const bool valid = j <= jhi && j <= prow[g] && (a.window <= 0 || prow[g] - j < a.window);
            sc[g][t][e] = valid ? sc[g][t][e] : -INFINITY;
          }
    }
    bf16x8_t pf[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, sc[g][t][e]);
      const float mn = fmaxf(m[g], xor16_max(xor32_max(mx)) * sl2);
      float alpha = __builtin_amdgcn_exp2f(m[g] - mn);
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sc[g][t][e] = __builtin_amdgcn_exp2f(fmaf(sc[g][t][e], sl2, -mn));
          sum += sc[g][t][e];
        }
      l[g] = l[g] * alpha + sum;
      m[g] = mn;
      pf[g] = __builtin_bit_cast(bf16x8_t, make_uint4(pack2(sc[g][0][0], sc[g][0][1]), pack2(sc[g][0][2], sc[g][0][3]), pack2(sc[g][1][0], sc[g][1][1]),
                                                      pack2(sc[g][1][2], sc[g][1][3])));
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {   // wave-uniform
        asm volatile("" : "+v"(alpha));                        // (not multiplied ahead of the condition)
#pragma unroll
        for (int db = 0; db < 2 * NDB; ++db)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[g][db][e] *= alpha;
      }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v + 1 < NV) read_v(v + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < VG; ++d)
#pragma unroll
        for (int g = 0; g < 2; ++g) o[g][VG * v + d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[v & 1][d], pf[g], o[g][VG * v + d], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int i = 0; i < nt; ++i) tile(cache, smem_raw + (~i & 1) * Z::BYTES, smem_raw + (i & 1) * Z::BYTES, i);
  // results through LDS (tiles and table are done with), 16 rows at a time, so that whole rows are written 16 bytes a lane
  __syncthreads();
  char* os = smem_raw + wave * 16 * Z::OP;
  constexpr int PR = R / 8, RPI = 64 / PR;   // pieces of a row, rows of an instruction
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const float sum = xor16_sum(xor32_sum(l[g])), inv = sum > 0.f ? 1.0f / sum : 0.f;
#pragma unroll
    for (int db = 0; db < 2 * NDB; ++db)
      *reinterpret_cast<uint2*>(os + li * Z::OP + 32 * db + 8 * lg) =
          make_uint2(pack2(o[g][db][0] * inv, o[g][db][1] * inv), pack2(o[g][db][2] * inv, o[g][db][3] * inv));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int u = 0; u < 16 / RPI; ++u) {
      const int row = RPI * u + lane / PR;
      const int64_t to = (int64_t)__shfl((int)orow[g], row, 64) * R + 8 * (lane % PR);
      const uint4 w = *reinterpret_cast<const uint4*>(os + row * Z::OP + 16 * (lane % PR));
      if (wrow + 16 * g + row < nrows) *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(a.out) + to) = w;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (the rows are read before the other group's replace them)
    __builtin_amdgcn_wave_barrier();
  }
}

// The same with 32 rows per wave and 32x32x16 products, for steps of few row tiles (launch_rows): a fragment that is read from LDS serves 32
// rows, and the next ones are read ahead of a group's products. Two waves share 32 rows: both form the scores and weights, each its half
// of the value columns, so that sums and queries take 64 + 72 registers at rank 256 and two waves share a SIMD. (Whole rows
// per wave spill with two waves per SIMD; with one its sums move between the two kinds of registers: 337 us of 16 x 1024 rows against 324.)
// The weights enter the products in two bf16 parts: split keys, which such steps had before, round relative to every split's own
// largest weight, and whole keys with rounded weights were up to 4 % further from 64 bits.
template <int NDB, int NROT> struct LatentTile {
  static constexpr int KCH = 4 * NDB + 2 * NROT, NPF = (32 * KCH + 255) / 256, BYTES = NPF * 256 * 16;
  static constexpr int X = KCH % 16 == 0 ? 16 : KCH % 8 == 0 ? 8 : KCH % 4 == 0 ? 4 : 2;   // pieces that change places
  static __device__ __forceinline__ int swz(int row) {
    return X == 16 ? (row & 3) << 2 | (row >> 2 & 3) : X == 8 ? (row >> 1 & 1) << 2 | (row >> 2 & 3) : row / (16 / X) % X;
  }
  static constexpr int HC = 2, ROWS = 128 / HC;   // waves that share rows, each with its value columns; rows of a workgroup
  static constexpr int TABLE = 1024;                            // key rows in LDS
  static constexpr int LDS = 2 * BYTES + 4 * TABLE;
};

template <int NDB, int NROT>
__global__ void __launch_bounds__(256, 2) latent_attn_wide_kernel(LatentAttnArgs a, uint32_t bs_mul, int bs_shift) {
  using Z = LatentTile<NDB, NROT>;
  constexpr int HC = Z::HC, NO = NDB / HC;   // 32-column blocks of a wave
  constexpr int KCH = Z::KCH, NPF = Z::NPF, KT = 32, NLAT = 2 * NDB, NK = NLAT + NROT;   // 16-wide steps of a row: latent, in all
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];   // two tiles, key rows
  int s, row0;
  if (!tile_of<Z::ROWS>(a, s, row0)) return;
  const int lane = threadIdx.x & 63, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.heads;
  constexpr int R = 32 * NDB, Dk = R + 16 * NROT;
  const int q0 = a.cu_q ? a.cu_q[s] : s;
  const int nq = a.cu_q ? a.cu_q[s + 1] - q0 : 1;
  const int nrows = nq * H;
  const int ctx = a.ctx_lens[s];
  const int last_row = min(row0 + Z::ROWS, nrows) - 1;
  const int p_first = (int)a.positions[q0 + row0 / H], p_last = (int)a.positions[q0 + last_row / H];
  const int jlo = a.window > 0 ? max(0, p_first - a.window + 1) : 0;
  const int jhi = min(p_last, ctx - 1);
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  const int li = lane & 31, hi = lane >> 5;

  // cache rows of the workgroup's keys in LDS, TABLE keys at a time
  const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
  int* rows = reinterpret_cast<int*>(smem_raw + 2 * Z::BYTES);
  int jt = jlo;
  auto stage_rows = [&]() {
    for (int u = tid; u < Z::TABLE && jt + u <= jhi; u += 256) {
      const int jb = a.block_size == 1 ? jt + u : (int)(__umulhi((uint32_t)(jt + u), bs_mul) >> bs_shift);
      rows[u] = (int)((uint32_t)bt[jb] * (uint32_t)a.block_size + (uint32_t)(jt + u - jb * a.block_size));
    }
    __syncthreads();
  };
  stage_rows();
  // tile rows by DMA: piece u of this thread is 16 bytes of key krow[u] (beyond the tile: of its last key, into the slack)
  int krow[NPF], pcol[NPF];
#pragma unroll
  for (int u = 0; u < NPF; ++u) {
    const int idx = tid + 256 * u, row = min(idx / KCH, KT - 1);
    krow[u] = row;
    pcol[u] = 8 * (idx < KT * KCH ? (idx - row * KCH) ^ Z::swz(row) : 0);
  }
  auto fetch = [&](int j0, int buf) {   // (keys beyond the last repeat it)
    if (min(j0 + KT - 1, jhi) - jt >= Z::TABLE) {
      __syncthreads();
      jt = j0;
      stage_rows();
    }
    const int at = j0 - jt, end = jhi - jt;
    int row[NPF];
#pragma unroll
    for (int u = 0; u < NPF; ++u) row[u] = rows[min(at + krow[u], end)];
    __builtin_amdgcn_sched_barrier(0);   // (all lookups, then the loads: they would go in turns, each waited for)
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      char* to = smem_raw + buf * Z::BYTES + (256 * u + 64 * wave) * 16;
      __builtin_amdgcn_global_load_lds((global_cvoid*)(cache + ((uint64_t)(uint32_t)row[u] * Dk + pcol[u])), (lds_void*)to, 16, 0, 0);
    }
  };
  const int nt = jhi < jlo ? 0 : (jhi - jlo) / KT + 1;
  if (nt > 0) fetch(jlo, 0);

  const int wrow = row0 + wave / HC * 32, myrow = wrow + li;
  const bool rok = myrow < nrows, wave_live = wrow < nrows, all_rows = wrow + 31 < nrows;
  const int64_t tq = rok ? q0 + myrow / H : q0;
  const int hq = rok ? myrow % H : 0;
  const int64_t orow = (int64_t)hq * a.total_q + tq;
  const int prow = rok ? (int)a.positions[tq] : -1;
  const int pw_min = wave_live ? (int)a.positions[q0 + wrow / H] : 0;
  const int pw_max = wave_live ? (int)a.positions[q0 + min(wrow + 31, nrows - 1) / H] : 0;
  // this lane's query fragments: qf[k] = Q[row][16 k + 8 hi .. + 8]. (Rows beyond the last repeat the first; every load is
  // unconditional, so that all are in flight together.)
  bf16x8_t qf[NK];
  const bf16_t* qlat = reinterpret_cast<const bf16_t*>(a.q_lat) + orow * R;
#pragma unroll
  for (int k = 0; k < NLAT; ++k) qf[k] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(qlat + 16 * k + 8 * hi));
  if constexpr (NROT > 0) {
    bf16_t qr[NROT][8];
    float fr[NROT][4];
    const bf16_t* qp = reinterpret_cast<const bf16_t*>(a.q_rot) + tq * a.q_stride + (int64_t)hq * a.q_hstride + 8 * hi;
#pragma unroll
    for (int k = 0; k < NROT; ++k) {
#pragma unroll
      for (int e = 0; e < 8; ++e) qr[k][e] = qp[16 * k + e];
#pragma unroll
      for (int i = 0; i < 4; ++i) fr[k][i] = a.sh.rot_pairs > 0 ? a.sh.inv_freq[min(8 * k + 4 * hi + i, a.sh.rot_pairs - 1)] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < NROT; ++k) {
      float f[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float u = bf2f(qr[k][2 * i]), w = bf2f(qr[k][2 * i + 1]);
        float sn, cs;
        __sincosf((float)prow * fr[k][i], &sn, &cs);
        const bool turned = 8 * k + 4 * hi + i < a.sh.rot_pairs;
        f[2 * i] = turned ? u * cs - w * sn : u;
        f[2 * i + 1] = turned ? w * cs + u * sn : w;
      }
      qf[NLAT + k] = __builtin_bit_cast(bf16x8_t, pack8(f));
    }
  }

  constexpr float LOG2E = 1.4426950408889634f;
  const float sl2 = a.scale * LOG2E;
  const bool has_sink = a.sink != nullptr && rok;
  float m = has_sink ? a.sink[hq] * LOG2E : -1e30f;
  float l = has_sink && hi == 0 ? 1.0f : 0.0f;   // (the sum of this lane's keys)
  f32x16_t o[NO];
#pragma unroll
  for (int db = 0; db < NO; ++db) o[db] = f32x16_t{};
  // K fragments: key li of 32, piece 2 k + hi; V fragments: keys 4 hi .. and 8 + 4 hi .. of 16 (the order in which the weights lie
  // in registers), columns 32 db ..
  const int ksw = Z::swz(li), vrow = 4 * hi + (lane & 15) / 4, vsw = Z::swz(vrow), vsw8 = Z::swz(vrow + 8);
  const int kat = 16 * li * KCH, vat = 16 * vrow * KCH + 8 * (lane & 1), vpc = 4 * NO * (wave % HC) + 2 * (lane >> 4 & 1) + (lane >> 1 & 1);
  // The queries are here. (Without this the compiler waits for them in the loop, behind the next tile's DMA and so for that too.)
  __builtin_amdgcn_s_waitcnt(15 << 8 | 7 << 4);
  for (int i = 0; i < nt; ++i) {
    const int j0 = jlo + i * KT;
    // tile i is in LDS for every wave, and every wave has left the other buffer
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(7 << 4);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (i + 1 < nt) fetch(j0 + KT, (i + 1) & 1);
    const char* ks = smem_raw + (i & 1) * Z::BYTES;
    f32x16_t sc = {};
    constexpr int KG = NK % 2 == 0 ? 2 : 1, NG = NK / KG;   // fragments of KG steps ahead
    static_assert(NG * KG == NK, "whole groups");
    bf16x8_t kf[2][KG];
    auto read_k = [&](int g) {
#pragma unroll
      for (int k = 0; k < KG; ++k)
        kf[g & 1][k] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(ks + kat + 16 * ((2 * (KG * g + k) + hi) ^ ksw)));
    };
    read_k(0);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if (g + 1 < NG) read_k(g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < KG; ++k) sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[g & 1][k], qf[KG * g + k], sc, 0, 0, 0);
    }
    // interior tiles (every key visible to every row of the wave) skip the per-score mask
    const bool inner = all_rows && j0 + KT - 1 <= min(pw_min, jhi) && (a.window <= 0 || pw_max - j0 < a.window);
    if (!inner) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int j = j0 + 8 * (e / 4) + 4 * hi + e % 4;
        const bool valid = rok && j <= jhi && j <= prow && (a.window <= 0 || prow - j < a.window);
        sc[e] = valid ? sc[e] : -INFINITY;
      }
    }
    float mx = sc[0];
#pragma unroll
    for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sc[e]);
    const float mn = fmaxf(m, xor32_max(mx) * sl2);
    if (__builtin_amdgcn_ballot_w64(mn != m) != 0) {   // wave-uniform
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      l *= alpha;
#pragma unroll
      for (int db = 0; db < NO; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[db][e] *= alpha;
      m = mn;
    }
    float sum[2] = {};
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      sc[e] = __builtin_amdgcn_exp2f(fmaf(sc[e], sl2, -m));
      sum[e & 1] += sc[e];
    }
    l += sum[0] + sum[1];
    // 16 keys and VG column blocks a group, fragments of the next group ahead
    constexpr int VG = NO < 2 ? NO : 2, NV = 2 * NO / VG;
    bf16x8_t vf[2][VG];
    auto read_v = [&](int g) {
      const int u = g / (NO / VG), d0 = g % (NO / VG) * VG;
#pragma unroll
      for (int d = 0; d < VG; ++d) {
        const char* at = ks + vat + 256 * KCH * u;
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at + 16 * ((4 * (d0 + d) + vpc) ^ vsw)));
        const short4_t up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at + 128 * KCH + 16 * ((4 * (d0 + d) + vpc) ^ vsw8)));
        vf[g & 1][d] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    read_v(0);
#pragma unroll
    for (int g = 0; g < NV; ++g) {
      const int u = g / (NO / VG), d0 = g % (NO / VG) * VG, e = 8 * (u & 1);
      const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, make_uint4(pack2(sc[e], sc[e + 1]), pack2(sc[e + 2], sc[e + 3]),
                                                                  pack2(sc[e + 4], sc[e + 5]), pack2(sc[e + 6], sc[e + 7])));
      const uint4 h = __builtin_bit_cast(uint4, pf);
      auto rest = [&](int i, uint32_t b) { return rest2(sc[e + i], sc[e + i + 1], b); };
      const bf16x8_t pl = __builtin_bit_cast(bf16x8_t, make_uint4(rest(0, h.x), rest(2, h.y), rest(4, h.z), rest(6, h.w)));
      if (g + 1 < NV) read_v(g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < VG; ++d) o[d0 + d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[g & 1][d], pl, o[d0 + d], 0, 0, 0);
#pragma unroll
      for (int d = 0; d < VG; ++d) o[d0 + d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[g & 1][d], pf, o[d0 + d], 0, 0, 0);
    }
  }
  // results: a row's columns 32 db + 8 q + 4 hi .. in the registers; lanes 32 apart exchange halves, so that each stores 8 columns
  l = xor32_sum(l);
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  bf16_t* op = reinterpret_cast<bf16_t*>(a.out) + orow * R + 32 * NO * (wave % HC) + 8 * hi;
#pragma unroll
  for (int db = 0; db < NO; ++db)
#pragma unroll
    for (int q = 0; q < 16; q += 8) {
      const auto x = __builtin_amdgcn_permlane32_swap(pack2(o[db][q] * inv, o[db][q + 1] * inv), pack2(o[db][q + 4] * inv, o[db][q + 5] * inv), false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(pack2(o[db][q + 2] * inv, o[db][q + 3] * inv), pack2(o[db][q + 6] * inv, o[db][q + 7] * inv), false, false);
      if (rok) *reinterpret_cast<uint4*>(op + 32 * db + 2 * q) = make_uint4(x[0], y[0], x[1], y[1]);
    }
}

template <int NDB, int NROT> hipError_t launch_wide(const LatentAttnArgs& a, hipStream_t s) {
  int log = 1;
  while ((int64_t)1 << log < a.block_size) ++log;
  const uint32_t bs_mul = a.block_size == 1 ? 0 : (uint32_t)(((uint64_t)1 << (31 + log)) / a.block_size + 1);
  const dim3 grid((unsigned)(((int64_t)a.max_q * a.heads + LatentTile<NDB, NROT>::ROWS - 1) / LatentTile<NDB, NROT>::ROWS), (unsigned)a.num_seqs);
  auto* fn = latent_attn_wide_kernel<NDB, NROT>;
  constexpr int lds = LatentTile<NDB, NROT>::LDS;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, grid, dim3(256), lds, s, a, bs_mul, log - 1);
  return hipGetLastError();
}
template <int NDB, int NROT> hipError_t launch_two(const LatentAttnArgs& a, hipStream_t s) {
  int log = 1;
  while ((int64_t)1 << log < a.block_size) ++log;
  const uint32_t bs_mul = a.block_size == 1 ? 0 : (uint32_t)(((uint64_t)1 << (31 + log)) / a.block_size + 1);
  constexpr int ROWS = TwoTile<NDB, NROT>::ROWS, lds = TwoTile<NDB, NROT>::LDS;
  auto* fn = latent_attn_two_kernel<NDB, NROT>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3((unsigned)(((int64_t)a.max_q * a.heads + ROWS - 1) / ROWS), (unsigned)a.num_seqs), dim3(256), lds, s, a, bs_mul, log - 1);
  return hipGetLastError();
}
template <int NDB, int NROT> hipError_t launch_mfma_rq(const LatentAttnArgs& a, hipStream_t s) {
  // floor(j / block_size) = (j * bs_mul) >> (32 + bs_shift) for 31-bit j
  int log = 1;
  while ((int64_t)1 << log < a.block_size) ++log;
  const uint32_t bs_mul = a.block_size == 1 ? 0 : (uint32_t)(((uint64_t)1 << (31 + log)) / a.block_size + 1);
  const dim3 grid((unsigned)(((int64_t)a.max_q * a.heads + 63) / 64), (unsigned)a.num_seqs);
  hipLaunchKernelGGL((latent_attn_mfma_rq_kernel<NDB, NROT>), grid, dim3(256), (RqTile<NDB, NROT>::LDS), s, a, bs_mul, log - 1);
  return hipGetLastError();
}

// the register-query kernel exists for rank in {64, 128, 256} x rot_dim in {0, 16, 32, 64}; unsplit steps only. It writes results
// 16 bytes at a time and passes row numbers between lanes in 32 bits (the other kernel: 8 bytes, 64 bits).
inline bool mfma_rq_fits(const LatentAttnArgs& a) {
  const int r = a.sh.rank, t = a.sh.rot_dim;
  return (int64_t)a.max_q * a.heads > 32 && (r == 64 || r == 128 || r == 256) &&
         (t == 0 || t == 16 || t == 32 || t == 64) && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0 &&
         (int64_t)a.heads * a.total_q < (int64_t(1) << 31);
}

// A workgroup has 64 rows in either kernel. Up to two of them per CU go with 32 rows per wave (whose maxima are taken before the scale: a
// positive one), more with 16, of which three workgroups share a CU and which start faster, for few keys too. 16 / 32 rows per wave, rank 256 + 32, us: 1 x 300 rows of 16 heads
// 23.5 / 17.9, 1 x 1500 behind 400 118 / 78, 8 x 128 14.4 / 12.8; 32 x 30 9.7 / 10.8; 8 x 500 behind 100 50 / 54, 16 x 1024 309 / 324.
inline bool wide_takes(const LatentAttnArgs& a) {
  const int64_t wgs = ((int64_t)a.max_q * a.heads + 63) / 64 * a.num_seqs, keys = (int64_t)a.bt_cols * a.block_size;
  return wgs <= 2 * (int64_t)num_cus() && keys > 64 && a.scale > 0.f;
}
// Two groups of 16 rows per wave: where there is more than one turn of its workgroups (two per CU), and enough keys that starting them, which takes
// longer, doesn't count; in one turn where all sequences have the same rows and see many keys (with others the longest ends alone). One group / two, rank
// 256 + 32, us: 16 x 1024 rows of 16 heads 243 / 193 (the step; the others launched alone, back to back); 8 of 786 - 1000 101 / 89; 32 of 125 - 250, 32 heads 73 / 65; 16 of 200 - 400, 32 heads 67 / 63; 6 x 300 behind
// 300, 32 heads, window 512 63 / 47; 8 x 500 behind 300 73 / 61; 4 x 1000 70 / 66. Not: 4 of 889 - 1000 70 / 74; 32 x 200 39 / 42; 32 of 50 - 100 behind 150 - 300
// 33 / 37; 24 x 100 19 / 19. (58 random steps that it takes: 0.88 of the time, one slower by more than 1 %, 18 of up to 243 rows of 12 heads in tables ten times as wide 27 / 29, as
// the tables' width stands for the keys.) Without a rotary part, or with one of 64 (13 registers in scratch), the gain is 2 - 10 % smaller: twice the work.
inline bool two_takes(const LatentAttnArgs& a) {
  const int64_t cus = num_cus(), wgs = (int64_t)a.total_q * a.heads / 128, keys = (int64_t)a.bt_cols * a.block_size - a.max_q / 2;
  const int64_t seen = a.window > 0 ? std::min<int64_t>(keys, a.window) : keys;   // by a row, about
  if (a.sh.rank != 256 || !(a.scale > 0.f) || seen < 1) return false;
  if (wgs > 2 * cus && wgs * seen >= (a.sh.rot_dim == 16 || a.sh.rot_dim == 32 ? 680 : 1360) * cus) return true;
  return (int64_t)a.max_q * a.num_seqs == a.total_q && 4 * wgs > 5 * cus && seen >= 400;
}
template <int NDB, int NROT> hipError_t launch_rows(const LatentAttnArgs& a, hipStream_t s) {
  if (wide_takes(a)) return launch_wide<NDB, NROT>(a, s);
  if constexpr (NDB == 8)
    if (two_takes(a)) return launch_two<NDB, NROT>(a, s);
  return launch_mfma_rq<NDB, NROT>(a, s);
}
template <int NDB> hipError_t launch_mfma_rq_rot(const LatentAttnArgs& a, hipStream_t s) {
  switch (a.sh.rot_dim) {
    case 0: return launch_rows<NDB, 0>(a, s);   // no rotary part: latents without positions
    case 16: return launch_rows<NDB, 1>(a, s);
    case 32: return launch_rows<NDB, 2>(a, s);
    case 64: return launch_rows<NDB, 4>(a, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_mfma_rq_any(const LatentAttnArgs& a, hipStream_t s) {
  switch (a.sh.rank) {
    case 64: return launch_mfma_rq_rot<2>(a, s);
    case 128: return launch_mfma_rq_rot<4>(a, s);
    case 256: return launch_mfma_rq_rot<8>(a, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_mfma_any(const LatentAttnArgs& a, hipStream_t s) {
  if (decode_fits(a)) return launch_decode_any(a, s);
  if (a.impl != 3 && a.nsplit <= 1 && mfma_rq_fits(a)) return launch_mfma_rq_any(a, s);
  // one wave per workgroup when a sequence brings at most 32 rows (decode steps of other widths): small LDS, many workgroups
  return (int64_t)a.max_q * a.heads <= 32 ? launch_mfma_ndb<1>(a, s) : launch_mfma_ndb<4>(a, s);
}

constexpr int LDS_MAX = 128 * 1024;

inline size_t lds_bytes(int bk, int qs, int ksd) { return sizeof(float) * ((size_t)RW * qs + (size_t)bk * ksd + (size_t)RW * bk); }

template <int BK, int CC, bool F32>
hipError_t launch_one(const LatentAttnArgs& a, int qs, int ksd, dim3 grid, hipStream_t s) {
  static bool attr_set = false;  // once per instantiation; hipFuncSetAttribute is not a stream operation
  auto* fn = latent_attn_kernel<BK, CC, F32>;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       LDS_MAX);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL(fn, grid, dim3(256), lds_bytes(BK, qs, ksd), s, a, qs, ksd);
  return hipGetLastError();
}

template <int BK, bool F32>
hipError_t launch_cc(const LatentAttnArgs& a, int qs, int ksd, dim3 grid, hipStream_t s) {
  const int r = a.sh.rank;
  if (r <= 128) return launch_one<BK, 2, F32>(a, qs, ksd, grid, s);
  if (r <= 512) return launch_one<BK, 8, F32>(a, qs, ksd, grid, s);
  if (r <= 1024) return launch_one<BK, 16, F32>(a, qs, ksd, grid, s);
  return hipErrorInvalidValue;
}

template <bool F32> hipError_t launch_bk(const LatentAttnArgs& a, hipStream_t s) {
  const int dk = a.sh.rank + a.sh.rot_dim;
  const int qs = (dk + 3) & ~3, ksd = dk | 1;
  const dim3 grid((unsigned)(((int64_t)a.max_q * a.heads + RW - 1) / RW), (unsigned)a.num_seqs);
  if (lds_bytes(64, qs, ksd) <= 64 * 1024) return launch_cc<64, F32>(a, qs, ksd, grid, s);
  if (lds_bytes(32, qs, ksd) <= LDS_MAX) return launch_cc<32, F32>(a, qs, ksd, grid, s);
  if (lds_bytes(16, qs, ksd) <= LDS_MAX) return launch_cc<16, F32>(a, qs, ksd, grid, s);
  return hipErrorInvalidValue;
}

}  // namespace

bool latent_attn_uses_mfma(const LatentAttnArgs& a) { return a.impl != 1 && mfma_ok(a); }
bool latent_attn_decodes(const LatentAttnArgs& a) { return decode_fits(a); }
bool latent_attn_fits_rows(const LatentAttnArgs& a) { return latent_attn_uses_mfma(a) && a.impl != 3 && mfma_rq_fits(a); }

const char* latent_attn_form(const LatentAttnArgs& a) {
  if (!latent_attn_uses_mfma(a)) return "fma";
  return a.impl != 3 && a.nsplit <= 1 && mfma_rq_fits(a) ? "rows" : a.nsplit > 1 ? "split" : "tiles";
}

const char* latent_attn_kernel(const LatentAttnArgs& a) {
  if (decode_fits(a)) return "decode";
  const char* form = latent_attn_form(a);
  if (form[0] == 'r' && wide_takes(a)) return "wide";
  if (form[0] == 'r' && two_takes(a)) return "two rows";
  return form[0] == 's' && a.fine ? "fine split" : form;
}

hipError_t launch_latent_attn(const LatentAttnArgs& a, hipStream_t s) {
  if (a.num_seqs == 0 || a.total_q == 0) return hipSuccess;
  if (a.heads < 1 || a.sh.rank < 1 || a.sh.rot_dim < 0 || a.sh.rot_pairs * 2 > a.sh.rot_dim || a.block_size < 1 ||
      a.max_q < 1)
    return hipErrorInvalidValue;
  if (a.impl != 1 && mfma_ok(a)) return launch_mfma_any(a, s);
  if (a.impl >= 2) return hipErrorInvalidValue;  // the matrix-core form was demanded and does not apply
  return a.f32 ? launch_bk<true>(a, s) : launch_bk<false>(a, s);
}

}  // namespace die
