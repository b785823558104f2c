// S[c, :] <- exp(d A[c, :]) S[c, :] + d x B; y = S[c, :] . C + D x; y * silu(z) for channels of 9 - 16 states (gfx950).
//
// A channel's 16 states (zero beyond N) lie on LPC = 4 or 16 lanes. A trip is 16 tokens. What depends on token and channel only (step
// size, gate, input) is formed once, by the lane that owns the token (tokens own place modulo LPC), and reaches the channel's other
// lanes as a DPP operand of the products that take it; the read-outs of LPC tokens are summed over the lanes together, halving what
// is kept at each step, so that every lane ends with its own token's sum and stores it. B and C are staged in LDS as fp32, two buffers,
// one barrier per trip; the next trip's loads are in flight during the current one.
//
// Bound by vector issue: per token and 64 channels 16 exponentials, 64 multiply-adds and products, with 4 lanes some 50, with 16 some 130
// instructions beside them. Against whole rows of tokens formed by every lane, loads waited for at each trip (us, 4096 channels of 16
// states, before -> after): 1 x 1024 tokens 381 -> 55, 2 x 1024 382 -> 83, 4 x 1024 384 -> 134, 8 x 1024 436 -> 182, 16 x 1024 482 -> 316 (issue
// alone: some 270), 32 x 17 21.7 -> 18.3; one row each of 18 / 64 sequences, 8192 channels 18.1 -> 7.9, 43.8 -> 21.3 (3.2 TB/s of states).
#include "common.h"
#include "lane_reduce.h"
#include "selective_scan.h"

namespace die {

namespace {

constexpr int TB = 16;   // tokens of a trip
constexpr int NT = 256;
constexpr int BT = 20;   // pitch of a state's tokens in LDS (16 lanes): 16-byte reads of 8 lanes fall on different banks

template <bool FAST> struct Stored { using T = bf16_t; };
template <> struct Stored<false> { using T = float; };
__device__ __forceinline__ float value(bf16_t x) { return bf2f(x); }
__device__ __forceinline__ float value(float x) { return x; }

template <int CTRL> __device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
// of lane E of the own group of LPC lanes
template <int LPC, int E> __device__ __forceinline__ float of_lane(float x) { return dpp<LPC == 4 ? E * 0x55 : 0x150 + E>(x); }

// silu(z) and exp(d A): bf16 steps use the hardware's exponential and reciprocal, A holding log2(e) A
template <bool FAST> __device__ __forceinline__ float silu_of(float z) {
  if constexpr (FAST)
    return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z));
  else
    return z / (1.0f + expf(-z));
}
template <bool FAST> __device__ __forceinline__ float decay_of(float da) {
  if constexpr (FAST)
    return __builtin_amdgcn_exp2f(da);
  else
    return expf(da);
}
constexpr float LOG2E = 1.4426950408889634f;

// v[0 .. 2 N) -> v[0 .. N): of the lane's half of the tokens, summed with the mirrored lane, which keeps the other half
template <int N, int CTRL> __device__ __forceinline__ void halve(float* v, bool upper) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float keep = upper ? v[i + N] : v[i], give = upper ? v[i] : v[i + N];
    v[i] = keep + dpp<CTRL>(give);
  }
}

template <int NP> __device__ __forceinline__ void load_states(const float* p, int n0, int N, bool ok, float* to) {
  if constexpr (NP == 4) {
    if (N % 4 == 0) {
      const float4 v = ok && n0 < N ? *reinterpret_cast<const float4*>(p + n0) : make_float4(0.f, 0.f, 0.f, 0.f);
      to[0] = v.x, to[1] = v.y, to[2] = v.z, to[3] = v.w;
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) to[i] = ok && n0 + i < N ? p[n0 + i] : 0.f;
}
template <int NP> __device__ __forceinline__ void store_states(float* p, int n0, int N, const float* v) {
  if constexpr (NP == 4) {
    if (N % 4 == 0) {
      if (n0 < N) *reinterpret_cast<float4*>(p + n0) = make_float4(v[0], v[1], v[2], v[3]);
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (n0 + i < N) p[n0 + i] = v[i];
}

template <int LPC, bool FAST>
__global__ void __launch_bounds__(NT) scan_lanes_kernel(SelectiveScanArgs a, RaggedRows r, int blocks, int per_xcd) {
  using T = typename Stored<FAST>::T;
  constexpr int NP = 16 / LPC, CH = NT / LPC, OWN = TB / LPC;
  __shared__ __attribute__((aligned(16))) float bc[2][2][LPC == 4 ? TB * 16 : 16 * BT];   // B, C of two trips
  const int s = blockIdx.y, tid = threadIdx.x;
  // (16 lanes: neighbouring blocks share the cache lines of x, dt, z and out, so they run on the same XCD)
  const int cb = per_xcd > 0 ? (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  const int part = tid % LPC, c = cb * CH + tid / LPC;
  const int I = a.I, N = a.N;
  const int q0 = __builtin_amdgcn_readfirstlane(r.cu_q[s]), L = __builtin_amdgcn_readfirstlane(r.cu_q[s + 1]) - q0;
  if (L <= 0 || cb >= blocks) return;
  const bool live = c < I;
  const int cc = live ? c : I - 1;
  const T* xp = reinterpret_cast<const T*>(a.x) + (int64_t)q0 * a.xstride + cc;
  const T* dp = reinterpret_cast<const T*>(a.dt) + (int64_t)q0 * a.dtstride + cc;
  const T* zp = reinterpret_cast<const T*>(a.z) + (int64_t)q0 * a.zstride + cc;
  const int bt = tid / 16, bn = tid % 16;   // the token and state whose B and C this thread stages
  const T* bp = reinterpret_cast<const T*>(a.bc) + (int64_t)q0 * a.bcstride + min(bn, N - 1);
  T xr[OWN], dr[OWN], zr[OWN], br, cr;
  const T *const xl = xp + part * a.xstride, *const dl = dp + part * a.dtstride, *const zl = zp + part * a.zstride, *const bl = bp + bt * a.bcstride;
  auto fetch = [&](int64_t t0) {
    const int last = L - 1 - (int)t0;
    const T* p;
    if (last >= TB - 1) {   // (the lane's rows by one address and the same offsets for all lanes)
#pragma unroll
      for (int o = 0; o < OWN; ++o) {
        xr[o] = xl[(t0 + LPC * o) * a.xstride];
        dr[o] = dl[(t0 + LPC * o) * a.dtstride];
        zr[o] = zl[(t0 + LPC * o) * a.zstride];
      }
      p = bl + t0 * a.bcstride;
    } else {
#pragma unroll
      for (int o = 0; o < OWN; ++o) {
        const int64_t row = t0 + min(LPC * o + part, last);
        xr[o] = xp[row * a.xstride];
        dr[o] = dp[row * a.dtstride];
        zr[o] = zp[row * a.zstride];
      }
      p = bp + (t0 + min(bt, last)) * a.bcstride;
    }
    br = p[a.boff];
    cr = p[a.coff];
  };
  fetch(0);
  const bool fresh = r.positions[q0] <= 0;
  float* st = a.state + ((int64_t)r.state_slots[s] * I + cc) * N;
  float S[NP], A[NP];
  load_states<NP>(st, part * NP, N, !fresh, S);
  load_states<NP>(a.A + (int64_t)cc * N, part * NP, N, true, A);
  if (FAST) {
#pragma unroll
    for (int i = 0; i < NP; ++i) A[i] *= LOG2E;
  }
  const float Dc = a.D[cc], dtb = a.dt_bias[cc];
  const bool up8 = part & 8, up4 = part & 4, up2 = part & 2, up1 = part & 1;
  const int put = LPC == 4 ? bt * 16 + bn : bn * BT + bt;
  T* out = reinterpret_cast<T*>(a.out) + (int64_t)q0 * I + cc;

  auto trip = [&](int t0, auto whole) {
    constexpr bool WHOLE = decltype(whole)::value != 0;
    const int nb = L - t0;
    const float* Bs = bc[t0 / TB % 2][0];
    const float* Cs = bc[t0 / TB % 2][1];
    const_cast<float*>(Bs)[put] = bn < N ? value(br) : 0.f;
    const_cast<float*>(Cs)[put] = bn < N ? value(cr) : 0.f;
    float d[OWN], dx[OWN], w[OWN], g[OWN], y[TB];
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const float x = value(xr[o]);
      d[o] = softplus_of<FAST>(value(dr[o]) + dtb);
      dx[o] = d[o] * x;
      w[o] = Dc * x;
      g[o] = silu_of<FAST>(value(zr[o]));
    }
    __syncthreads();
    if (t0 + TB < L) fetch(t0 + TB);
    if constexpr (LPC == 4) {
      static_for<OWN>([&](auto o) {
        static_for<4>([&](auto e) {
          constexpr int O = o.value, t = 4 * O + e.value;
          if (WHOLE || t < nb) {
            const f32x4_t b = *reinterpret_cast<const f32x4_t*>(Bs + t * 16 + 4 * part);
            const f32x4_t q = *reinterpret_cast<const f32x4_t*>(Cs + t * 16 + 4 * part);
            float p = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              S[i] = fmaf(decay_of<FAST>(of_lane<4, e.value>(d[O]) * A[i]), S[i], of_lane<4, e.value>(dx[O]) * b[i]);
              p = i == 0 ? S[i] * q[i] : fmaf(S[i], q[i], p);
            }
            y[t] = p;
          } else {
            y[t] = 0.f;
          }
        });
        halve<2, 0x1B>(y + 4 * o.value, up2);
        halve<1, 0xB1>(y + 4 * o.value, up1);
        y[o.value] = y[4 * o.value];
      });
    } else {
      static_for<4>([&](auto o) {
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(Bs + part * BT + 4 * o.value);
        const f32x4_t q = *reinterpret_cast<const f32x4_t*>(Cs + part * BT + 4 * o.value);
        static_for<4>([&](auto e) {
          constexpr int t = 4 * o.value + e.value;
          if (WHOLE || t < nb) {
            S[0] = fmaf(decay_of<FAST>(of_lane<16, t>(d[0]) * A[0]), S[0], of_lane<16, t>(dx[0]) * b[e.value]);
            y[t] = S[0] * q[e.value];
          } else {
            y[t] = 0.f;
          }
        });
      });
      halve<8, 0x140>(y, up8);
      halve<4, 0x141>(y, up4);
      halve<2, 0x1B>(y, up2);
      halve<1, 0xB1>(y, up1);
    }
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int t = LPC * o + part;
      if (live && (WHOLE || t < nb)) {
        const float v = (y[o] + w[o]) * g[o];
        T* to = out + (int64_t)(t0 + t) * I;
        if constexpr (FAST)
          *to = f2bf(v);
        else
          *to = v;
      }
    }
  };
  int t0 = 0;
  for (; t0 + TB <= L; t0 += TB) trip(t0, IntC<1>{});
  if (t0 < L) trip(t0, IntC<0>{});
  if (live) store_states<NP>(st, part * NP, N, S);
}

// One row per sequence: a channel's states on 4 lanes, read and written as they lie.
template <bool FAST> __global__ void __launch_bounds__(NT) scan_step_kernel(SelectiveScanArgs a, RaggedRows r) {
  using T = typename Stored<FAST>::T;
  const int s = blockIdx.y, part = threadIdx.x % 4, c = blockIdx.x * (NT / 4) + threadIdx.x / 4;
  const int I = a.I, N = a.N;
  const bool live = c < I;
  const int cc = live ? c : I - 1;
  float* st = a.state + ((int64_t)r.state_slots[s] * I + cc) * N;
  const bool fresh = r.positions[s] <= 0;
  float S[4], A[4];
  load_states<4>(st, part * 4, N, true, S);   // (a new sequence reads its slot but not its content)
  load_states<4>(a.A + (int64_t)cc * N, part * 4, N, true, A);
  const float x = value(reinterpret_cast<const T*>(a.x)[(int64_t)s * a.xstride + cc]);
  const float z = value(reinterpret_cast<const T*>(a.z)[(int64_t)s * a.zstride + cc]);
  const float d = softplus_of<FAST>(value(reinterpret_cast<const T*>(a.dt)[(int64_t)s * a.dtstride + cc]) + a.dt_bias[cc]);
  const T* bc = reinterpret_cast<const T*>(a.bc) + (int64_t)s * a.bcstride;
  const float dx = d * x;
  float p = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = 4 * part + i;
    const float b = n < N ? value(bc[a.boff + n]) : 0.f, q = n < N ? value(bc[a.coff + n]) : 0.f;
    S[i] = fmaf(decay_of<FAST>(d * (FAST ? A[i] * LOG2E : A[i])), fresh ? 0.f : S[i], dx * b);
    p = fmaf(S[i], q, p);
  }
  p = group_sum<4>(p);
  if (!live) return;
  store_states<4>(st, part * 4, N, S);
  if (part == 0) {
    const float v = (p + a.D[cc] * x) * silu_of<FAST>(z);
    T* to = reinterpret_cast<T*>(a.out) + (int64_t)s * I + c;
    if constexpr (FAST)
      *to = f2bf(v);
    else
      *to = v;
  }
}

template <bool FAST> hipError_t launch_scan(const SelectiveScanArgs& a, RaggedRows r, hipStream_t s) {
  if (r.cu_q == nullptr) {
    hipLaunchKernelGGL((scan_step_kernel<FAST>), dim3((a.I + 63) / 64, r.num_seqs), dim3(NT), 0, s, a, r);
    return hipGetLastError();
  }
  // 16 lanes while 4 would leave SIMDs without a wave (4 sequences of 1024 tokens and 4096 channels: 134 us on 16 lanes; 8: 182 on 4, where
  // 16 lanes' instructions alone take some 250)
  const int64_t lanes = (int64_t)a.I * r.num_seqs * 4, simds = 4 * (int64_t)num_cus();
  if (lanes <= 64 * simds) {
    const int blocks = (a.I + 15) / 16;
    hipLaunchKernelGGL((scan_lanes_kernel<16, FAST>), dim3((blocks + 7) / 8 * 8, r.num_seqs), dim3(NT), 0, s, a, r, blocks, (blocks + 7) / 8);
  } else {
    const int blocks = (a.I + 63) / 64;
    hipLaunchKernelGGL((scan_lanes_kernel<4, FAST>), dim3(blocks, r.num_seqs), dim3(NT), 0, s, a, r, blocks, 0);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_scan_lanes(const SelectiveScanArgs& a, RaggedRows r, hipStream_t s) {
  return a.f32 ? launch_scan<false>(a, r, s) : launch_scan<true>(a, r, s);
}

}  // namespace die
