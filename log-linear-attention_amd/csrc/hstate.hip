// Recurrent (decode) path of log-linear attention for gfx950: token steps of the
// Fenwick level state HState and the prefill of its low levels.
//
// Replaces hattention_step / step_state / step_output (hattention/kernel.py:577-633,
// recurrent.py:9-166), the token loops around them (hattention_recurrent, the tail
// and the low levels of a prefill, kernel.py:438-449, 555-570) and the MAMBA2 fast
// path of postprocess_prefill_hstate_ (kernel.py:378-465).  The reference runs a
// torch einsum per level and a Python loop over levels that reads device counts
// back to the host at every level (recurrent.py:42-54); here the cascades are
// planned on the host from a host copy of the counts (the counts depend only on
// the step number) and any number of tokens, including GDELTA's l2norm of q and k
// and the Mamba-2 layer's pre- and post-processing, is one launch.
//
// States: fp32 [B, H, K, V, L] (level innermost), the reference's HState layout.
//
// A step with cascade depth c (levels 0 .. c-1 are full and cascade upwards,
// recurrent.py:42-54) is, per (k, v):
//   S[c] += S[0] + ... + S[c-1];  S[0 .. c-1] = 0           (cascade_weak)
//   MAMBA2: S[l] *= exp(g)                                   (insert, :88-89)
//   GDELTA: S[l] <- exp(g) (S[l] - beta k (k^T S[l]))        (insert, :90-91; step_state :146-154)
//   S[0] = k v^T (MAMBA2) or beta k v^T (GDELTA)             (insert, :93)
//   o[v] = sum_k q[k] sum_l lambda[l] S[k][v][l]              (step_output, :159-166)
#include <hip/hip_runtime.h>

#include <numeric>
#include <type_traits>

#include "common.h"
#include "hstate.h"
#include "layer_math.h"

namespace hattn {

constexpr int kHsCols = 16;   // value columns per workgroup of the prefill levels
constexpr int kHsRowGroups = 256 / kHsCols;

// The level counts (shared by all rows) after the step: the cascade (weak: levels
// 0 .. c-1 merge into level c; strong: levels 0 .. m-1 move up one level, m - 1
// merging into m), then one more token at level 0.
__device__ inline void cascade_counts(int* counts, int L, int cascade, int strong) {
  if (strong) {
    int prev = 0;
    for (int e = 0; e < L; ++e) {
      const int cur = counts[e];
      counts[e] = e == 0 ? 0 : (e < cascade ? prev : (e == cascade ? cur + prev : cur));
      prev = cur;
    }
  } else {
    int moved = 0;
    for (int e = 0; e < cascade; ++e) {
      moved += counts[e];
      counts[e] = 0;
    }
    if (cascade > 0) counts[cascade] += moved;
  }
  counts[0] += 1;
}

// Element u + i, i < n, of a tensor with dtype code dt (0 bf16, 2 fp32); p, u and dt
// are uniform.  Through a buffer descriptor: a lane keeps a 32-bit offset and no
// address, and reads 0 from n on.
__device__ __forceinline__ float hs_ld(const void* p, long long u, unsigned int i, int dt,
                                       int n = 1) {
  const int es = dt == 0 ? 2 : 4;
  const rsrc_t r = make_rsrc((const char*)p + u * es, (size_t)n * es);
  return dt == 0 ? (float)buf_load<__bf16>(r, 2 * i, 0) : buf_load<float>(r, 4 * i, 0);
}
__device__ __forceinline__ void hs_st(void* p, long long u, unsigned int i, float x, int dt) {
  if (dt == 0) ((__bf16*)p + u)[i] = (__bf16)x;
  else ((float*)p + u)[i] = x;
}
__device__ __forceinline__ float hs_round(float x, int dt) { return dt == 0 ? (float)(__bf16)x : x; }

__device__ __forceinline__ float wave_sum(float x) {
  x = row_sum16(x);
  x += __shfl_xor(x, 16, 64);
  x += __shfl_xor(x, 32, 64);
  return x;
}
// lane i gets lane i - 1's value, lane 0 gets 0 (wave_shr:1)
__device__ __forceinline__ float lane_before(float x) { return dpp_f32<0x138, 0xf, true>(0.f, x); }
__device__ __forceinline__ float lane_value(float x, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}

// Token steps with the state in registers.
//
// A workgroup owns VB value columns of one (b, h): for every row k the VB * LA
// contiguous floats [v][level].  Lane n of each wave holds the NV elements from
// NV n on, of the wave's R rows (blockDim = 64 ceil(K / R)), from one load per row
// to one store per row, however many tokens are stepped in between; so the state
// moves through HBM once, in whole lines, with R loads in flight per lane.  (Staged
// through LDS and one launch a token, this took 109 us for a GDELTA step of B 4, H
// 16, K = V = 128, L 18, and 14 us for each of the 64 tokens that rebuild the low
// levels after a prefill.)
//   cascade   S[c] += S[0 .. c-1] is a sum over the c elements before S[c] in the
//             flat [v][level] order: a shift along the lanes.
//   u = k^T S, w = q^T S   sums over a wave's rows in registers (k, q of a row are
//             wave-uniform: readlane), then over the waves through LDS, double
//             buffered, so one barrier a token.
//   update    S = a S - k (a beta u), level 0 = k (beta v)
//   output    q^T S after the update = a (w - beta (q . k) u) per level, and
//             (q . k) beta v at level 0; the first wave weights and sums the levels.
// The next token's operands are loaded before the current token is computed.
// (STRONG is an instance of its own: the two cascades in one kernel cost 70 spilled
// registers.)  NV (elements per lane) sets the number of workgroups: the host takes the widest
// that still fills the chip.
template <int KIND, int NV, int R, bool STRONG, int KMAX>
__global__ __launch_bounds__(64 * KMAX / R) void hstate_steps_kernel(const HsArgs p) {
  extern __shared__ float red[];     // [2][u, w][wave][64 NV]
  __shared__ float part[64 * NV];    // weighted levels of the output, first wave only
  typedef float vecN __attribute__((ext_vector_type(NV)));
  constexpr bool GDN = KIND == kHsGdelta, LAYER = KIND == kHsLayer;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = blockDim.x >> 6;
  const int bh = blockIdx.x, b = bh / p.H, h = bh - b * p.H, gq = h / (p.H / p.G);
  const int K = p.K, V = p.V, L = p.L, LA = p.LA;
  const int v0 = blockIdx.y * p.VB, vbc = p.VB < V - v0 ? p.VB : V - v0;
  const bool act = lane * NV < vbc * LA;
  const int e0 = act ? lane * NV : 0;
  const int vv0 = e0 / LA, ll0 = e0 - vv0 * LA;
  int ll[NV];
  int vi = v0 + vv0;   // column of this lane's level-0 element, if it has one
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    ll[i] = ll0 + i >= LA ? ll0 + i - LA : ll0 + i;
    if (i > 0 && ll[i] == 0) ++vi;
  }
  if (vi >= V) vi = V - 1;   // a lane at the end that has none
  // elements are contiguous unless only the first LA of L levels are stepped
  // (NV = 1 then)
  const unsigned int at0 = LA == L ? e0 : vv0 * L + ll0;
  const int row0 = wave * R, klane = row0 & 63;
  // (a uniform row address and a 32-bit lane offset: no address registers per row)
  float* base = p.states + (((size_t)bh * K + row0) * V + v0) * L;
  const int rstride = V * L;

  float s[R][NV];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    vecN x{};
    if (!p.zero && row0 + r < K) x = *(const vecN*)(base + r * rstride + at0);
    if constexpr (NV == 1) s[r][0] = x[0];
    else
#pragma unroll
      for (int i = 0; i < NV; ++i) s[r][i] = x[i];
  }

  struct Token {
    float k[4], q[4], g, beta, v, lam[NV], x;
  };
  const HsLayer& y = p.layer;
  auto fetch = [&](int i0) {
    Token n;
    const int t = p.t0 + i0;
    const long long qo = b * p.q_b + t * p.q_t + gq * K, so = b * p.s_b + t * p.s_t + h;
    const long long vo = b * p.v_b + t * p.v_t + h * V, lo = b * p.l_b + t * p.l_t + h * L;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = lane + 64 * j;
      n.k[j] = p.update && 64 * j < K ? hs_ld(p.k, qo, i, p.dt_qk, K) : 0.f;
      n.q[j] = p.output && 64 * j < K ? hs_ld(p.q, qo, i, p.dt_qk, K) : 0.f;
    }
    n.beta = GDN && p.update ? hs_ld(p.beta, so, 0, p.dt_b) : 1.f;
    n.x = 0.f;
    n.v = p.update ? hs_ld(p.v, vo, vi, LAYER ? y.dt_x : p.dt_v, V) : 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) n.lam[i] = p.output ? hs_ld(p.l, lo, ll[i], p.dt_l, L) : 0.f;
    if (LAYER) {
      // the Mamba-2 layer's inputs: v = x dt', g = A dt', lambda of (L, dl), each
      // rounded to its dtype as the separate layer kernels do
      const float d = layer_dtp(hs_ld(y.dt, so, 0, y.dt_dt),
                                y.bias ? hs_ld(y.bias, h, 0, y.dt_bias) : 0.f, y.softplus);
      n.g = layer_g(hs_ld(y.A, h, 0, y.dt_A), d);
      n.v = hs_round(n.v * d, p.dt_v);
#pragma unroll
      for (int i = 0; i < NV; ++i)
        n.lam[i] = hs_round(lambda_of(hs_ld(y.Lp, h * L, ll[i], y.dt_Lp, L), n.lam[i], y.mode), y.dt_lam);
      if (y.D) n.x = hs_ld(p.v, vo, v0 + lane, y.dt_x, V);
    } else {
      n.g = p.update ? p.g[so] : 0.f;
    }
    return n;
  };

  Token nx = fetch(0);
  for (int t = 0; t < p.T; ++t) {
    Token tk = nx;
    if (t + 1 < p.T) nx = fetch(t + 1);
    if (p.norm) {
      // q / |q| * scale, k / |k| (kernel.py:20-23, 626-629 with the eps of fla's
      // l2norm), rounded to the input dtype after the norm and after the scale, as
      // the reference's l2norm_fwd / l2norm_and_scale_fwd store their outputs
      float nq = 0.f, nk = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        nq += tk.q[j] * tk.q[j];
        nk += tk.k[j] * tk.k[j];
      }
      const float rq = rsqrtf(wave_sum(nq) + 1e-6f), rk = rsqrtf(wave_sum(nk) + 1e-6f);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        tk.q[j] = hs_round(hs_round(tk.q[j] * rq, p.dt_qk) * p.scale, p.dt_qk);
        tk.k[j] = hs_round(tk.k[j] * rk, p.dt_qk);
      }
    }
    float qk = 0.f;
    if (p.output && p.update) {
#pragma unroll
      for (int j = 0; j < 4; ++j) qk += tk.q[j] * tk.k[j];
      qk = wave_sum(qk);
    }
    const int kj = row0 >> 6;
    const float kr = kj == 0 ? tk.k[0] : kj == 1 ? tk.k[1] : kj == 2 ? tk.k[2] : tk.k[3];
    const float qr = kj == 0 ? tk.q[0] : kj == 1 ? tk.q[1] : kj == 2 ? tk.q[2] : tk.q[3];

    if (p.update) {
      const int c = p.casc[t];
      bool keep[NV], into[NV];
      if (STRONG) {
        // cascade_strong (recurrent.py:56-74) with merge level c: levels 0 .. c-1
        // move up one level, c - 1 merging into c (c = L: the top level's content
        // leaves the state); level 0 ends empty
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          keep[i] = ll[i] >= c && ll[i] > 0;
          into[i] = ll[i] <= c && ll[i] > 0;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const float before = lane_before(s[r][NV - 1]);
#pragma unroll
          for (int i = NV - 1; i >= 0; --i)
            s[r][i] = (keep[i] ? s[r][i] : 0.f) + (into[i] ? (i > 0 ? s[r][i > 0 ? i - 1 : 0] : before) : 0.f);
        }
      } else {
        // cascade_weak: level 0 ends empty too (at c = 0 the insert overwrites it)
        int at = c - ll0;           // this lane's element of level c, if it has one
        if (at < 0) at += LA;
        const bool has = at < NV;
        const int lim = has ? c - at : -(1 << 20);
        bool own[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          keep[i] = ll[i] >= c && ll[i] > 0;
          into[i] = i == at;
          own[i] = has && i < at && at - i <= c;
        }
        const int far = (c + NV - 1) / NV;   // lanes before that hold levels below c
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float sum = 0.f, cur[NV];
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            sum += own[i] ? s[r][i] : 0.f;
            cur[i] = s[r][i];
          }
          for (int d = 1; d <= far; ++d)
#pragma unroll
            for (int i = 0; i < NV; ++i) {
              cur[i] = lane_before(cur[i]);
              sum += NV * d - i <= lim ? cur[i] : 0.f;
            }
#pragma unroll
          for (int i = 0; i < NV; ++i)
            s[r][i] = (keep[i] ? s[r][i] : 0.f) + (into[i] && c > 0 ? sum : 0.f);
        }
      }
    }

    float u[NV], w[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) u[i] = w[i] = 0.f;
    const bool need_u = GDN && p.update;
    if (need_u)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float kk = lane_value(kr, klane + r);
#pragma unroll
        for (int i = 0; i < NV; ++i) u[i] += kk * s[r][i];
      }
    if (p.output)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float qq = lane_value(qr, klane + r);
#pragma unroll
        for (int i = 0; i < NV; ++i) w[i] += qq * s[r][i];
      }
    float* ru = red + (size_t)(t & 1) * 2 * nw * 64 * NV;
    float* rw = ru + nw * 64 * NV;
    if (need_u || p.output) {
      vecN x;
      if (need_u) {
        if constexpr (NV == 1) x = u[0];
        else
#pragma unroll
          for (int i = 0; i < NV; ++i) x[i] = u[i];
        *(vecN*)(ru + (wave * 64 + lane) * NV) = x;
      }
      if (p.output) {
        if constexpr (NV == 1) x = w[0];
        else
#pragma unroll
          for (int i = 0; i < NV; ++i) x[i] = w[i];
        *(vecN*)(rw + (wave * 64 + lane) * NV) = x;
      }
      __syncthreads();
      if (need_u) {
        vecN acc{};
        for (int j = 0; j < nw; ++j) acc += *(const vecN*)(ru + (j * 64 + lane) * NV);
        if constexpr (NV == 1) u[0] = acc[0];
        else
#pragma unroll
          for (int i = 0; i < NV; ++i) u[i] = acc[i];
      }
    }

    const float a = p.update ? __expf(tk.g) : 1.f;
    if (p.output && wave == 0) {
      vecN acc{};
      for (int j = 0; j < nw; ++j) acc += *(const vecN*)(rw + (j * 64 + lane) * NV);
      if constexpr (NV == 1) w[0] = acc[0];
      else
#pragma unroll
        for (int i = 0; i < NV; ++i) w[i] = acc[i];
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        float z = w[i];
        if (p.update) {
          z = GDN ? a * (z - tk.beta * qk * u[i]) : a * z;
          if (ll[i] == 0) z = qk * (tk.beta * tk.v);
        }
        if (act) part[e0 + i] = tk.lam[i] * z;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if (lane < vbc) {
        float z = 0.f;
        for (int e = 0; e < LA; ++e) z += part[lane * LA + e];
        const long long oo = b * p.o_b + (p.t0 + t) * p.o_t + h * V + v0;
        if (LAYER) {
          z = hs_round(z, p.dt_v);
          if (y.D) z = layer_out(z, tk.x, hs_ld(y.D, h, 0, y.dt_D));
        }
        hs_st(p.o, oo, lane, z, LAYER ? y.dt_out : p.dt_v);
      }
      __builtin_amdgcn_wave_barrier();
    }

    if (p.update) {
      float m[NV], kr2 = kr;
      asm("" : "+v"(kr2));   // read the rows' k again instead of holding R scalars
#pragma unroll
      for (int i = 0; i < NV; ++i) m[i] = ll[i] == 0 ? tk.beta * tk.v : -(a * tk.beta) * u[i];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float kk = lane_value(kr2, klane + r);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          if (GDN) s[r][i] = __builtin_fmaf(kk, m[i], a * s[r][i]);
          else s[r][i] = ll[i] == 0 ? kk * m[i] : a * s[r][i];
        }
      }
    }
  }

  if (p.update && act)
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (row0 + r < K) {
        vecN x;
        if constexpr (NV == 1) x = s[r][0];
        else
#pragma unroll
          for (int i = 0; i < NV; ++i) x[i] = s[r][i];
        *(vecN*)(base + r * rstride + at0) = x;
      }
  // levels above the stepped ones that end empty
  if (p.clear)
    for (int i = tid; i < K * vbc; i += blockDim.x) {
      const int kk = i / vbc;
      float* d = p.states + (((size_t)bh * K + kk) * V + v0 + (i - kk * vbc)) * L;
      for (int e = LA; e < L; ++e)
        if (p.clear >> e & 1) d[e] = 0.f;
    }
  // counts (shared by all rows)
  if (p.counts != nullptr && blockIdx.y == 0 && bh == 0) {
    if (p.set_counts) {
      if (tid < L) p.counts[tid] = p.final_counts[tid];
    } else if (p.update && tid == 0) {
      cascade_counts(p.counts, L, p.casc[0], STRONG);
    }
  }
}

// Levels 0 .. nlo - 1 after a prefill of T tokens (MAMBA2 fast path of
// postprocess_prefill_hstate_, kernel.py:420-436): level 0 holds k v^T of token
// T - 1; level e >= 1 holds the 2^(e-1) tokens before the tokens of levels
// < e, i.e. chunk offsets [64 - 2^e, 64 - 2^(e-1)) of the last chunk, each token
// s weighted by exp(sum_{u = s+1}^{T-1} g_u) (the reverse chunk-local cumsum
// gr[s + 1] of :420).  Grid (B * H, V / 16); the last chunk's k rows and its
// weighted v columns are staged in LDS as fp32.  Levels in the bit mask `clear`
// (those above that hold no token) are set to zero, and the level counts stored.
template <typename TK, typename TV>
__global__ __launch_bounds__(256) void mamba2_prefill_levels_kernel(
    float* __restrict__ states, const TK* __restrict__ k, const TV* __restrict__ v,
    const float* __restrict__ g, int T, int G, int H, int K, int V, int L, int nlo,
    unsigned int clear, HsCounts counts) {
  __shared__ float sk[64 * 256];      // [token][k]
  __shared__ float sv[64 * kHsCols];  // [token][column], weighted
  __shared__ float sw[64];            // sw[j]: weight of chunk offset j
  const int tid = threadIdx.x;
  const int v0 = blockIdx.y * kHsCols, bh = blockIdx.x, b = bh / H, h = bh % H;
  const int gq = h / (H / G);
  const int t0 = T - 64;     // the host guarantees T >= 64 (a prefill of whole chunks)
  if (tid < 64) {
    // lane i scans g of offset 63 - i: P_i = sum_{m <= i} g_{t0 + 63 - m}, the
    // suffix sum from offset 63 - i; offset j's weight is exp(P_{62 - j})
    float r = g[((size_t)b * T + t0 + 63 - tid) * H + h];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const float z = __shfl_up(r, d, 64);
      if (tid >= d) r += z;
    }
    if (tid <= 62) sw[62 - tid] = __expf(r);
    else sw[63] = 1.f;
  }
  for (int i = tid; i < 64 * K; i += 256) {
    const int j = i / K, kk = i % K;
    sk[j * 256 + kk] = to_f32<TK>(k[(((size_t)b * T + t0 + j) * G + gq) * K + kk]);
  }
  __syncthreads();
  for (int i = tid; i < 64 * kHsCols; i += 256) {
    const int j = i / kHsCols, c = i % kHsCols;
    sv[i] = sw[j] * to_f32<TV>(v[(((size_t)b * T + t0 + j) * H + h) * V + v0 + c]);
  }
  __syncthreads();
  const int vv = tid % kHsCols, kg = tid / kHsCols;
  float* sbase = states + (size_t)bh * K * V * L;
  for (int kk = kg; kk < K; kk += kHsRowGroups) {
    float* p = sbase + ((size_t)kk * V + v0 + vv) * L;
    p[0] = sk[63 * 256 + kk] * sv[63 * kHsCols + vv];
    for (int e = 1; e < nlo; ++e) {
      float acc = 0.f;
      for (int j = 64 - (1 << e); j < 64 - (1 << (e - 1)); ++j)
        acc += sk[j * 256 + kk] * sv[j * kHsCols + vv];
      p[e] = acc;
    }
    for (int e = nlo; e < L; ++e)
      if (clear >> e & 1) p[e] = 0.f;
  }
  if (counts.out != nullptr && blockIdx.y == 0 && bh == 0 && tid < L) counts.out[tid] = counts.v[tid];
}

}  // namespace hattn

enum { HS_BF16 = 0, HS_FP16 = 1, HS_FP32 = 2 };

namespace {

// Calls f with a value of the element type named by dtype code dt (bf16 or
// fp32); returns false for any other code.
template <typename F>
bool with_type(int dt, F&& f) {
  if (dt == HS_BF16) {
    f(__bf16{});
    return true;
  }
  if (dt == HS_FP32) {
    f(float{});
    return true;
  }
  return false;
}

bool known_type(int dt) { return dt == HS_BF16 || dt == HS_FP32; }

template <int KIND, int NV, int R, bool STRONG = false, int KMAX = 256>
hipError_t launch_steps(const HsArgs& a, int B, int nblk, hipStream_t stream) {
  const int nw = (a.K + R - 1) / R;
  const size_t smem = (size_t)2 * 2 * nw * 64 * NV * sizeof(float);
  hipLaunchKernelGGL((hattn::hstate_steps_kernel<KIND, NV, R, STRONG, KMAX>), dim3(B * a.H, nblk), dim3(64 * nw),
                     smem, stream, a);
  return hipGetLastError();
}

}  // namespace

hipError_t hattn_hstate_steps_launch(HsArgs a, int B, int gdn, hipStream_t stream,
                                     int* unsupported) {
  const HsLayer& y = a.layer;
  bool known = known_type(a.dt_qk) && known_type(a.dt_v) && known_type(a.dt_l) &&
               (!gdn || known_type(a.dt_b));
  if (y.on)
    for (int dt : {y.dt_x, y.dt_dt, y.dt_A, y.dt_bias, y.dt_Lp, y.dt_D, y.dt_lam, y.dt_out})
      known = known && known_type(dt);
  *unsupported = known ? 0 : 1;
  if (!known) return hipSuccess;
  // Columns per workgroup: as many as fit 64 NV elements of whole [level] groups, in
  // steps that keep every column block NV-aligned, evened out over the blocks.
  auto columns = [&](int nv, int* nblk) {
    const int step = nv / std::gcd(nv, a.LA), most = 64 * nv / a.LA / step * step;
    if (most == 0) return 0;
    *nblk = (a.V + most - 1) / most;
    const int vb = ((a.V + *nblk - 1) / *nblk + step - 1) / step * step;
    *nblk = (a.V + vb - 1) / vb;
    return vb;
  };
  // The widest lane load that still gives two workgroups per CU; a single element
  // per lane where the levels stepped are not contiguous, the state is not
  // aligned, or a lane's elements would span more than two columns.
  int nv = 4, nblk = 0;
  for (; nv > 1; nv >>= 1) {
    const bool fits = a.LA == a.L && !a.strong && a.LA >= nv && ((uintptr_t)a.states & (4 * nv - 1)) == 0;
    if (fits && (a.VB = columns(nv, &nblk)) != 0 && (long)B * a.H * nblk >= kHsBlocks) break;
  }
  if (nv == 1) a.VB = columns(1, &nblk);
  auto pick = [&](auto kind) {
    constexpr int KIND = decltype(kind)::value;
    if (a.strong) return launch_steps<KIND, 1, 16, true>(a, B, nblk, stream);
    if (nv == 4) return a.K > 64 ? launch_steps<KIND, 4, 32>(a, B, nblk, stream)
                                 : launch_steps<KIND, 4, 16, false, 64>(a, B, nblk, stream);
    if (nv == 2) return launch_steps<KIND, 2, 16>(a, B, nblk, stream);
    return launch_steps<KIND, 1, 16>(a, B, nblk, stream);
  };
  if (gdn) return pick(std::integral_constant<int, kHsGdelta>{});
  return pick(std::integral_constant<int, kHsMamba2>{});
}

hipError_t hattn_mamba2_prefill_levels_launch(float* states, const void* k, const void* v,
                                              const float* g, int B, int T, int G, int H, int K,
                                              int V, int L, int nlo, int dt_k, int dt_v,
                                              unsigned int clear, const HsCounts& counts,
                                              hipStream_t stream, int* unsupported) {
  using namespace hattn;
  const dim3 grid(B * H, V / kHsCols), block(256);
  *unsupported = 0;
  if (!known_type(dt_k) || !known_type(dt_v)) {
    *unsupported = 1;
    return hipSuccess;
  }
  with_type(dt_k, [&](auto tk) {
    using TK = decltype(tk);
    with_type(dt_v, [&](auto tv) {
      using TV = decltype(tv);
      hipLaunchKernelGGL((mamba2_prefill_levels_kernel<TK, TV>), grid, block, 0, stream, states,
                         (const TK*)k, (const TV*)v, g, T, G, H, K, V, L, nlo, clear, counts);
    });
  });
  return hipGetLastError();
}
