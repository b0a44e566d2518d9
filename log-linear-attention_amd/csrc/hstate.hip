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
constexpr int kHsBatch = 8;   // tokens whose operands are in LDS at a time

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
// address, and reads 0 from n on.  hs_raw leaves the bits as loaded and hs_val makes
// them a float, apart, so that a token's loads are all under way before the first
// is waited for (converted within the branch on dt, each load was waited for on the
// spot: 2 us a token).
__device__ __forceinline__ unsigned int hs_raw(const void* p, long long u, unsigned int i, int dt,
                                               int n = 1) {
  const int es = dt == 0 ? 2 : 4;
  const rsrc_t r = make_rsrc((const char*)p + u * es, (size_t)n * es);
  if (dt == 0) return __builtin_amdgcn_raw_buffer_load_b16(r, 2 * i, 0, 0);
  return __builtin_amdgcn_raw_buffer_load_b32(r, 4 * i, 0, 0);
}
__device__ __forceinline__ float hs_val(unsigned int raw, int dt) {
  return __builtin_bit_cast(float, raw << (dt == 0 ? 16 : 0));
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
//   operands  of a batch of tokens at a time in LDS, each token prepared by one
//             wave (l2norm, the layer's v, g and lambda, q . k); the rows' k and q
//             are then broadcast reads.  With every wave preparing every token for
//             itself the 37 tokens after a GDELTA prefill took 6 us each.
//   cascade   S[c] += S[0 .. c-1] is a sum over the c elements before S[c] in the
//             flat [v][level] order: a shift along the lanes.
//   u = k^T S, w = q^T S   sums over a wave's rows in registers, then over the
//             waves through LDS: u at once (one barrier a token, GDELTA only), w
//             at the end of the batch.
//   update    S = a S - k (a beta u), level 0 = k (beta v)
//   output    q^T S after the update = a (w - beta (q . k) u) per level, and
//             (q . k) beta v at level 0; weighted and summed over the levels at the
//             end of the batch, one wave a token.
// (STRONG is an instance of its own: the two cascades in one kernel cost 70 spilled
// registers.)  NV (elements per lane) sets the number of workgroups: the host takes
// the widest that still fills the chip.  Measured: one GDELTA step of B 4, H 16, K =
// V = 128, L 18 in 41 us (3.7 TB/s of the 4.8 that a copy reaches), 40 tokens at B
// 1, H 16, K = V = 64 / 128 in 64 / 160 us: there the cascade's shifts and the
// barrier of u bound a token.
template <int NV>
struct HsVec {
  typedef float type __attribute__((ext_vector_type(NV)));
};
template <>
struct HsVec<1> {
  typedef float type;
};
template <int NV>
__device__ __forceinline__ float hs_get(const typename HsVec<NV>::type& x, int i) {
  if constexpr (NV == 1) return x;
  else return x[i];
}
template <int NV>
__device__ __forceinline__ void hs_set(typename HsVec<NV>::type& x, int i, float y) {
  if constexpr (NV == 1) x = y;
  else x[i] = y;
}

template <int KIND, int NV, int R, bool STRONG, int KMAX>
__global__ __launch_bounds__(64 * KMAX / R) void hstate_steps_kernel(const HsArgs p) {
  typedef typename HsVec<NV>::type vecN;
  constexpr bool GDN = KIND == kHsGdelta, LAYER = KIND == kHsLayer;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = blockDim.x >> 6;
  const int KP = nw * R;
  // dynamic LDS, nb tokens a batch: their k and q [nb][KP], the waves' w
  // [nb][wave][64 NV], u summed over the waves [nb][64 NV], the waves' u
  // [2][wave][64 NV]
  extern __shared__ floatx4 dyn[];
  const int nb = p.batch;
  float* tok_k = (float*)dyn;
  float* tok_q = tok_k + nb * KP;
  float* red_w = tok_q + nb * KP;
  float* sum_u = red_w + nb * nw * 64 * NV;
  float* red_u = sum_u + nb * 64 * NV;
  __shared__ float tok_l[kHsBatch][kHsMaxLevels], tok_v[kHsBatch][64], tok_x[LAYER ? kHsBatch : 1][64];
  __shared__ float tok_s[kHsBatch][4];   // exp(g), beta, q . k

  const int bh = blockIdx.x, b = bh / p.H, h = bh - b * p.H, gq = h / (p.H / p.G);
  const int K = p.K, V = p.V, L = p.L, LA = p.LA;
  const int v0 = blockIdx.y * p.VB, vbc = p.VB < V - v0 ? p.VB : V - v0;
  const bool act = lane * NV < vbc * LA;
  const int e0 = act ? lane * NV : 0;
  const int vv0 = e0 / LA, ll0 = e0 - vv0 * LA;
  int ll[NV];
  int vi = vv0;   // column of this lane's level-0 element, if it has one
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    ll[i] = ll0 + i >= LA ? ll0 + i - LA : ll0 + i;
    if (i > 0 && ll[i] == 0) ++vi;
  }
  vi &= 63;       // (a lane at the end that has none)
  // a lane's elements are contiguous unless only the first LA of L levels are stepped
  const bool whole = LA == L;
  const unsigned int at0 = whole ? e0 : vv0 * L + ll0;
  const int row0 = wave * R;
  // (a uniform row address and a 32-bit lane offset: no address registers per row)
  float* base = p.states + (((size_t)bh * K + row0) * V + v0) * L;
  const int rstride = V * L;
  auto at = [&](int i) { return at0 + i + (ll0 + i >= LA ? L - LA : 0); };

  float s[R][NV];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    vecN x{};
    if (!p.zero && row0 + r < K) x = *(const vecN*)(base + r * rstride + at0);
#pragma unroll
    for (int i = 0; i < NV; ++i) s[r][i] = hs_get<NV>(x, i);
  }

  const HsLayer& y = p.layer;
  // token t0 + i0 + j of the batch at i0, prepared by one wave
  auto prepare = [&](int i0, int j) {
    const int t = p.t0 + i0 + j;
    const long long qo = b * p.q_b + t * p.q_t + gq * K, so = b * p.s_b + t * p.s_t + h;
    const long long vo = b * p.v_b + t * p.v_t + h * V, lo = b * p.l_b + t * p.l_t + h * L;
    unsigned int kraw[4], qraw[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int i = lane + 64 * c;
      kraw[c] = p.update && 64 * c < K ? hs_raw(p.k, qo, i, p.dt_qk, K) : 0;
      qraw[c] = p.output && 64 * c < K ? hs_raw(p.q, qo, i, p.dt_qk, K) : 0;
    }
    const int dt_x = LAYER ? y.dt_x : p.dt_v;
    const unsigned int graw = p.update && !LAYER ? hs_raw(p.g, so, 0, 2) : 0;
    const unsigned int braw = GDN && p.update ? hs_raw(p.beta, so, 0, p.dt_b) : 0;
    const unsigned int vraw = p.update ? hs_raw(p.v, vo, v0 + lane, dt_x, V) : 0;
    const unsigned int lraw = p.output ? hs_raw(p.l, lo, lane, p.dt_l, L) : 0;
    unsigned int draw = 0, biasraw = 0, araw = 0, lpraw = 0;
    if (LAYER) {
      draw = hs_raw(y.dt, so, 0, y.dt_dt);
      if (y.bias) biasraw = hs_raw(y.bias, h, 0, y.dt_bias);
      araw = hs_raw(y.A, h, 0, y.dt_A);
      lpraw = hs_raw(y.Lp, h * L, lane, y.dt_Lp, L);
    }
    float kx[4], qx[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      kx[c] = hs_val(kraw[c], p.dt_qk);
      qx[c] = hs_val(qraw[c], p.dt_qk);
    }
    const float beta = GDN && p.update ? hs_val(braw, p.dt_b) : 1.f, xv = hs_val(vraw, dt_x);
    float g = hs_val(graw, 2), vx = xv, lx = hs_val(lraw, p.dt_l);
    if (LAYER) {
      // the Mamba-2 layer's inputs: v = x dt', g = A dt', lambda of (L, dl), each
      // rounded to its dtype as the separate layer kernels do
      const float d = layer_dtp(hs_val(draw, y.dt_dt), hs_val(biasraw, y.dt_bias), y.softplus);
      g = layer_g(hs_val(araw, y.dt_A), d);
      vx = hs_round(xv * d, p.dt_v);
      lx = hs_round(lambda_of(hs_val(lpraw, y.dt_Lp), lx, y.mode), y.dt_lam);
      tok_x[j][lane] = xv;
    }
    if (p.norm) {
      // q / |q| * scale, k / |k| (kernel.py:20-23, 626-629 with the eps of fla's
      // l2norm), rounded to the input dtype after the norm and after the scale, as
      // the reference's l2norm_fwd / l2norm_and_scale_fwd store their outputs
      float nq = 0.f, nk = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        nq += qx[c] * qx[c];
        nk += kx[c] * kx[c];
      }
      const float rq = rsqrtf(wave_sum(nq) + 1e-6f), rk = rsqrtf(wave_sum(nk) + 1e-6f);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        qx[c] = hs_round(hs_round(qx[c] * rq, p.dt_qk) * p.scale, p.dt_qk);
        kx[c] = hs_round(kx[c] * rk, p.dt_qk);
      }
    }
    float qk = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) qk += qx[c] * kx[c];
    qk = wave_sum(qk);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (lane + 64 * c < KP) {
        tok_k[j * KP + lane + 64 * c] = kx[c];
        tok_q[j * KP + lane + 64 * c] = qx[c];
      }
    tok_v[j][lane] = vx;
    if (lane < kHsMaxLevels) tok_l[j][lane] = lx;
    if (lane == 0) {
      tok_s[j][0] = p.update ? __expf(g) : 1.f;
      tok_s[j][1] = beta;
      tok_s[j][2] = qk;
    }
  };

  for (int t = 0; t < p.T; ++t) {
    const int j = t & (nb - 1);
    if (j == 0) {
      if (t > 0) __syncthreads();   // the last batch's output reads
      for (int i = wave; i < nb && t + i < p.T; i += nw) prepare(t, i);
      __syncthreads();
    }
    const float a = tok_s[j][0], beta = tok_s[j][1], qk = tok_s[j][2];
    const floatx4* kr = (const floatx4*)(tok_k + j * KP + row0);
    const floatx4* qr = (const floatx4*)(tok_q + j * KP + row0);

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
        int own_c = c - ll0;        // this lane's element of level c, if it has one
        if (own_c < 0) own_c += LA;
        const bool has = own_c < NV;
        const int lim = has ? c - own_c : -(1 << 20);
        bool own[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          keep[i] = ll[i] >= c && ll[i] > 0;
          into[i] = i == own_c && c > 0;
          own[i] = has && i < own_c && own_c - i <= c;
        }
        const int far = (c + NV - 1) / NV;   // lanes before that hold levels below c
        auto hop = [&](int d, float (&cur)[NV], float& sum) {
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            cur[i] = lane_before(cur[i]);
            sum += NV * d - i <= lim ? cur[i] : 0.f;
          }
        };
        if constexpr (NV < 4) {
          // the hops outside, the rows inside: straight code for a hop (a loop per row
          // was half of a token)
          float sum[R], cur[R][NV];
#pragma unroll
          for (int r = 0; r < R; ++r) {
            sum[r] = 0.f;
#pragma unroll
            for (int i = 0; i < NV; ++i) {
              sum[r] += own[i] ? s[r][i] : 0.f;
              cur[r][i] = s[r][i];
            }
          }
          for (int d = 1; d <= far; ++d)
#pragma unroll
            for (int r = 0; r < R; ++r) hop(d, cur[r], sum[r]);
#pragma unroll
          for (int r = 0; r < R; ++r)
#pragma unroll
            for (int i = 0; i < NV; ++i)
              s[r][i] = (keep[i] ? s[r][i] : 0.f) + (into[i] ? sum[r] : 0.f);
        } else {
          // one hop reaches all levels below c <= NV; no registers to hold the hops of
          // every row
#pragma unroll
          for (int r = 0; r < R; ++r) {
            float sum = 0.f, cur[NV];
#pragma unroll
            for (int i = 0; i < NV; ++i) {
              sum += own[i] ? s[r][i] : 0.f;
              cur[i] = s[r][i];
            }
            hop(1, cur, sum);
            for (int d = 2; d <= far; ++d) hop(d, cur, sum);
#pragma unroll
            for (int i = 0; i < NV; ++i)
              s[r][i] = (keep[i] ? s[r][i] : 0.f) + (into[i] ? sum : 0.f);
          }
        }
      }
    }

    float u[NV], w[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) u[i] = w[i] = 0.f;
    const bool need_u = GDN && p.update;
    if (need_u)
#pragma unroll
      for (int r = 0; r < R; r += 4) {
        const floatx4 kk = kr[r / 4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int i = 0; i < NV; ++i) u[i] += kk[m] * s[r + m][i];
      }
    if (p.output)
#pragma unroll
      for (int r = 0; r < R; r += 4) {
        const floatx4 qq = qr[r / 4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int i = 0; i < NV; ++i) w[i] += qq[m] * s[r + m][i];
      }
    vecN x;
    if (p.output) {
#pragma unroll
      for (int i = 0; i < NV; ++i) hs_set<NV>(x, i, w[i]);
      *(vecN*)(red_w + ((j * nw + wave) * 64 + lane) * NV) = x;
    }
    if (need_u) {
      float* ru = red_u + (t & 1) * nw * 64 * NV;
#pragma unroll
      for (int i = 0; i < NV; ++i) hs_set<NV>(x, i, u[i]);
      *(vecN*)(ru + (wave * 64 + lane) * NV) = x;
      __syncthreads();
      vecN acc{};
      for (int i = 0; i < nw; ++i) acc += *(const vecN*)(ru + (i * 64 + lane) * NV);
#pragma unroll
      for (int i = 0; i < NV; ++i) u[i] = hs_get<NV>(acc, i);
      if (p.output && wave == 0) *(vecN*)(sum_u + (j * 64 + lane) * NV) = acc;
    }

    if (p.update) {
      float m[NV];
      const float vx = beta * tok_v[j][vi];
#pragma unroll
      for (int i = 0; i < NV; ++i) m[i] = ll[i] == 0 ? vx : -(a * beta) * u[i];
#pragma unroll
      for (int r = 0; r < R; r += 4) {
        const floatx4 kk = kr[r / 4];
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            float& z = s[r + n][i];
            if (GDN) z = __builtin_fmaf(kk[n], m[i], a * z);
            else z = ll[i] == 0 ? kk[n] * m[i] : a * z;
          }
      }
    }

    if (p.output && (j == nb - 1 || t + 1 == p.T)) {
      __syncthreads();
      for (int n = wave; n <= j; n += nw) {
        const float an = tok_s[n][0], bn = tok_s[n][1], qkn = tok_s[n][2];
        float* rw = red_w + (n * nw * 64 + lane) * NV;
        vecN acc{}, un{};
        for (int i = 0; i < nw; ++i) acc += *(const vecN*)(rw + i * 64 * NV);
        if (need_u) un = *(const vecN*)(sum_u + (n * 64 + lane) * NV);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          float z = hs_get<NV>(acc, i);
          if (p.update) {
            z = GDN ? an * (z - bn * qkn * hs_get<NV>(un, i)) : an * z;
            if (ll[i] == 0) z = qkn * (bn * tok_v[n][vi]);
          }
          hs_set<NV>(acc, i, tok_l[n][ll[i]] * z);
        }
        // this wave alone reads and writes token n's sums
        *(vecN*)rw = acc;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (lane < vbc) {
          const float* part = red_w + n * nw * 64 * NV + lane * LA;
          float z = 0.f;
#pragma unroll 8
          for (int e = 0; e < LA; ++e) z += part[e];
          const long long oo = b * p.o_b + (p.t0 + t - j + n) * p.o_t + h * V + v0;
          if (LAYER) {
            z = hs_round(z, p.dt_v);
            if (y.D) z = layer_out(z, tok_x[n][lane], hs_val(hs_raw(y.D, h, 0, y.dt_D), y.dt_D));
          }
          hs_st(p.o, oo, lane, z, LAYER ? y.dt_out : p.dt_v);
        }
      }
    }
  }

  if (p.update && act)
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (row0 + r < K) {
        if (whole) {
          vecN x;
#pragma unroll
          for (int i = 0; i < NV; ++i) hs_set<NV>(x, i, s[r][i]);
          *(vecN*)(base + r * rstride + at0) = x;
        } else {
#pragma unroll
          for (int i = 0; i < NV; ++i) base[r * rstride + at(i)] = s[r][i];
        }
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
hipError_t launch_steps(HsArgs a, int B, int nblk, hipStream_t stream) {
  const int nw = (a.K + R - 1) / R;
  // (a power of two; four tokens at K > 128, where eight would leave one workgroup
  // per CU; fewer where a workgroup's 64 KB would not hold them beside the static
  // arrays: 64640 bytes at K = 256, NV = 4 are the most that occurs)
  a.batch = a.T == 1 ? 1 : a.K > 128 ? 4 : hattn::kHsBatch;
  constexpr size_t kStatic = sizeof(float) * hattn::kHsBatch *
                             (kHsMaxLevels + 64 + (KIND == kHsLayer ? 64 : 0) + 4) + 256;
  auto bytes = [&](int batch) {
    return (size_t)(batch * (2 * nw * R + (nw + 1) * 64 * NV) + 2 * nw * 64 * NV) * sizeof(float);
  };
  while (a.batch > 1 && bytes(a.batch) + kStatic > 65536) a.batch /= 2;
  const size_t smem = bytes(a.batch);
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
  // The widest lane load that still gives kHsBlocks workgroups; narrower where the
  // state is not aligned or a lane's elements would span more than two columns.
  int nv = 4, nblk = 0;
  for (; nv > 1; nv >>= 1) {
    const bool fits = !a.strong && a.LA >= nv &&
                      (a.LA == a.L ? ((uintptr_t)a.states & (4 * nv - 1)) == 0 : a.zero != 0);
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
  if (y.on) return pick(std::integral_constant<int, kHsLayer>{});
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
