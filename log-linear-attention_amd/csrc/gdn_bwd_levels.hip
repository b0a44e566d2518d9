// The level kernels of the Gated DeltaNet backward (what they compute and where they
// stand among its launches: gdn_bwd.hip).
#include "gdn_bwd.h"

namespace hattn {

// ---------------------------------------------------------------------------
// Kernel 3: reverse state scan
// ---------------------------------------------------------------------------
template <int KD, int BV, bool DB>
struct GdnDhSmem {
  static constexpr int LK = KD + 8, LVS = BV + 8, NB = DB ? 2 : 1;
  __bf16 kwq[NB][3][kGC * LK];   // the chunk's K_new, W_new, q_new [t][k]
  __bf16 dO[NB][kGC * LVS];      // dO slice [t][v]
  float lam[NB][kGBwdMaxLev][kGC];
};

// One wave per inter-chunk level, as the forward scan: wave w holds dh of level
// e = (this workgroup's first level) + w, [K x BV] in fp32 (tile (kt, nt): rows
// 16 kt + 4 lq + i, columns 16 nt + ln), and the levels never meet.  dh feeds the
// product with K_new, and dV_new the one with W_new^T, as B operands straight from
// the accumulators (cat8e pairs with A operands read in the same order of the
// contraction index: frag_k2, tr_frag_d).  NW waves per workgroup: with few (row,
// V slice) pairs the levels are spread over two workgroups of four, which halves
// the LDS reads of each (they bound a chunk: a wave reads every A operand itself).
// Two LDS buffers where they fit (K <= 192): one barrier a chunk.
// (The previous reverse scan kept all levels in one workgroup, three barriers a
// level, and formed the sums of kernel 4 on the way: 2.46 ms at B 4, T 8192, H 16, K
// = V = 128; 10.1 ms for 128 of the 384 columns of V at B 1, T 16384, H 6, K = 192,
// where it had 24 workgroups.)
template <int KD, int BV, int NW, typename TL, typename E>
__global__ __launch_bounds__(64 * NW) void gdn_dh_scan_kernel(
    const __bf16* __restrict__ qn, const __bf16* __restrict__ wn, const __bf16* __restrict__ kn,
    const __bf16* __restrict__ dO, const float* __restrict__ gcum, const TL* __restrict__ l,
    __bf16* __restrict__ dhs, int nrows, int T, int H, int V, int L, int nlev, int nparts,
    int strong) {
  constexpr bool DB = KD <= 192;
  using Sm = GdnDhSmem<KD, BV, DB>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  Sm& s = *(Sm*)smem_raw;
  constexpr int LK = Sm::LK, LVS = Sm::LVS, NTH = 64 * NW;
  constexpr int NKT = KD / 16, NVT = BV / 16, NC = KD / 32;
  constexpr int UPR = KD / 8, KU = kGC * UPR / NTH;      // 16-byte units per row / per thread
  constexpr int VU = (kGC * BV / 4 + NTH - 1) / NTH;     // 8-byte units of the dO slice per thread
  constexpr int LU = (kGBwdMaxLev * kGC + NTH - 1) / NTH;
  static_assert(kGC * UPR % NTH == 0, "units per thread");
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane >> 4, ln = lane & 15;
  const XcdMap mp = xcd_map(blockIdx.x, V / BV * nparts);
  if (mp.row >= nrows) return;
  const int row = mp.row, v0 = (mp.slice / nparts) * BV;
  const int e = (mp.slice % nparts) * NW + w;            // this wave's level
  const bool act = e < nlev;
  const int b = row / H, h = row % H;
  const int NT = T / kGC;
  const size_t rowtok = (size_t)b * T * H + h;           // (token 0 of the row) * H + h
  const unsigned HV = (unsigned)H * V, HK = (unsigned)H * KD, HL = (unsigned)H * L;

  u32x4 rk[KU], rw[KU], rq[KU];
  uint2 rv[VU];
  TL rl[LU];
  float rg;
  const rsrc_t grs = make_rsrc(gcum + rowtok + (size_t)(kGC - 1) * H, (size_t)T * H * 4);
  auto stage_load = [&](int jc) __attribute__((always_inline)) {
    const size_t tokoff = rowtok + (size_t)jc * kGC * H;
    rg = buf_load<float>(grs, 0, (unsigned)((size_t)jc * kGC * H * 4));
#pragma unroll
    for (int r = 0; r < KU; ++r) {
      const int u = tid + NTH * r;
      const size_t off = tokoff * KD + (unsigned)(u / UPR) * HK + 8 * (u % UPR);
      rk[r] = *(const u32x4*)(kn + off);
      rw[r] = *(const u32x4*)(wn + off);
      rq[r] = *(const u32x4*)(qn + off);
    }
#pragma unroll
    for (int r = 0; r < VU; ++r) {
      const int u = min(tid + NTH * r, kGC * BV / 4 - 1);
      rv[r] = *(const uint2*)(dO + tokoff * V + v0 + (unsigned)(u / (BV / 4)) * HV + 4 * (u % (BV / 4)));
    }
#pragma unroll
    for (int r = 0; r < LU; ++r) {
      const int u = min(tid + NTH * r, nlev * kGC - 1);
      rl[r] = l[tokoff * L + (unsigned)(u / nlev) * HL + 7 + u % nlev];
    }
  };
  auto stage_store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < KU; ++r) {
      const int u = tid + NTH * r, at = (u / UPR) * LK + 8 * (u % UPR);
      *(u32x4*)(s.kwq[buf][0] + at) = rk[r];
      *(u32x4*)(s.kwq[buf][1] + at) = rw[r];
      *(u32x4*)(s.kwq[buf][2] + at) = rq[r];
    }
#pragma unroll
    for (int r = 0; r < VU; ++r) {
      const int u = tid + NTH * r;
      if (u < kGC * BV / 4) *(uint2*)(s.dO[buf] + (u / (BV / 4)) * LVS + 4 * (u % (BV / 4))) = rv[r];
    }
#pragma unroll
    for (int r = 0; r < LU; ++r) {
      const int u = tid + NTH * r;
      if (u < nlev * kGC) s.lam[buf][u % nlev][u / nlev] = to_f32<TL>(rl[r]);
    }
  };

  floatx4 st[NKT][NVT];
#pragma unroll
  for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
    for (int nt = 0; nt < NVT; ++nt) st[kt][nt] = zero4();

  stage_load(NT - 1);
  stage_store(0);
  __syncthreads();
  int buf = 0;
  for (int ic = NT - 1; ic >= 0; --ic) {
    const float eL = fexp(rg);   // exp(Gc_last) of chunk ic
    const int per = 2 << e;
    const bool bit = (ic >> e) & 1;
    const bool rd = act && (strong ? e >= 1 : bit);
    const bool live = act && ic < NT - 1 && (ic & (per - 1)) != per - 1;   // dh_{c+1} reaches this chunk
    const __bf16* Kt = s.kwq[buf][0];
    const __bf16* Wt = s.kwq[buf][1];
    const __bf16* Qt = s.kwq[buf][2];
    if (live) {
      // dh_{c+1} -> dhs[row][chunk][level][v][k]
      const rsrc_t rh = make_rsrc(dhs + ((((size_t)row * NT + ic) * nlev + e) * V + v0) * KD,
                                  (size_t)BV * KD * 2);
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int nt = 0; nt < NVT; ++nt)
          buf_store8(__builtin_bit_cast(uint2, cvt4e<E>(st[kt][nt])), rh,
                     (unsigned)(((16 * nt + ln) * KD + 16 * kt + 4 * lq) * 2), 0);
    }
    // the next chunk's operands, into registers while this one is computed
    stage_load(max(ic - 1, 0));
    if (live) {
      floatx4 dv[4][NVT];   // -dV_new[t = 16 tt + 4 lq + i][v = 16 nt + ln]
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int nt = 0; nt < NVT; ++nt) dv[tt][nt] = zero4();
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        bf16x8 bh[NVT];
#pragma unroll
        for (int nt = 0; nt < NVT; ++nt) bh[nt] = cat8e<E>(st[2 * c][nt], st[2 * c + 1][nt]);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          const bf16x8 a = frag_k2(Kt, LK, 16 * tt + ln, 32 * c + 4 * lq);
#pragma unroll
          for (int nt = 0; nt < NVT; ++nt) dv[tt][nt] = mfma16<E>(a, bh[nt], dv[tt][nt]);
        }
      }
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int nt = 0; nt < NVT; ++nt) st[kt][nt] *= eL;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        bf16x8 bv[NVT];
#pragma unroll
        for (int nt = 0; nt < NVT; ++nt) bv[nt] = cat8e<E>(-dv[2 * c][nt], -dv[2 * c + 1][nt]);
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
          const bf16x8 a = tr_frag_d(Wt, LK, 32 * c, 16 * kt);
#pragma unroll
          for (int nt = 0; nt < NVT; ++nt) st[kt][nt] = mfma16<E>(a, bv[nt], st[kt][nt]);
        }
      }
    } else {
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int nt = 0; nt < NVT; ++nt) st[kt][nt] = zero4();
    }
    if (rd) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        // (lambda_e o dO)[t][v], rounded as a 16-bit operand
        const floatx4 l0 = *(const floatx4*)(&s.lam[buf][e][32 * c + 4 * lq]);
        const floatx4 l1 = *(const floatx4*)(&s.lam[buf][e][32 * c + 16 + 4 * lq]);
        bf16x8 bo[NVT];
#pragma unroll
        for (int nt = 0; nt < NVT; ++nt) {
          const bf16x8 x = tr_frag_d(s.dO[buf], LVS, 32 * c, 16 * nt);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            bo[nt][j] = to16<E>(from16<E>(x[j]) * l0[j]);
            bo[nt][4 + j] = to16<E>(from16<E>(x[4 + j]) * l1[j]);
          }
        }
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
          const bf16x8 a = tr_frag_d(Qt, LK, 32 * c, 16 * kt);
#pragma unroll
          for (int nt = 0; nt < NVT; ++nt) st[kt][nt] = mfma16<E>(a, bo[nt], st[kt][nt]);
        }
      }
    }
    if constexpr (!DB) __syncthreads();   // the chunk's operands are read
    buf = DB ? buf ^ 1 : 0;
    stage_store(buf);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Kernel 4: the sums over the levels, per chunk
// ---------------------------------------------------------------------------
template <int KD>
struct GdnLevelSmem {
  static constexpr int NW = KD <= 128 ? 4 : 8;   // waves
  static constexpr int NP = NW / 4;              // parts of K of dq_new
  static constexpr int LK = KD + 8;
  union {
    __bf16 tile[2][2][32 * LK];   // [buffer][h, dh][v][k]: 32 columns of V of one level
    __bf16 z[2][kGC * LK];        // 64 rows of Z [k of h][k of dh], 16-bit hi and lo
  };
  __bf16 kn[kGC * LK];            // K_new [t][k]
  float lam[kGBwdMaxLev][kGC];    // weight of each set level's read
  float y[NP][kGBwdMaxLev][kGC];  // rowdot(q_new, dO h_j^T), by part of K
  float red[NW];
};

// Four waves, or eight where four would hold more than the registers take (K > 128).
// Wave (wr, wc) = (w >> 1, w & 1) owns column half wc of its share wr of the rows of Z,
// and, of the [64 x K] results, token tile w & 3 and part w >> 2 of K of dq_new, token
// tiles 8 / NW wr + x and column half wc of dK_new.  The V columns go by in blocks of
// 32, the levels of a block from the top: a clear level's dh joins the running sum R
// (fp32, in the order of a B operand) and gives its part of dU; a set level's h gives
// its part of Z with R + dh, and of dq_new and dlambda.  A level's [32 x K] pieces of h
// and dh go through two LDS buffers, loaded one step ahead.  Z, whose products with
// W_new and K_new contract over either index, then passes through LDS 64 rows at a time
// as a 16-bit hi and lo part, so it loses nothing to rounding.
template <int KD, typename TL, typename E>
__global__ __launch_bounds__(64 * GdnLevelSmem<KD>::NW) void gdn_bwd_level_kernel(
    const __bf16* __restrict__ qn, const __bf16* __restrict__ wn, const __bf16* __restrict__ kn,
    const __bf16* __restrict__ un, const __bf16* __restrict__ dO, const TL* __restrict__ l,
    const __bf16* __restrict__ hs, const __bf16* __restrict__ dhs, __bf16* __restrict__ dqn,
    __bf16* __restrict__ dwn, __bf16* __restrict__ dkn, float* __restrict__ du,
    float* __restrict__ dl_p, float* __restrict__ del_p, int T, int H, int V, int L, int nlev,
    int strong) {
  using Sm = GdnLevelSmem<KD>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  Sm& s = *(Sm*)smem_raw;
  constexpr int NW = Sm::NW, NTH = 64 * NW, LK = Sm::LK, NKT = KD / 16, NH = KD / 32;
  constexpr int ZR = 2 * NKT / NW, NX = NKT / Sm::NP, TT = 8 / NW;   // row tiles of Z, K tiles of dq_new, token tiles of dK_new
  constexpr int UPR = KD / 8, HU = (32 * UPR + NTH - 1) / NTH;       // 16-byte units per row / per thread
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane >> 4, ln = lane & 15, wr = w >> 1, wc = w & 1;
  const int tw = w & 3, kp = w >> 2;
  const int NT = T / kGC;
  const int ic = blockIdx.x % NT, row = blockIdx.x / NT;
  const int b = row / H, h = row % H;
  const size_t tok0 = (size_t)b * T + (size_t)ic * kGC;
  const size_t hk = (size_t)H * KD, hv = (size_t)H * V;
  const size_t rowk = (tok0 * H + h) * KD, rowv = (tok0 * H + h) * V;
  const bool have_dh = ic + 1 < NT;
  const __bf16* hrow = hs + ((size_t)row * gdn_set_before(NT) + gdn_set_before(ic)) * V * KD;
  const __bf16* drow = dhs + ((size_t)row * NT + ic) * nlev * V * KD;
  auto is_set = [&](int e) { return (ic >> e) & 1; };
  // dh_{c+1} of level e reaches this chunk (a level with bit e clear never ends its block)
  auto has_dh = [&](int e) { return have_dh && (ic & ((2 << e) - 1)) != (2 << e) - 1; };
  // the next level at or below e with something to do in this chunk, or -1
  auto work_at = [&](int e) {
    while (e >= 0 && !is_set(e) && !have_dh) --e;
    return e;
  };

  u32x4 ph[HU], pd[HU];
  auto fetch = [&](int vb, int e) __attribute__((always_inline)) {
    const __bf16* ps = hrow + ((size_t)__builtin_popcount(ic & ((1 << e) - 1)) * V + 32 * vb) * KD;
    const __bf16* pt = drow + ((size_t)e * V + 32 * vb) * KD;
    if (is_set(e))
#pragma unroll
      for (int i = 0; i < HU; ++i) ph[i] = *(const u32x4*)(ps + 8 * min(tid + NTH * i, 32 * UPR - 1));
    if (has_dh(e))
#pragma unroll
      for (int i = 0; i < HU; ++i) pd[i] = *(const u32x4*)(pt + 8 * min(tid + NTH * i, 32 * UPR - 1));
  };
  auto put = [&](int buf, int e) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < HU; ++i) {
      const int u = tid + NTH * i, at = (u / UPR) * LK + 8 * (u % UPR);
      if (32 * UPR % NTH != 0 && u >= 32 * UPR) break;
      if (is_set(e)) *(u32x4*)(s.tile[buf][0] + at) = ph[i];
      if (has_dh(e)) *(u32x4*)(s.tile[buf][1] + at) = pd[i];
    }
  };
  const int top = work_at(nlev - 1);
  if (top >= 0) fetch(0, top);

  if (tid < 256) g2s_tile<KD>(kn + rowk, hk, s.kn, LK);
  for (int u = tid; u < nlev * kGC; u += NTH) {
    const int t = u / nlev, e = u % nlev;
    // what level e's stored state (bit e set) weighs in the output of token t: its
    // lambda, and with strong also that of every clear level e' >= 1 above, whose state
    // contains it (strong reads level 0 nowhere)
    const TL* lt = l + ((tok0 + t) * H + h) * L + 7;
    float x = strong && e == 0 ? 0.f : to_f32<TL>(lt[e]);
    if (strong)
      for (int e2 = e + 1; e2 < nlev; ++e2)
        if (!is_set(e2)) x += to_f32<TL>(lt[e2]);
    s.lam[e][t] = x;
#pragma unroll
    for (int x2 = 0; x2 < Sm::NP; ++x2) s.y[x2][e][t] = 0.f;
  }
  // q_new of this wave's tokens in the layout of the products' results
  bf16x4 qd[NX];
#pragma unroll
  for (int kt = 0; kt < NX; ++kt)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      qd[kt][i] = qn[rowk + (size_t)(16 * tw + 4 * lq + i) * hk + 16 * (NX * kp + kt) + ln];
  if (top >= 0) put(0, top);
  __syncthreads();

  floatx4 z[ZR][NH], adq[NX], adk[TT][NH];
#pragma unroll
  for (int x = 0; x < ZR; ++x)
#pragma unroll
    for (int y = 0; y < NH; ++y) z[x][y] = zero4();
#pragma unroll
  for (int x = 0; x < NX; ++x) adq[x] = zero4();
#pragma unroll
  for (int x = 0; x < TT; ++x)
#pragma unroll
    for (int y = 0; y < NH; ++y) adk[x][y] = zero4();

  int buf = 0;
  for (int vb = 0; vb < V / 32; ++vb) {
    const bf16x8 ao = *(const bf16x8*)(dO + rowv + (size_t)(16 * tw + ln) * hv + 32 * vb + 8 * lq);
    bf16x8 au[TT];
#pragma unroll
    for (int x = 0; x < TT; ++x)
      au[x] = *(const bf16x8*)(un + rowv + (size_t)(16 * (TT * wr + x) + ln) * hv + 32 * vb + 8 * lq);
    float R[NH][8];
#pragma unroll
    for (int y = 0; y < NH; ++y)
#pragma unroll
      for (int j = 0; j < 8; ++j) R[y][j] = 0.f;
    floatx4 adu[TT];   // token tile tw, column tiles TT kp + x
#pragma unroll
    for (int x = 0; x < TT; ++x) adu[x] = zero4();

    for (int e = top; e >= 0;) {
      int ne = work_at(e - 1), nvb = vb;
      if (ne < 0) {
        ne = top;
        nvb = vb + 1;
      }
      const bool more = nvb < V / 32;
      if (more) fetch(nvb, ne);
      const __bf16* Ht = s.tile[buf][0];
      const __bf16* Dt = s.tile[buf][1];
      if (!is_set(e)) {
#pragma unroll
        for (int y = 0; y < NH; ++y) {
          const bf16x8 d = tr_frag(Dt, LK, 0, 16 * (NH * wc + y));
#pragma unroll
          for (int j = 0; j < 8; ++j) R[y][j] += from16<E>(d[j]);
        }
#pragma unroll
        for (int c = 0; c < NH; ++c) {
          const bf16x8 a = *(const bf16x8*)(s.kn + (16 * tw + ln) * LK + 32 * c + 8 * lq);
#pragma unroll
          for (int x = 0; x < TT; ++x)
            adu[x] = mfma16<E>(a, *(const bf16x8*)(Dt + (16 * (TT * kp + x) + ln) * LK + 32 * c + 8 * lq), adu[x]);
        }
      } else {
        // dq_new and dlambda: X = dO h^T, this wave's tokens and part of K
        const floatx4 lam4 = *(const floatx4*)(&s.lam[e][16 * tw + 4 * lq]);
        float yv[4] = {0.f, 0.f, 0.f, 0.f};
        bf16x8 ah[ZR];
#pragma unroll
        for (int kt = 0; kt < NX; ++kt) {
          const bf16x8 bh = tr_frag(Ht, LK, 0, 16 * (NX * kp + kt));
          if constexpr (NW == 4) {   // the fragments are also those of its rows of Z
            if (kt / ZR == wr) ah[kt % ZR] = bh;
          }
          const floatx4 x = mfma16<E>(ao, bh, zero4());
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            adq[kt][i] += lam4[i] * x[i];
            yv[i] += from16<E>(qd[kt][i]) * x[i];
          }
        }
        if constexpr (NW != 4)
#pragma unroll
          for (int x = 0; x < ZR; ++x) ah[x] = tr_frag(Ht, LK, 0, 16 * (ZR * wr + x));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float ys = row_sum16(yv[i]);
          if (ln == 0) s.y[kp][e][16 * tw + 4 * lq + i] += ys;
        }
        if (have_dh) {
          const bool own = has_dh(e);
#pragma unroll
          for (int y = 0; y < NH; ++y) {
            bf16x8 g;
            if (own) {
              const bf16x8 d = tr_frag(Dt, LK, 0, 16 * (NH * wc + y));
#pragma unroll
              for (int j = 0; j < 8; ++j) g[j] = to16<E>(R[y][j] + from16<E>(d[j]));
            } else {
#pragma unroll
              for (int j = 0; j < 8; ++j) g[j] = to16<E>(R[y][j]);
            }
#pragma unroll
            for (int x = 0; x < ZR; ++x) z[x][y] = mfma16<E>(ah[x], g, z[x][y]);
          }
        }
      }
      buf ^= 1;
      if (more) put(buf, ne);
      __syncthreads();
      e = nvb == vb ? ne : -1;
    }

    // U (sum_e wr dh)^T, the sum as hi + lo
    if (have_dh)
#pragma unroll
      for (int y = 0; y < NH; ++y) {
        bf16x8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          hi[j] = to16<E>(R[y][j]);
          lo[j] = to16<E>(R[y][j] - from16<E>(hi[j]));
        }
#pragma unroll
        for (int x = 0; x < TT; ++x) {
          adk[x][y] = mfma16<E>(au[x], hi, adk[x][y]);
          adk[x][y] = mfma16<E>(au[x], lo, adk[x][y]);
        }
      }
#pragma unroll
    for (int x = 0; x < TT; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        du[rowv + (size_t)(16 * tw + 4 * lq + i) * hv + 32 * vb + 16 * (TT * kp + x) + ln] = adu[x][i];
  }

  // ---- d exp(Gc_last) = trace Z -------------------------------------------------------
  float tr = 0.f;
#pragma unroll
  for (int x = 0; x < ZR; ++x)
#pragma unroll
    for (int y = 0; y < NH; ++y)
      if (ZR * wr + x == NH * wc + y)
#pragma unroll
        for (int i = 0; i < 4; ++i) tr += 4 * lq + i == ln ? z[x][y][i] : 0.f;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) tr += __shfl_xor(tr, off, 64);
  if (lane == 0) s.red[w] = tr;
  __syncthreads();
  if (tid == 0) {
    float x = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) x += s.red[i];
    del_p[(size_t)row * NT + ic] = x;
  }

  // ---- dW_new = -K_new Z^T, dK_new -= W_new Z, 64 rows of Z at a time ------------------
#pragma unroll
  for (int rb = 0; rb < KD / 64; ++rb) {
    if (have_dh) {
#pragma unroll
      for (int x = 0; x < ZR; ++x) {
        const int r = 16 * (ZR * wr + x);   // this tile's first row of Z
        if (r / 64 == rb) {
#pragma unroll
          for (int y = 0; y < NH; ++y)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int at = (r - 64 * rb + 4 * lq + i) * LK + 16 * (NH * wc + y) + ln;
              const float v = z[x][y][i];
              const __bf16 hi = to16<E>(v);
              s.z[0][at] = hi;
              s.z[1][at] = to16<E>(v - from16<E>(hi));
            }
        }
      }
      __syncthreads();
    }
    constexpr int NY = 4 / Sm::NP;   // column tiles of the block per wave
    floatx4 adw[NY];
#pragma unroll
    for (int y = 0; y < NY; ++y) adw[y] = zero4();
    if (have_dh) {
#pragma unroll
      for (int c = 0; c < NH; ++c) {
        const bf16x8 a = *(const bf16x8*)(s.kn + (16 * tw + ln) * LK + 32 * c + 8 * lq);
#pragma unroll
        for (int y = 0; y < NY; ++y)
#pragma unroll
          for (int p = 0; p < 2; ++p)
            adw[y] = mfma16<E>(a, *(const bf16x8*)(s.z[p] + (16 * (NY * kp + y) + ln) * LK + 32 * c + 8 * lq), adw[y]);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        bf16x8 aw[TT];
#pragma unroll
        for (int x = 0; x < TT; ++x) {
          aw[x] = *(const bf16x8*)(wn + rowk + (size_t)(16 * (TT * wr + x) + ln) * hk + 64 * rb + 32 * c + 8 * lq);
#pragma unroll
          for (int j = 0; j < 8; ++j) aw[x][j] = to16<E>(-from16<E>(aw[x][j]));
        }
#pragma unroll
        for (int y = 0; y < NH; ++y)
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            const bf16x8 bz = tr_frag(s.z[p], LK, 32 * c, 16 * (NH * wc + y));
#pragma unroll
            for (int x = 0; x < TT; ++x) adk[x][y] = mfma16<E>(aw[x], bz, adk[x][y]);
          }
      }
    }
#pragma unroll
    for (int y = 0; y < NY; ++y)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dwn[rowk + (size_t)(16 * tw + 4 * lq + i) * hk + 64 * rb + 16 * (NY * kp + y) + ln] = (__bf16)-adw[y][i];
    __syncthreads();
  }
#pragma unroll
  for (int kt = 0; kt < NX; ++kt)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      dqn[rowk + (size_t)(16 * tw + 4 * lq + i) * hk + 16 * (NX * kp + kt) + ln] = (__bf16)adq[kt][i];
#pragma unroll
  for (int x = 0; x < TT; ++x)
#pragma unroll
    for (int y = 0; y < NH; ++y)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dkn[rowk + (size_t)(16 * (TT * wr + x) + 4 * lq + i) * hk + 16 * (NH * wc + y) + ln] = (__bf16)adk[x][y][i];

  // ---- dlambda ------------------------------------------------------------------------
  for (int u = tid; u < nlev * kGC; u += NTH) {
    const int t = u / nlev, e = u % nlev;
    auto read = [&](int j) { return Sm::NP == 1 ? s.y[0][j][t] : s.y[0][j][t] + s.y[Sm::NP - 1][j][t]; };
    float x = 0.f;
    if (strong ? e >= 1 : is_set(e)) {
      if (is_set(e)) {
        x = read(e);
      } else {
        for (int j = 0; j < e; ++j)
          if (is_set(j)) x += read(j);
      }
    }
    dl_p[((tok0 + t) * H + h) * nlev + e] = x;
  }
}

// ---------------------------------------------------------------------------
// host launcher
// ---------------------------------------------------------------------------
template <int KD, int NW, typename TL, typename E>
static hipError_t gdn_dh_scan_launch(const GdnBwdWs& w, const void* dO, const float* gcum,
                                     const void* l, int rows, int T, int H, int V, int L, int nlev,
                                     int strong, hipStream_t stream) {
  constexpr int BV = gdn_scan_bv(KD);
  auto ks = gdn_dh_scan_kernel<KD, BV, NW, TL, E>;
  const int smem = (int)sizeof(GdnDhSmem<KD, BV, KD <= 192>);
  const int nparts = (nlev + NW - 1) / NW;
  hipError_t e = hipFuncSetAttribute((const void*)ks, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(ks, dim3((rows + 7) / 8 * 8 * (V / BV) * nparts), dim3(64 * NW), smem, stream,
                     w.qn, w.wn, w.kn, (const __bf16*)dO, gcum, (const TL*)l, w.dhs, rows, T, H, V,
                     L, nlev, nparts, strong);
  return hipGetLastError();
}

template <int KD, typename TL, typename E>
static hipError_t gdn_levels_launch(const GdnBwdWs& w, const void* dO, const float* gcum,
                                    const void* l, int B, int T, int H, int V, int L, int nlev,
                                    int strong, hipStream_t stream) {
  hipError_t e;
  if (nlev > 0) {
    // four levels per workgroup where one workgroup per (row, V slice) would leave
    // CUs idle
    const bool narrow = nlev <= 4 || (long)B * H * (V / gdn_scan_bv(KD)) < kGdnScanGroups;
    e = narrow ? gdn_dh_scan_launch<KD, 4, TL, E>(w, dO, gcum, l, B * H, T, H, V, L, nlev, strong, stream)
               : gdn_dh_scan_launch<KD, 8, TL, E>(w, dO, gcum, l, B * H, T, H, V, L, nlev, strong, stream);
    if (e != hipSuccess) return e;
  }
  auto ks = gdn_bwd_level_kernel<KD, TL, E>;
  const int smem = (int)sizeof(GdnLevelSmem<KD>);
  if ((e = hipFuncSetAttribute((const void*)ks, hipFuncAttributeMaxDynamicSharedMemorySize, smem)) !=
      hipSuccess)
    return e;
  hipLaunchKernelGGL(ks, dim3(B * H * (T / kGC)), dim3(64 * GdnLevelSmem<KD>::NW), smem, stream, w.qn,
                     w.wn, w.kn, w.un, (const __bf16*)dO, (const TL*)l, w.hs, w.dhs, w.dq_p, w.dw_p,
                     w.dk_p, w.du, w.dl_p, w.del_p, T, H, V, L, nlev, strong);
  return hipGetLastError();
}

}  // namespace hattn

hipError_t hattn_gdn_bwd_levels_launch(const hattn::GdnBwdWs& w, const void* dO, const float* gcum,
                                       const void* l, int B, int T, int H, int K, int V, int L,
                                       int nlev, int dt_l, int strong, int h16, hipStream_t stream,
                                       int* unsupported) {
  using namespace hattn;
#define HATTN_GDN_LV(KD_, TL_, E_) \
  return gdn_levels_launch<KD_, TL_, E_>(w, dO, gcum, l, B, T, H, V, L, nlev, strong, stream);
#define HATTN_GDN_L(KD_)                                           \
  if (K == KD_) {                                                  \
    if (h16 && dt_l == 2 && !strong) HATTN_GDN_LV(KD_, float, _Float16) \
    if (!h16 && dt_l == 0) HATTN_GDN_LV(KD_, __bf16, __bf16)       \
    if (!h16 && dt_l == 2) HATTN_GDN_LV(KD_, float, __bf16)        \
  }
  HATTN_GDN_L(64)
  HATTN_GDN_L(128)
  HATTN_GDN_L(192)
  HATTN_GDN_L(256)
#undef HATTN_GDN_L
#undef HATTN_GDN_LV
  *unsupported = 1;
  return hipSuccess;
}
