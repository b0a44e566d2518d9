// The level kernels of the Gated DeltaNet backward (what they compute and where they
// stand among its launches: gdn_bwd.hip).
#include "gdn_bwd.h"

namespace hattn {

// ---------------------------------------------------------------------------
// Kernel 3: reverse state scan
// ---------------------------------------------------------------------------
// V columns per workgroup: 32 where the state and its operands fit the registers (four
// waves: one per SIMD), so that an A operand serves two products; two LDS buffers where
// they fit.
constexpr int gdn_dh_bv(int K, int NW) { return K <= 128 || (K <= 192 && NW == 4) ? 32 : 16; }
constexpr bool gdn_dh_two_buffers(int K, int BV) { return K <= 128 || (K <= 192 && BV == 16); }

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
// Two LDS buffers where they fit: one barrier a chunk.
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
  constexpr bool DB = gdn_dh_two_buffers(KD, BV);
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
      // dh_{c+1} -> dhs[row][chunk][level], as fragments
      store_state_frags<KD, BV, E>(st, dhs + (((size_t)row * NT + ic) * nlev + e) * V * KD, v0);
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
// Kernels 4: the sums over the levels, per chunk
// ---------------------------------------------------------------------------
// 8 values of a 16-bit row in the order of the stored fragments: 4 lq, 16 + 4 lq, + 0..3
__device__ __forceinline__ bf16x8 row_frag(const __bf16* p) {
  const int lq = (threadIdx.x & 63) >> 4;
  const bf16x4 lo = *(const bf16x4*)(p + 4 * lq), hi = *(const bf16x4*)(p + 16 + 4 * lq);
  return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// dq_new = sum over the read levels e of lambda_e o X_e, X_e = dO h_e^T, and dlambda_e =
// rowdot(q_new, X_e).  Four waves, wave w the K columns K/4 w .. of every token; the
// chunk's dO is staged in LDS, kReadCols columns of V at a time, and each wave loads its
// part of the states' fragments PF blocks ahead.  No barrier between levels and few
// registers: several workgroups per CU hide the loads.
// (With dO's fragments loaded from memory by every wave, 8 bytes from each of 16 rows an
// instruction, the L1 lookups bound the kernel: 976 us at B 4, T 8192, H 16, K = V = 128.)
constexpr int kReadCols = 128;
template <int KD, typename TL, typename E>
__global__ __launch_bounds__(256, KD <= 64 ? 3 : 2) void gdn_bwd_read_kernel(
    const __bf16* __restrict__ qn, const __bf16* __restrict__ dO, const TL* __restrict__ l,
    const __bf16* __restrict__ hs, __bf16* __restrict__ dqn, float* __restrict__ dl_p, int T,
    int H, int V, int L, int nlev, int strong) {
  constexpr int NKT = KD / 16, NQ = NKT / 4, PF = 4, LD = kReadCols + 8;
  __shared__ __attribute__((aligned(16))) __bf16 so[kGC * LD];   // dO [t][v] of the column group
  __shared__ float lam[kGBwdMaxLev][kGC];      // weight of each stored level's read
  __shared__ float ysum[4][kGBwdMaxLev][kGC];  // rowdot(q_new, dO h_j^T), by wave
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane >> 4, ln = lane & 15;
  const int NT = T / kGC;
  const int ic = blockIdx.x % NT, row = blockIdx.x / NT;
  const int b = row / H, h = row % H;
  const size_t tok0 = (size_t)b * T + (size_t)ic * kGC;
  const size_t hk = (size_t)H * KD, hv = (size_t)H * V;
  const size_t rowk = (tok0 * H + h) * KD, rowv = (tok0 * H + h) * V;
  const int nset = __builtin_popcount(ic);
  const __bf16* hrow = hs + ((size_t)row * gdn_set_before(NT) + gdn_set_before(ic)) * V * KD +
                       (NQ * w * 64 + lane) * 8;
  auto is_set = [&](int e) { return ((ic >> e) & 1) != 0; };

  for (int u = tid; u < nlev * kGC; u += 256) {
    const int t = u / nlev, e = u % nlev;
    // what level e's stored state (bit e set) weighs in the output of token t: its
    // lambda, and with strong also that of every clear level e' >= 1 above, whose state
    // contains it (strong reads level 0 nowhere)
    const TL* lt = l + ((tok0 + t) * H + h) * L + 7;
    float x = strong && e == 0 ? 0.f : to_f32<TL>(lt[e]);
    if (strong)
      for (int e2 = e + 1; e2 < nlev; ++e2)
        if (!is_set(e2)) x += to_f32<TL>(lt[e2]);
    lam[e][t] = x;
#pragma unroll
    for (int i = 0; i < 4; ++i) ysum[i][e][t] = 0.f;
  }
  bf16x4 qd[4][NQ];   // q_new in the layout of the products' results
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int x = 0; x < NQ; ++x)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        qd[tt][x][j] = qn[rowk + (size_t)(16 * tt + 4 * lq + j) * hk + 16 * (NQ * w + x) + ln];

  floatx4 adq[4][NQ], xa[4][NQ];
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int x = 0; x < NQ; ++x) adq[tt][x] = xa[tt][x] = zero4();

  for (int c0 = 0; c0 < V && nset > 0; c0 += kReadCols) {
    const int nvb = min(kReadCols, V - c0) / 32, nsteps = nset * nvb;
    bf16x8 fr[PF][NQ];
    // step = (rank of the level) nvb + block of 32 columns; past the end the last one
    // again: a load under a condition would be waited for at the branch
    auto fetch = [&](int i, int step) __attribute__((always_inline)) {
      const int st = min(step, nsteps - 1);
      const __bf16* p = hrow + ((size_t)(st / nvb) * V + c0 + 32 * (st % nvb)) * KD;
#pragma unroll
      for (int x = 0; x < NQ; ++x) fr[i][x] = *(const bf16x8*)(p + x * 512);
    };
#pragma unroll
    for (int i = 0; i < PF; ++i) fetch(i, i);
    if (c0 > 0) __syncthreads();   // the last group's dO is read
    for (int u = tid; u < kGC * nvb * 4; u += 256) {
      const int t = u / (4 * nvb), c = 8 * (u % (4 * nvb));
      *(u32x4*)(so + t * LD + c) = *(const u32x4*)(dO + rowv + (size_t)t * hv + c0 + c);
    }
    __syncthreads();
    int e = -1, left = 0;   // the current level, its blocks to come
    for (int s0 = 0; s0 < nsteps; s0 += PF) {
#pragma unroll
      for (int i = 0; i < PF; ++i) {
        if (s0 + i < nsteps) {
          if (left == 0) {
            do ++e;
            while (!is_set(e));
            left = nvb;
          }
          const int vb = nvb - left;
#pragma unroll
          for (int tt = 0; tt < 4; ++tt) {
            const bf16x8 a = row_frag(so + (16 * tt + ln) * LD + 32 * vb);
#pragma unroll
            for (int x = 0; x < NQ; ++x) xa[tt][x] = mfma16<E>(a, fr[i][x], xa[tt][x]);
          }
          fetch(i, s0 + i + PF);
          if (--left == 0) {
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
              const floatx4 lam4 = *(const floatx4*)(&lam[e][16 * tt + 4 * lq]);
              float y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int x = 0; x < NQ; ++x) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  adq[tt][x][j] += lam4[j] * xa[tt][x][j];
                  y[j] += xa[tt][x][j] * from16<E>(qd[tt][x][j]);
                }
                xa[tt][x] = zero4();
              }
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const float ys = row_sum16(y[j]);
                if (ln == 0) ysum[w][e][16 * tt + 4 * lq + j] += ys;
              }
            }
          }
        }
      }
    }
  }
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int x = 0; x < NQ; ++x)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        dqn[rowk + (size_t)(16 * tt + 4 * lq + j) * hk + 16 * (NQ * w + x) + ln] = (__bf16)adq[tt][x][j];
  __syncthreads();
  for (int u = tid; u < nlev * kGC; u += 256) {
    const int t = u / nlev, ee = u % nlev;
    auto read = [&](int j) { return ysum[0][j][t] + ysum[1][j][t] + ysum[2][j][t] + ysum[3][j][t]; };
    float x = 0.f;
    if (strong ? ee >= 1 : is_set(ee)) {
      if (is_set(ee)) {
        x = read(ee);
      } else {
        for (int j = 0; j < ee; ++j)
          if (is_set(j)) x += read(j);
      }
    }
    dl_p[((tok0 + t) * H + h) * nlev + ee] = x;
  }
}

template <int KD>
struct GdnLevelSmem {
  static constexpr int LK = KD + 8;
  static constexpr int NWC = KD <= 128 ? 2 : 4, NW = 2 * NWC;   // column parts of Z, waves
  union {
    __bf16 z[2][kGC * LK];     // 64 rows of Z [k of h][k of dh], 16-bit hi and lo
    float du[NW][4][4][64];    // each wave's share of dU: [token, column tile][row][lane]
  };
  float red[NW];
  int bad[NW];
};

// dU, Z, dW_new, dK_new and trace Z.  Four waves (eight for K > 128, where four would
// hold more than the registers take); wave (wr, wc) owns row half wr and column half
// (quarter) wc of Z, and token tiles 2 wr, 2 wr + 1 and column part wc of dK_new.  The V columns go by in blocks of 32, the levels of a block from
// the top: a clear level's dh joins the running sum R (fp32, in the order of a B
// operand), a set level gives its part of Z with R + dh.  Every wave loads the fragments
// of h and dh that it needs, PF levels ahead: no LDS and no barrier between levels.  A
// block's sum of all clear levels' dh then gives its dU (turned around by a selector
// product, as 16-bit hi and lo, like every fp32 operand here) and its part of dK_new.  Z,
// whose products with W_new and K_new contract over either index, passes through LDS 64
// rows at a time.
// fp16: sums that are larger than any of their terms (dh over the levels, Z over all of
// V) are kept in range: Z's planes are scaled by a power of two from its largest element,
// and where a sum of dh overflows, all is done again on dh / 8.  (Unscaled, dK and dg were
// NaN at gradients 16 times below those at which any dh leaves fp16.  The scaling takes
// 140 of 6030 us of a training step at B 4, T 8192, H 16, K = V = 128, 53 of 2150 at B 1,
// T 4096, H 8, K 256, V 128; at K 192, V 384 other registers spill and it is 140 of 1690
// us faster.)
// Bound by waits for its loads (three quarters of a wave's cycles) at two workgroups a CU:
// 1525 us at B 4, T 8192, H 16, K = V = 128.  Its 256 registers do not hold everything:
// 46 spill at K = 128, 67 at 192, 364 at 256, none at 64.
// (One kernel with the reads as well took 2.6 ms there: one workgroup per CU, two thirds
// of its cycles waiting.)
template <int KD, typename E>
__global__ __launch_bounds__(64 * GdnLevelSmem<KD>::NW, KD <= 128 ? 2 : 1) void gdn_bwd_level_kernel(
    const __bf16* __restrict__ wn, const __bf16* __restrict__ kn, const __bf16* __restrict__ un,
    const __bf16* __restrict__ hs, const __bf16* __restrict__ dhs, __bf16* __restrict__ dwn,
    __bf16* __restrict__ dkn, float* __restrict__ du, float* __restrict__ del_p, int T, int H,
    int V, int nlev) {
  using Sm = GdnLevelSmem<KD>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  Sm& s = *(Sm*)smem_raw;
  constexpr int NW = Sm::NW, NWC = Sm::NWC, NTH = 64 * NW, LK = Sm::LK;
  constexpr int NKT = KD / 16, NC = NKT / NWC, ZR = NKT / 2, NP = (NC + 1) / 2;
  constexpr int PF = KD <= 64 ? 2 : 1;   // levels loaded ahead (registers)
  constexpr bool kHalf = __is_same(E, _Float16);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane >> 4, ln = lane & 15, wr = w / NWC, wc = w % NWC;
  const int NT = T / kGC;
  const int ic = blockIdx.x % NT, row = blockIdx.x / NT;
  const int b = row / H, h = row % H;
  const size_t tok0 = (size_t)b * T + (size_t)ic * kGC;
  const size_t hk = (size_t)H * KD, hv = (size_t)H * V;
  const size_t rowk = (tok0 * H + h) * KD, rowv = (tok0 * H + h) * V;
  if (ic + 1 == NT) {
    // no later chunk: every dh is zero
    for (int u = tid; u < kGC * KD; u += NTH) {
      const size_t at = rowk + (size_t)(u / KD) * hk + u % KD;
      dwn[at] = dkn[at] = (__bf16)0.f;
    }
    for (int u = tid; u < kGC * V; u += NTH) du[rowv + (size_t)(u / V) * hv + u % V] = 0.f;
    if (tid == 0) del_p[(size_t)row * NT + ic] = 0.f;
    return;
  }
  const int nvb = V / 32;
  const __bf16* hrow = hs + ((size_t)row * gdn_set_before(NT) + gdn_set_before(ic)) * V * KD +
                       (ZR * wr * 64 + lane) * 8;
  const __bf16* drow = dhs + ((size_t)row * NT + ic) * nlev * V * KD + (NC * wc * 64 + lane) * 8;
  auto is_set = [&](int e) { return ((ic >> e) & 1) != 0; };
  // dh_{c+1} of level e reaches this chunk (a level with bit e clear never ends its block)
  auto has_dh = [&](int e) { return (ic & ((2 << e) - 1)) != (2 << e) - 1; };
  struct Step {
    int vb, e;
  };
  auto after = [&](Step x) {
    if (--x.e < 0) {
      x.e = nlev - 1;
      ++x.vb;
    }
    return x;
  };
  struct Frags {
    bf16x8 hf[ZR], df[NC];
  };
  auto fetch = [&](Frags& f, Step x) __attribute__((always_inline)) {
    if (x.vb >= nvb) return;
    const __bf16* ph = hrow + ((size_t)__builtin_popcount(ic & ((1 << x.e) - 1)) * V + 32 * x.vb) * KD;
    const __bf16* pd = drow + ((size_t)x.e * V + 32 * x.vb) * KD;
    if (is_set(x.e))
#pragma unroll
      for (int i = 0; i < ZR; ++i) f.hf[i] = *(const bf16x8*)(ph + i * 512);
    if (has_dh(x.e))
#pragma unroll
      for (int i = 0; i < NC; ++i) f.df[i] = *(const bf16x8*)(pd + i * 512);
  };
  Frags fr[PF];
  auto fetch_first = [&]() __attribute__((always_inline)) {
    Step x{0, nlev - 1};
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      fetch(fr[i], x);
      x = after(x);
    }
    return x;
  };
  Step ahead = fetch_first();
  // K_new of this wave's tokens and columns, two K tiles a fragment (an odd last one
  // alone), for the blocks' dU
  bf16x8 kf[2][NP];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < NP; ++y) {
      const __bf16* p = kn + rowk + (size_t)(16 * (2 * wr + x) + ln) * hk + 16 * (NC * wc + 2 * y);
      if (2 * y + 1 < NC) {
        kf[x][y] = row_frag(p);
      } else {
        const bf16x4 k4 = *(const bf16x4*)(p + 4 * lq);
        const __bf16 zero = to16<E>(0.f);
        kf[x][y] = bf16x8{k4[0], k4[1], k4[2], k4[3], zero, zero, zero, zero};
      }
    }

  floatx4 z[ZR][NC], adk[2][NC];
  // fp16: the sums of dh over levels are taken times hs1, so that they stay below the
  // format's 65504 where every dh does (1, or 1/8 in a second pass)
  float hs1 = 1.f, zmax = 0.f;
  // the tiles on Z's diagonal: columns NC wc + y are rows ZR wr + (wc mod XD) NC + y
  constexpr int XD = ZR / NC;
  const bool diag = wc / XD == wr;
  // trace Z, of which d exp(Gc_last) and with it dg are made: its products and sums in fp32,
  // from the stored h and dh (taken from Z, whose products have R + dh rounded to 16 bits,
  // dg's error against 64 bits was 1.2 % larger where decays are slow: 16 shapes of T 512
  // to 8192; a training step 5584 -> 5666 us at B 4, T 8192, H 16, K = V = 128)
  float tr = 0.f;
  float R[NC][8];
  bf16x8 au[2];   // U of this wave's tokens, the block's columns

  auto begin_block = [&](int vb) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
      au[x] = row_frag(un + rowv + (size_t)(16 * (2 * wr + x) + ln) * hv + 32 * vb);
#pragma unroll
    for (int y = 0; y < NC; ++y)
#pragma unroll
      for (int j = 0; j < 8; ++j) R[y][j] = 0.f;
  };
  auto end_block = [&](int vb) __attribute__((always_inline)) {
    bf16x8 sel[2];   // selectors of the first and second 16 of 32 contraction indices
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const __bf16 one = to16<E>(4 * lq + j == ln ? 1.f : 0.f), zero = to16<E>(0.f);
      sel[0][j] = one;
      sel[0][4 + j] = zero;
      sel[1][j] = zero;
      sel[1][4 + j] = one;
    }
    floatx4 adu[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x) adu[x][0] = adu[x][1] = zero4();
#pragma unroll
    for (int y = 0; y < NP; ++y) {
      bf16x8 part[2][2];   // [K tile of the pair][hi, lo]
#pragma unroll
      for (int m = 0; m < 2; ++m)
        if (2 * y + m < NC) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            part[m][0][j] = to16<E>(R[2 * y + m][j]);
            part[m][1][j] = to16<E>(R[2 * y + m][j] - from16<E>(part[m][0][j]));
          }
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int p = 0; p < 2; ++p)
              adk[x][2 * y + m] = mfma16<E>(au[x], part[m][p], adk[x][2 * y + m]);
        }
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int vt = 0; vt < 2; ++vt) {
          // rows k, columns v of the pair (an odd last tile alone: zero beside it)
          const floatx4 d0 = mfma16<E>(part[0][p], sel[vt], zero4());
          const floatx4 d1 = 2 * y + 1 < NC ? mfma16<E>(part[1][p], sel[vt], zero4()) : zero4();
          const bf16x8 bd = cat8e<E>(d0, d1);
#pragma unroll
          for (int x = 0; x < 2; ++x) adu[x][vt] = mfma16<E>(kf[x][y], bd, adu[x][vt]);
        }
    }
    // the column parts' shares: wave wc sums tiles (x, vt) = (m >> 1, m & 1), m = wc, ..
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int vt = 0; vt < 2; ++vt)
#pragma unroll
        for (int i = 0; i < 4; ++i) s.du[w][2 * x + vt][i][lane] = adu[x][vt][i];
    __syncthreads();
#pragma unroll
    for (int m0 = 0; m0 < 4; m0 += NWC) {
      const int m = m0 + wc;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = 0.f;
#pragma unroll
        for (int c = 0; c < NWC; ++c) x += s.du[NWC * wr + c][m][i][lane];
        if (kHalf) x *= 1.f / hs1;
        du[rowv + (size_t)(16 * (2 * wr + (m >> 1)) + 4 * lq + i) * hv + 32 * vb + 16 * (m & 1) + ln] = x;
      }
    }
    __syncthreads();
  };
  auto dh_of = [&](__bf16 x) { return kHalf ? from16<E>(x) * hs1 : from16<E>(x); };
  auto level = [&](Frags& f, int e) __attribute__((always_inline)) {
    if (!is_set(e)) {
#pragma unroll
      for (int y = 0; y < NC; ++y)
#pragma unroll
        for (int j = 0; j < 8; ++j) R[y][j] += dh_of(f.df[y][j]);
      return;
    }
    const bool own = has_dh(e);
    auto add_trace = [&](int y) __attribute__((always_inline)) {
      if (diag) {
        const bf16x8 h = XD > 1 && (wc & 1) ? f.hf[(XD - 1) * NC + y] : f.hf[y];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          tr += from16<E>(h[j]) * (own ? R[y][j] + dh_of(f.df[y][j]) : R[y][j]);
      }
    };
#pragma unroll
    for (int y = 0; y < NC; ++y) {
      bf16x8 g;
      if (own) {
#pragma unroll
        for (int j = 0; j < 8; ++j) g[j] = to16<E>(R[y][j] + dh_of(f.df[y][j]));
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) g[j] = to16<E>(R[y][j]);
      }
      // (where it spills least: before the products, at K = 256 after them)
      if (KD <= 192) add_trace(y);
#pragma unroll
      for (int x = 0; x < ZR; ++x) z[x][y] = mfma16<E>(f.hf[x], g, z[x][y]);
      if (KD > 192) add_trace(y);
    }
  };
  bool again = false;
  do {
    Step at{0, nlev - 1};
    if (again) {
      ahead = fetch_first();
      tr = 0.f;
    }
#pragma unroll
    for (int x = 0; x < ZR; ++x)
#pragma unroll
      for (int y = 0; y < NC; ++y) z[x][y] = zero4();
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < NC; ++y) adk[x][y] = zero4();
    begin_block(0);
    while (at.vb < nvb) {
#pragma unroll
      for (int i = 0; i < PF; ++i) {
        if (at.vb < nvb) {
          level(fr[i], at.e);
          fetch(fr[i], ahead);
          ahead = after(ahead);
          const Step nx = after(at);
          if (nx.vb != at.vb) {
            end_block(at.vb);
            if (nx.vb < nvb) begin_block(nx.vb);
          }
          at = nx;
        }
      }
    }
    if constexpr (kHalf) {
      // the largest of this wave's Z (NaN: an infinite operand met a zero), and whether
      // a sum overflowed: an infinity among dK_new's accumulators or Z
      float big = 0.f, sum = 0.f;
#pragma unroll
      for (int x = 0; x < ZR; ++x)
#pragma unroll
        for (int y = 0; y < NC; ++y)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            big = fmaxf(big, fabsf(z[x][y][i]));
            sum += 0.f * z[x][y][i];
          }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < NC; ++y)
#pragma unroll
          for (int i = 0; i < 4; ++i) sum += 0.f * adk[x][y][i];
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        big = fmaxf(big, __shfl_xor(big, off, 64));
        sum += __shfl_xor(sum, off, 64);
      }
      if (lane == 0) {
        s.red[w] = big;
        s.bad[w] = sum == 0.f ? 0 : 1;
      }
      __syncthreads();
      int bad = 0;
      zmax = 0.f;
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        bad |= s.bad[i];
        zmax = fmaxf(zmax, s.red[i]);
      }
      __syncthreads();
      again = bad && !again;
      if (again) hs1 = 0.125f;
    }
  } while (again);
  float zs = 1.f;
  if constexpr (kHalf) {
    // Z's planes hold Z 2^k with its largest element below 2^15: Z is a sum of h dh over
    // V, far above the 65504 of an fp16 where h and dh are not
    int ex = 0;
    if (zmax > 0.f && zmax < INFINITY) (void)frexpf(zmax, &ex);
    zs = ldexpf(1.f, min(max(15 - ex, -60), 20));
#pragma unroll
    for (int x = 0; x < ZR; ++x)
#pragma unroll
      for (int y = 0; y < NC; ++y) z[x][y] *= zs;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < NC; ++y) adk[x][y] *= zs;
    zs = 1.f / (zs * hs1);
  }

  // ---- d exp(Gc_last) = trace Z -------------------------------------------------------
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) tr += __shfl_xor(tr, off, 64);
  if (lane == 0) s.red[w] = tr * (1.f / hs1);

  // ---- dW_new = -K_new Z^T, dK_new -= W_new Z, 64 rows of Z at a time ------------------
  // of dW_new: token tile tw, column tiles NY kp + y of the 64
  constexpr int NY = 16 / NW;
  const int tw = w & 3, kp = w >> 2;
#pragma unroll
  for (int rb = 0; rb < KD / 64; ++rb) {
#pragma unroll
    for (int x = 0; x < ZR; ++x) {
      const int r = 16 * (ZR * wr + x);   // this tile's first row of Z
      if (r / 64 == rb) {
#pragma unroll
        for (int y = 0; y < NC; ++y)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int to = (r - 64 * rb + 4 * lq + i) * LK + 16 * (NC * wc + y) + ln;
            const float v = z[x][y][i];
            const __bf16 hi = to16<E>(v);
            s.z[0][to] = hi;
            s.z[1][to] = to16<E>(v - from16<E>(hi));
          }
      }
    }
    __syncthreads();
    floatx4 adw[NY];
#pragma unroll
    for (int y = 0; y < NY; ++y) adw[y] = zero4();
#pragma unroll
    for (int c = 0; c < KD / 32; ++c) {
      const bf16x8 a = *(const bf16x8*)(kn + rowk + (size_t)(16 * tw + ln) * hk + 32 * c + 8 * lq);
#pragma unroll
      for (int y = 0; y < NY; ++y)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          adw[y] = mfma16<E>(a, *(const bf16x8*)(s.z[p] + (16 * (NY * kp + y) + ln) * LK + 32 * c + 8 * lq), adw[y]);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      bf16x8 aw[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        aw[x] = *(const bf16x8*)(wn + rowk + (size_t)(16 * (2 * wr + x) + ln) * hk + 64 * rb + 32 * c + 8 * lq);
#pragma unroll
        for (int j = 0; j < 8; ++j) aw[x][j] = to16<E>(-from16<E>(aw[x][j]));
      }
#pragma unroll
      for (int y = 0; y < NC; ++y)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const bf16x8 bz = tr_frag(s.z[p], LK, 32 * c, 16 * (NC * wc + y));
#pragma unroll
          for (int x = 0; x < 2; ++x) adk[x][y] = mfma16<E>(aw[x], bz, adk[x][y]);
        }
    }
#pragma unroll
    for (int y = 0; y < NY; ++y)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dwn[rowk + (size_t)(16 * tw + 4 * lq + i) * hk + 64 * rb + 16 * (NY * kp + y) + ln] = (__bf16)(-adw[y][i] * zs);
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < NC; ++y)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dkn[rowk + (size_t)(16 * (2 * wr + x) + 4 * lq + i) * hk + 16 * (NC * wc + y) + ln] = (__bf16)(adk[x][y][i] * zs);
  if (tid == 0) {
    float x = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) x += s.red[i];
    del_p[(size_t)row * NT + ic] = x;
  }
}

// ---------------------------------------------------------------------------
// host launcher
// ---------------------------------------------------------------------------
template <int KD, int NW, typename TL, typename E>
static hipError_t gdn_dh_scan_launch(const GdnBwdWs& w, const void* dO, const float* gcum,
                                     const void* l, int rows, int T, int H, int V, int L, int nlev,
                                     int strong, hipStream_t stream) {
  constexpr int BV = gdn_dh_bv(KD, NW);
  auto ks = gdn_dh_scan_kernel<KD, BV, NW, TL, E>;
  const int smem = (int)sizeof(GdnDhSmem<KD, BV, gdn_dh_two_buffers(KD, BV)>);
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
    // four levels per workgroup where their workgroups still run all at once, one per CU
    const bool narrow = nlev <= 4 || 2L * B * H * (V / gdn_dh_bv(KD, 4)) <= kGdnScanGroups;
    e = narrow ? gdn_dh_scan_launch<KD, 4, TL, E>(w, dO, gcum, l, B * H, T, H, V, L, nlev, strong, stream)
               : gdn_dh_scan_launch<KD, 8, TL, E>(w, dO, gcum, l, B * H, T, H, V, L, nlev, strong, stream);
    if (e != hipSuccess) return e;
  }
  const int nchunks = B * H * (T / kGC);
  hipLaunchKernelGGL((gdn_bwd_read_kernel<KD, TL, E>), dim3(nchunks), dim3(256), 0, stream, w.qn,
                     (const __bf16*)dO, (const TL*)l, w.hs, w.dq_p, w.dl_p, T, H, V, L, nlev, strong);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  auto ks = gdn_bwd_level_kernel<KD, E>;
  const int smem = (int)sizeof(GdnLevelSmem<KD>);
  if ((e = hipFuncSetAttribute((const void*)ks, hipFuncAttributeMaxDynamicSharedMemorySize, smem)) !=
      hipSuccess)
    return e;
  hipLaunchKernelGGL(ks, dim3(nchunks), dim3(64 * GdnLevelSmem<KD>::NW), smem, stream, w.wn, w.kn, w.un, w.hs, w.dhs,
                     w.dw_p, w.dk_p, w.du, w.del_p, T, H, V, nlev);
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
