// Arguments of the HState token-step kernel (hstate.hip), filled by the C entry
// points (hattn_api.cpp).
#pragma once

#include <cstddef>
#include <cstdint>

constexpr int kHsMaxLevels = 32;    // levels of a state
constexpr int kHsMaxTokens = 256;   // tokens per launch: their cascades travel in the arguments
enum { kHsMamba2 = 0, kHsGdelta = 1, kHsLayer = 2 };   // what a step is
constexpr int kHsBlocks = 256;      // workgroups below which narrower column blocks are taken

// The Mamba-2 layer's decode step (hselective_state_update): the kernel forms v, g
// and lambda from the layer's inputs and adds the D residual.  HsArgs::v is x then,
// HsArgs::l is dl.  dt_*: dtype codes; dt_lam, dt_out: those of lambda and the output.
struct HsLayer {
  const void *dt, *A, *bias, *Lp, *D;   // bias, D may be null
  int on, softplus, mode;
  int dt_x, dt_dt, dt_A, dt_bias, dt_Lp, dt_D, dt_lam, dt_out;
};

struct HsArgs {
  float* states;
  int* counts;   // device level counts, or null
  const void *q, *k, *v, *beta, *l;
  const float* g;
  void* o;
  // element strides of a batch and of a token: q and k; beta and g; v; l; o
  long long q_b, q_t, s_b, s_t, v_b, v_t, l_b, l_t, o_b, o_t;
  int G, H, K, V, L;
  int LA;        // levels stepped: the first LA of the L
  int VB;        // value columns per workgroup (set by the launch)
  int batch;     // tokens whose operands are in LDS at a time (set by the launch)
  int T, t0;     // tokens, the first one's index in the operands
  int strong, update, output, norm;
  int zero;      // start from an empty state instead of reading it
  unsigned int clear;   // levels >= LA set to zero at the end (bit mask)
  int set_counts;       // store final_counts instead of advancing counts by one token
  int dt_qk, dt_v, dt_l, dt_b;
  float scale;
  HsLayer layer;
  int final_counts[kHsMaxLevels];
  unsigned char casc[kHsMaxTokens];   // cascade depth (weak) or merge level (strong) per token
};

struct HsCounts {
  int* out;      // device level counts, or null
  int v[kHsMaxLevels];
};
