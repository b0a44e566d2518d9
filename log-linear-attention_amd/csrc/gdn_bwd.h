// The Gated DeltaNet backward's workspace and its two halves: the level kernels
// (gdn_bwd_levels.hip) and the chunk-local kernel with the host side (gdn_bwd.hip).
#pragma once
#include "gdn_common.h"

namespace hattn {

struct GdnBwdWs {
  __bf16 *qn, *kn, *knT, *wn, *un, *hs;
  __bf16* dhs;                 // dh of every level after every chunk [row][chunk][level][v][k]
  __bf16 *dq_p, *dw_p, *dk_p;  // dq_new, dW_new, dK_new
  float *du, *dl_p, *del_p;
  size_t bytes;
};

}  // namespace hattn

// Launches the reverse state scan and the level sums: dq_p, dw_p, dk_p, du, dl_p and
// del_p of w from its q_new, W_new, K_new, U and level states.  dt_l: lambda's dtype
// code (0 bf16, 2 fp32); h16: fp16 operands (fp32 lambda).
hipError_t hattn_gdn_bwd_levels_launch(const hattn::GdnBwdWs& w, const void* dO, const float* gcum,
                                       const void* l, int B, int T, int H, int K, int V, int L,
                                       int nlev, int dt_l, int strong, int h16, hipStream_t stream,
                                       int* unsupported);
