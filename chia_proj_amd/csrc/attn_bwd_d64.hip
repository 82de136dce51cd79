// attn_bwd_d64.hip -- instantiations of the backward kernels for head_dim 64:
// 3 normalisers x ALiBi on/off x softcap on/off (dK/dV also with per-head c1).
#include "attn_bwd_kernel.h"

namespace chia {

template <int NORM, bool AL, bool SC, int SPLIT>
static void set_split(BwdKernels& k) {
  constexpr int OWN = kBwdSplit[SPLIT].own, GROUPS = kBwdSplit[SPLIT].groups;
  k.dq[SPLIT] = attn_bwd_dq_kernel<64, NORM, AL, SC, OWN, GROUPS>;
  k.dkdv[SPLIT][0] = attn_bwd_dkdv_kernel<64, NORM, AL, SC, false, OWN, GROUPS>;
  k.dkdv[SPLIT][1] = attn_bwd_dkdv_kernel<64, NORM, AL, SC, true, OWN, GROUPS>;
}

template <int NORM, bool AL, bool SC>
static BwdKernels bwd_inst() {
  BwdKernels k;
  set_split<NORM, AL, SC, 0>(k);
  set_split<NORM, AL, SC, 1>(k);
  set_split<NORM, AL, SC, 2>(k);
  return k;
}

BwdKernels select_bwd_kernels_d64(int norm, bool alibi, bool softcap) {
  static const BwdKernels table[3][2][2] = {
      {{bwd_inst<NORM_SOFTMAX, false, false>(), bwd_inst<NORM_SOFTMAX, false, true>()},
       {bwd_inst<NORM_SOFTMAX, true, false>(), bwd_inst<NORM_SOFTMAX, true, true>()}},
      {{bwd_inst<NORM_SIGMOID, false, false>(), bwd_inst<NORM_SIGMOID, false, true>()},
       {bwd_inst<NORM_SIGMOID, true, false>(), bwd_inst<NORM_SIGMOID, true, true>()}},
      {{bwd_inst<NORM_RELU, false, false>(), bwd_inst<NORM_RELU, false, true>()},
       {bwd_inst<NORM_RELU, true, false>(), bwd_inst<NORM_RELU, true, true>()}},
  };
  return table[norm][alibi ? 1 : 0][softcap ? 1 : 0];
}

}  // namespace chia
