// attn_fwd_q1_d128.hip -- instantiations of the one-query-block-per-wavefront
// forward core (attn_fwd_q1_kernel.h) for head_dim 128: 3 normalisers x
// ALiBi on/off x softcap on/off, with one group of four wavefronts per
// workgroup or two, and softcap softmax against the fixed reference for caps
// up to 54 (attn_fwd_q1_d64.hip: head_dim 64).
#include "attn_fwd_q1_kernel.h"

namespace chia {

template <int NORM, bool AL, bool SC, int NG, int RW, int KG, bool CAPFIX = false>
static KernelFn inst_q1() {
  return attn_fwd_q1_kernel<128, NORM, AL, SC, NG, CAPFIX, RW, KG>;
}

template <int NG, int RW, int KG>
static KernelFn select_shape(int norm, bool alibi, bool softcap, bool cap_fixed) {
  if (cap_fixed && norm == NORM_SOFTMAX && softcap)
    return alibi ? inst_q1<NORM_SOFTMAX, true, true, NG, RW, KG, true>()
                 : inst_q1<NORM_SOFTMAX, false, true, NG, RW, KG, true>();
  static const KernelFn table[3][2][2] = {
      {{inst_q1<NORM_SOFTMAX, false, false, NG, RW, KG>(), inst_q1<NORM_SOFTMAX, false, true, NG, RW, KG>()},
       {inst_q1<NORM_SOFTMAX, true, false, NG, RW, KG>(), inst_q1<NORM_SOFTMAX, true, true, NG, RW, KG>()}},
      {{inst_q1<NORM_SIGMOID, false, false, NG, RW, KG>(), inst_q1<NORM_SIGMOID, false, true, NG, RW, KG>()},
       {inst_q1<NORM_SIGMOID, true, false, NG, RW, KG>(), inst_q1<NORM_SIGMOID, true, true, NG, RW, KG>()}},
      {{inst_q1<NORM_RELU, false, false, NG, RW, KG>(), inst_q1<NORM_RELU, false, true, NG, RW, KG>()},
       {inst_q1<NORM_RELU, true, false, NG, RW, KG>(), inst_q1<NORM_RELU, true, true, NG, RW, KG>()}},
  };
  return table[norm][alibi ? 1 : 0][softcap ? 1 : 0];
}

KernelFn select_q1_kernel_d128(int which, bool alibi, bool softcap, bool cap_fixed) {
  const int norm = which % kNorms;
  switch (which / kNorms) {
    case Q1_ONE: return select_shape<1, 4, 1>(norm, alibi, softcap, cap_fixed);
    case Q1_KEYS2: return select_shape<1, 4, 2>(norm, alibi, softcap, cap_fixed);
    case Q1_KEYS4: return select_shape<1, 2, 4>(norm, alibi, softcap, cap_fixed);
  }
  return nullptr;
}

// Two groups per workgroup splitting each zigzag pair (causal grids).
KernelFn select_q1_split_kernel_d128(int norm, bool alibi, bool softcap, bool cap_fixed) {
  return select_shape<2, 4, 1>(norm, alibi, softcap, cap_fixed);
}

}  // namespace chia
