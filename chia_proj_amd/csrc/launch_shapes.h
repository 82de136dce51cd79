// launch_shapes.h -- what the kernel files and the launch code (attn_api.hip)
// have in common: normalisers, workgroup shapes, and the kernel selectors.
// Host-only programs may include it: the parameter structs stay incomplete.
#pragma once

namespace chia {

struct FwdParams;
struct BwdParams;
using KernelFn = void (*)(FwdParams);
using BwdKernelFn = void (*)(BwdParams);

enum Norm : int { NORM_SOFTMAX = 0, NORM_SIGMOID = 1, NORM_RELU = 2 };
constexpr int kNorms = 3;

// Workgroup shapes of the one-block forward core: 128 rows by four wavefronts,
// the same with two groups splitting a zigzag pair (head_dim 128), 128 rows by
// two groups of four wavefronts that split the keys, 64 rows by four groups of two.
enum Q1Shape : int { Q1_ONE = 0, Q1_ZIGZAG2 = 1, Q1_KEYS2 = 2, Q1_KEYS4 = 3 };

// Workgroup shapes of both backward kernels: wavefronts that own 32 rows (dQ) or 32 keys
// (dK/dV) each, times groups that split the walk over the key (query) tiles.
constexpr int kBwdSplits = 3;
struct BwdSplit {
  int own, groups;
};
constexpr BwdSplit kBwdSplit[kBwdSplits] = {{4, 1}, {4, 2}, {2, 4}};

// Backward kernels of one (head_dim, normaliser, ALiBi, softcap) instantiation.
struct BwdKernels {
  BwdKernelFn dq[kBwdSplits];
  BwdKernelFn dkdv[kBwdSplits][2];  // [split][1: a K/V group's heads differ in scale]
};

// The kernel selectors, one translation unit per core and head_dim.  `which`:
// normaliser + kNorms times the shape (Q1Shape).
KernelFn select_kernel_d64(int waves, int norm, bool alibi, bool softcap);
KernelFn select_q1_kernel_d64(int which, bool alibi, bool softcap, bool cap_fixed);
KernelFn select_kernel_d128(int norm);
KernelFn select_q1_kernel_d128(int which, bool alibi, bool softcap, bool cap_fixed);
KernelFn select_q1_split_kernel_d128(int norm, bool alibi, bool softcap, bool cap_fixed);
BwdKernels select_bwd_kernels_d64(int norm, bool alibi, bool softcap);
BwdKernels select_bwd_kernels_d128(int norm, bool alibi, bool softcap);

}  // namespace chia
