// launch_shapes.cpp -- what chia_attn_fwd and chia_attn_bwd launch, without a
// GPU: the kernel selectors return tags instead of kernels and
// hipLaunchKernel, defined here before the HIP runtime's, records the tag, the
// grid and the workgroup.  tests/test_launch_shapes.py builds it with the C
// ABI's host code (attn_api.hip) and feeds it one call a line:
//   fwd|bwd norm B H Hkv S D causal window dilation block prefix softcap alibi head_scale packed
// (packed: 0, or the tokens that q_stride[0] reports).  Answers, one a line:
//   fwd: <core> <threads> <grid> <fixed reference>, core one of paired, one,
//        zigzag2, keys2, keys4
//   bwd: <dQ split> <threads> <grid> <dK/dV split> <threads> <grid> <per-head c1>
// or "status <code>".
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "chia_attn.h"
#include "launch_shapes.h"

namespace {
struct Launch {
  uintptr_t tag;
  unsigned grid, threads;
};
std::vector<Launch> g_launches;

// Forward tags: core, then the fixed reference.  Backward: 0x1000 + split (dQ),
// 0x2000 + 2 split + per-head c1 (dK/dV).
enum Core { PAIRED, ONE, ZIGZAG2, KEYS2, KEYS4 };
const char* const kCore[] = {"paired", "one", "zigzag2", "keys2", "keys4"};
chia::KernelFn fwd_tag(int core, bool cap_fixed) { return (chia::KernelFn)(uintptr_t)(1 + 2 * core + cap_fixed); }
chia::KernelFn q1_tag(int which, bool cap_fixed) {
  switch (which / chia::kNorms) {
    case chia::Q1_ONE: return fwd_tag(ONE, cap_fixed);
    case chia::Q1_KEYS2: return fwd_tag(KEYS2, cap_fixed);
    case chia::Q1_KEYS4: return fwd_tag(KEYS4, cap_fixed);
  }
  return nullptr;
}
chia::BwdKernels bwd_tags() {
  chia::BwdKernels k;
  for (int s = 0; s < chia::kBwdSplits; ++s) {
    k.dq[s] = (chia::BwdKernelFn)(uintptr_t)(0x1000 + s);
    for (int c = 0; c < 2; ++c) k.dkdv[s][c] = (chia::BwdKernelFn)(uintptr_t)(0x2000 + 2 * s + c);
  }
  return k;
}
}  // namespace

namespace chia {
struct Fp8Params;
using Fp8KernelFn = void (*)(Fp8Params);
// as in attn_fwd_d64.hip and attn_fwd_d128.hip: the paired core has four
// wavefronts, and at head_dim 128 no softmax
KernelFn select_kernel_d64(int waves, int, bool, bool) { return waves == 4 ? fwd_tag(PAIRED, false) : nullptr; }
KernelFn select_kernel_d128(int norm) { return norm == NORM_SOFTMAX ? nullptr : fwd_tag(PAIRED, false); }
KernelFn select_q1_kernel_d64(int which, bool, bool, bool cap_fixed) { return q1_tag(which, cap_fixed); }
KernelFn select_q1_kernel_d128(int which, bool, bool, bool cap_fixed) { return q1_tag(which, cap_fixed); }
KernelFn select_q1_split_kernel_d128(int, bool, bool, bool cap_fixed) { return fwd_tag(ZIGZAG2, cap_fixed); }
BwdKernels select_bwd_kernels_d64(int, bool, bool) { return bwd_tags(); }
BwdKernels select_bwd_kernels_d128(int, bool, bool) { return bwd_tags(); }
Fp8KernelFn select_fp8_kernel(int, int, int, bool, bool) { return nullptr; }
}  // namespace chia

extern "C" hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
  g_launches.push_back(Launch{(uintptr_t)fn, grid.x, block.x});
  return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

int main() {
  char kind[8];
  long norm, B, H, Hkv, S, D, causal, window, dil, block, prefix, alibi, head_scale, packed;
  float softcap;
  while (std::scanf("%7s %ld %ld %ld %ld %ld %ld %ld %ld %ld %ld %ld %f %ld %ld %ld", kind, &norm, &B, &H, &Hkv, &S,
                    &D, &causal, &window, &dil, &block, &prefix, &softcap, &alibi, &head_scale, &packed) == 16) {
    chia_attn_args a;
    std::memset(&a, 0, sizeof(a));
    a.struct_size = sizeof(a);
    a.norm = (uint32_t)norm;
    a.batch = B;
    a.heads = H;
    a.kv_heads = Hkv;
    a.seqlen = S;
    a.head_dim = D;
    a.causal = (int32_t)causal;
    a.window = (int32_t)window;
    a.dilation = (int32_t)dil;
    a.block = (int32_t)block;
    a.prefix = (int32_t)prefix;
    a.softcap = softcap;
    a.scale = 0.125f;
    a.post_scale = 1.0f;
    // aligned, never dereferenced device pointers
    a.q = (const void*)0x10000;
    a.k = (const void*)0x20000;
    a.v = (const void*)0x30000;
    a.o = (void*)0x40000;
    if (alibi) a.alibi_slopes = (const float*)0x50000;
    if (head_scale) a.head_scale = (const float*)0x60000;
    if (packed) a.cu_seqlens = (const int32_t*)0x70000;
    for (int64_t* st : {a.q_stride, a.k_stride, a.v_stride, a.o_stride}) {
      st[0] = packed ? 0 : H * S * D;
      st[1] = S * D;
      st[2] = D;
    }
    if (packed) a.q_stride[0] = packed;
    g_launches.clear();
    if (!std::strcmp(kind, "fwd")) {
      const int st = chia_attn_fwd(&a, nullptr);
      if (st != CHIA_ATTN_OK || g_launches.size() != 1) {
        std::printf("status %d\n", st);
        continue;
      }
      const Launch& l = g_launches[0];
      const int core = (int)(l.tag - 1) / 2;
      std::printf("%s %u %u %d\n", kCore[core], l.threads, l.grid, (int)(l.tag - 1) % 2);
    } else {
      chia_attn_bwd_args w;
      std::memset(&w, 0, sizeof(w));
      w.struct_size = sizeof(w);
      w.fwd = &a;
      w.dout = (const void*)0x80000;
      w.dq = (void*)0x90000;
      w.dk = (void*)0xa0000;
      w.dv = (void*)0xb0000;
      w.lse = (const float*)0xc0000;
      w.workspace = (void*)0xd0000;
      w.workspace_bytes = chia_attn_bwd_workspace_size(&a);
      for (int64_t* st : {w.dout_stride, w.dq_stride, w.dk_stride, w.dv_stride}) {
        st[0] = packed ? 0 : H * S * D;
        st[1] = S * D;
        st[2] = D;
      }
      const int st = chia_attn_bwd(&w, nullptr);
      if (st != CHIA_ATTN_OK || g_launches.size() != 2) {
        std::printf("status %d\n", st);
        continue;
      }
      const Launch &q = g_launches[0], &k = g_launches[1];
      std::printf("%d %u %u %d %u %u %d\n", (int)(q.tag - 0x1000), q.threads, q.grid, (int)(k.tag - 0x2000) / 2,
                  k.threads, k.grid, (int)(k.tag - 0x2000) % 2);
    }
  }
  return 0;
}
