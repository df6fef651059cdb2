// dQ launches of the kernel in attn_bwd_dq_direct.h.
#include "attn_bwd_common.h"
#include "attn_bwd_dq_direct.h"

namespace pith {
namespace {

template <int DQK, bool CAUSAL, typename OutT>
__global__ __launch_bounds__(dq_direct::kThreads) void attn_bwd_dq_direct_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[dq_direct::kSmem<DQK>];
  dq_direct::body<DQK, CAUSAL, OutT>(p, smem, blockIdx.x);
}

template <int DQK>
void launch_one(BwdParams p, bool causal, bool f32_out, hipStream_t st) {
  p.q_tiles = (p.Sq + 127) / 128;
  const dim3 grid((unsigned)(p.q_tiles * p.Hq * p.B)), block(dq_direct::kThreads);
  if (causal) {
    if (f32_out) hipLaunchKernelGGL((attn_bwd_dq_direct_kernel<DQK, true, float>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((attn_bwd_dq_direct_kernel<DQK, true, __bf16>), grid, block, 0, st, p);
  } else {
    if (f32_out) hipLaunchKernelGGL((attn_bwd_dq_direct_kernel<DQK, false, float>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((attn_bwd_dq_direct_kernel<DQK, false, __bf16>), grid, block, 0, st, p);
  }
}

}  // namespace

void launch_dq_direct(const BwdParams& p, int dqk, bool causal, bool f32_out, hipStream_t st) {
  if (dqk == 192) launch_one<192>(p, causal, f32_out, st);
  else launch_one<128>(p, causal, f32_out, st);
}

}  // namespace pith
