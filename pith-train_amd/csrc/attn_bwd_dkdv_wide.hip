// dK/dV launches with 256 key rows per workgroup; the kernel body is in attn_bwd_dkdv_wide.h.
#include "attn_bwd_dkdv_wide.h"

namespace pith {
namespace {

template <bool CAUSAL, typename OutT, bool DESC = false>
__global__ __launch_bounds__(dkdv_wide::kThreads) void attn_bwd_dkdv_wide_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[dkdv_wide::kSmem];
  dkdv_wide::body<CAUSAL, OutT, DESC>(p, smem, blockIdx.x);
}

template <typename OutT>
void launch_out(const BwdParams& p, bool causal, unsigned grid, hipStream_t st) {
  const dim3 g(grid), block(dkdv_wide::kThreads);
  if (!causal) hipLaunchKernelGGL((attn_bwd_dkdv_wide_kernel<false, OutT>), g, block, 0, st, p);
  else if (p.walk_desc) hipLaunchKernelGGL((attn_bwd_dkdv_wide_kernel<true, OutT, true>), g, block, 0, st, p);
  else hipLaunchKernelGGL((attn_bwd_dkdv_wide_kernel<true, OutT>), g, block, 0, st, p);
}

}  // namespace

void launch_dkdv_wide(const BwdParams& p, bool causal, bool f32_out, unsigned grid, hipStream_t st) {
  if (f32_out) launch_out<float>(p, causal, grid, st);
  else launch_out<__bf16>(p, causal, grid, st);
}

}  // namespace pith
