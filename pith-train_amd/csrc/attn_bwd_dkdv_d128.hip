// dK/dV launches for head dims (128, 128); the kernel body is in attn_bwd_dkdv_d128.h.
#include "attn_bwd_common.h"
#include "attn_bwd_dkdv_d128.h"

namespace pith {
namespace {

template <bool CAUSAL, typename OutT, bool EMIT_DS, bool DESC = false>
__global__ __launch_bounds__(dkdv_d128::kThreads) void attn_bwd_dkdv_d128_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[dkdv_d128::kSmem];
  dkdv_d128::body<CAUSAL, OutT, EMIT_DS, DESC>(p, smem, blockIdx.x);
}

template <bool EMIT_DS>
void launch_variant(const BwdParams& p, bool causal, bool f32_out, unsigned grid, hipStream_t st) {
  const dim3 g(grid), block(dkdv_d128::kThreads);
  if (causal) {
    if (p.walk_desc) {
      if (f32_out) hipLaunchKernelGGL((attn_bwd_dkdv_d128_kernel<true, float, EMIT_DS, true>), g, block, 0, st, p);
      else hipLaunchKernelGGL((attn_bwd_dkdv_d128_kernel<true, __bf16, EMIT_DS, true>), g, block, 0, st, p);
    } else if (f32_out) hipLaunchKernelGGL((attn_bwd_dkdv_d128_kernel<true, float, EMIT_DS>), g, block, 0, st, p);
    else hipLaunchKernelGGL((attn_bwd_dkdv_d128_kernel<true, __bf16, EMIT_DS>), g, block, 0, st, p);
  } else {
    if (f32_out) hipLaunchKernelGGL((attn_bwd_dkdv_d128_kernel<false, float, EMIT_DS>), g, block, 0, st, p);
    else hipLaunchKernelGGL((attn_bwd_dkdv_d128_kernel<false, __bf16, EMIT_DS>), g, block, 0, st, p);
  }
}

}  // namespace

void launch_dkdv_d128(const BwdParams& p, bool causal, bool f32_out, unsigned grid, hipStream_t st) {
  if (p.ds) launch_variant<true>(p, causal, f32_out, grid, st);
  else launch_variant<false>(p, causal, f32_out, grid, st);
}

}  // namespace pith
