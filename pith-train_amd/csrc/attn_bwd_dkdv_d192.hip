// dK/dV launches for head dims (192, 128); the kernel body is in attn_bwd_dkdv_d192.h.
#include "attn_bwd_common.h"
#include "attn_bwd_dkdv_d192.h"

namespace pith {
namespace {

template <bool CAUSAL, typename OutT, bool EMIT_DS>
__global__ __launch_bounds__(dkdv_d192::kThreads) void attn_bwd_dkdv_d192_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[dkdv_d192::kSmem];
  dkdv_d192::body<CAUSAL, OutT, EMIT_DS>(p, smem, blockIdx.x);
}

}  // namespace

void launch_dkdv_d192(const BwdParams& p, bool causal, bool f32_out, unsigned grid, hipStream_t st) {
  const dim3 g(grid), block(dkdv_d192::kThreads);
  auto launch = [&](auto emit) {
    constexpr bool E = decltype(emit)::value;
    if (causal) {
      if (f32_out) hipLaunchKernelGGL((attn_bwd_dkdv_d192_kernel<true, float, E>), g, block, 0, st, p);
      else hipLaunchKernelGGL((attn_bwd_dkdv_d192_kernel<true, __bf16, E>), g, block, 0, st, p);
    } else {
      if (f32_out) hipLaunchKernelGGL((attn_bwd_dkdv_d192_kernel<false, float, E>), g, block, 0, st, p);
      else hipLaunchKernelGGL((attn_bwd_dkdv_d192_kernel<false, __bf16, E>), g, block, 0, st, p);
    }
  };
  if (p.ds != nullptr) launch(std::true_type{});
  else launch(std::false_type{});
}

}  // namespace pith
