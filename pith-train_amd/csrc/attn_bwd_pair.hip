// dK/dV and dQ of one chunk pair as ONE grid. The two kernels do not depend on each other (both recompute the scores from
// lse and delta), and launched one after the other the second waits until the last workgroup of the first has drained: on
// grids of less than a round half the device idles throughout (1021 rows x 16 heads: 128 workgroups of each kernel on 256
// compute units), on grids of a few rounds the tails do. Here a workgroup takes its role from its block id, the dK/dV
// workgroups first (they carry a third more work), the dQ ones behind them fill every unit that falls free.
// Measured, dK/dV + dQ, separate launches against one: 1 x 1021 x 16 heads of 192 causal 71 -> 42 us, 1 x 2048 x 16 of 192
// 122 -> 84 us, 2 x 2048 x 16/4 of 64 114 -> 79 us, 1 x 2304 x 32/4 of 128, no mask 383 -> 289 us. Which launches: one_grid.
#include "attn_bwd_common.h"
#include "attn_bwd_dkdv_d128.h"
#include "attn_bwd_dkdv_d192.h"
#include "attn_bwd_dkdv_d64.h"
#include "attn_bwd_dq_direct.h"
#include "attn_bwd_dq_duo.h"

namespace pith {
namespace {

constexpr int larger(int a, int b) { return a > b ? a : b; }

template <int DQK, bool CAUSAL, typename KvT, typename QT>
__global__ __launch_bounds__(DQK == 64 ? 256 : 512, 2) void attn_bwd_pair_kernel(BwdParams p, int dkdv_blocks) {
  const int block = blockIdx.x;
  if constexpr (DQK == 64) {
    __shared__ __attribute__((aligned(1024))) char smem[larger(dkdv_d64::kSmem, dq_duo::kSmem<64>)];
    if (block < dkdv_blocks) dkdv_d64::body<CAUSAL, KvT>(p, smem, block);
    else dq_duo::body<64, CAUSAL, QT>(p, smem, block - dkdv_blocks);
  } else if constexpr (DQK == 128) {
    __shared__ __attribute__((aligned(1024))) char smem[larger(dkdv_d128::kSmem, dq_direct::kSmem<128>)];
    if (block < dkdv_blocks) dkdv_d128::body<CAUSAL, KvT, false>(p, smem, block);
    else dq_direct::body<128, CAUSAL, QT>(p, smem, block - dkdv_blocks);
  } else {
    __shared__ __attribute__((aligned(1024))) char smem[larger(dkdv_d192::kSmem, dq_direct::kSmem<192>)];
    if (block < dkdv_blocks) dkdv_d192::body<CAUSAL, KvT>(p, smem, block);
    else dq_direct::body<192, CAUSAL, QT>(p, smem, block - dkdv_blocks);
  }
}

template <int DQK, typename KvT, typename QT>
void launch_one(BwdParams p, bool causal, unsigned dkdv_blocks, hipStream_t st) {
  p.q_tiles = (p.Sq + 127) / 128;
  const dim3 grid(dkdv_blocks + (unsigned)(p.q_tiles * p.Hq * p.B)), block(DQK == 64 ? 256 : 512);
  if (causal) hipLaunchKernelGGL((attn_bwd_pair_kernel<DQK, true, KvT, QT>), grid, block, 0, st, p, (int)dkdv_blocks);
  else hipLaunchKernelGGL((attn_bwd_pair_kernel<DQK, false, KvT, QT>), grid, block, 0, st, p, (int)dkdv_blocks);
}

template <typename KvT, typename QT>
void launch_types(const BwdParams& p, int dqk, bool causal, unsigned dkdv_blocks, hipStream_t st) {
  if (dqk == 64) launch_one<64, KvT, QT>(p, causal, dkdv_blocks, st);
  else if (dqk == 128) launch_one<128, KvT, QT>(p, causal, dkdv_blocks, st);
  else launch_one<192, KvT, QT>(p, causal, dkdv_blocks, st);
}

}  // namespace

bool launch_bwd_pair(const BwdParams& p, int dqk, bool causal, bool dkdv_f32, bool dq_f32, unsigned dkdv_blocks, hipStream_t st) {
  if (dkdv_f32 && !dq_f32) return false;  // no caller: gradients that travel in fp32 come with an fp32 dQ accumulator
  if (dkdv_f32) launch_types<float, float>(p, dqk, causal, dkdv_blocks, st);
  else if (dq_f32) launch_types<__bf16, float>(p, dqk, causal, dkdv_blocks, st);
  else launch_types<__bf16, __bf16>(p, dqk, causal, dkdv_blocks, st);
  return true;
}

}  // namespace pith
