// Backward of a query block over SEVERAL key/value chunks (a ring share whose chunks are all at hand) in one launch, or two:
// the workgroup bodies of the chunk-pair kernels behind other addressing.
//   dK/dV  a workgroup belongs to one chunk (found from its block id) and runs the masked body on that chunk's view of the
//          call; in chunks without a mask all key positions lie below the first query row.
//   dQ     a workgroup walks the key tiles of every chunk its rows see as one stream, dQ stays in registers throughout and is
//          written once, as bf16 (no fp32 accumulator that every ring step reads and writes, no cast at the end).
// As for chunk pairs, small launches put both into one grid (attn_bwd_pair.hip), here with the longer kind first: dQ
// workgroups walk all chunks, and started behind the dK/dV ones of every chunk they are what the launch ends on. Measured,
// dK/dV first against dQ first: 1021 rows x 16 heads of 192, 4 ranks, contiguous 135 -> 122 us; 1024 x 16 of 192, zigzag
// 118 -> 96; 1024 x 8/2 of 128, rank 0 102 -> 85; 2 x 1536 x 16/4 of 64 207 -> 179; 2048 x 4 of 192, 8 ranks 290 -> 245.
#include "attn_bwd_common.h"
#include "attn_bwd_dkdv_d128.h"
#include "attn_bwd_dkdv_d192.h"
#include "attn_bwd_dkdv_d64.h"
#include "attn_bwd_dq_direct.h"
#include "attn_bwd_dq_duo.h"

namespace pith {
namespace {

constexpr int larger(int a, int b) { return a > b ? a : b; }

template <int DQK>
constexpr int kDkdvSmem = DQK == 64 ? dkdv_d64::kSmem : DQK == 128 ? dkdv_d128::kSmem : dkdv_d192::kSmem;
template <int DQK>
constexpr int kDkdvThreads = DQK == 64 ? dkdv_d64::kThreads : 512;

template <int DQK, bool EMIT_DS = false>
__device__ __forceinline__ void dkdv_body(const BwdChunkParams& p, char* smem, int block) {
  int key_shift;
  const BwdParams r = dkdv_chunk_params<DQK, DQK == 64 ? 64 : 128>(p, block, key_shift);
  if constexpr (DQK == 64) dkdv_d64::body<true, __bf16>(r, smem, block, key_shift);
  else if constexpr (DQK == 128) dkdv_d128::body<true, __bf16, false>(r, smem, block, key_shift);
  else dkdv_d192::body<true, __bf16, EMIT_DS>(r, smem, block, key_shift);
}

template <int DQK, bool EMIT_DS = false>
__global__ __launch_bounds__(kDkdvThreads<DQK>, 2) void attn_bwd_dkdv_chunks_kernel(BwdChunkParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[kDkdvSmem<DQK>];
  dkdv_body<DQK, EMIT_DS>(p, smem, blockIdx.x);
}

template <int DQK>
__global__ __launch_bounds__(dq_duo::kThreads, 2) void attn_bwd_dq_duo_chunks_kernel(BwdChunkParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[dq_duo::kSmem<DQK>];
  dq_duo::body<DQK, true, __bf16, true>(p, smem, blockIdx.x);
}

template <int DQK>
__global__ __launch_bounds__(kDkdvThreads<DQK>, 2) void attn_bwd_pair_chunks_kernel(BwdChunkParams p, int dkdv_blocks, int dq_first) {
  const int dq_blocks = gridDim.x - dkdv_blocks;
  const int block = dq_first ? ((int)blockIdx.x < dq_blocks ? dkdv_blocks + blockIdx.x : blockIdx.x - dq_blocks) : blockIdx.x;
  if constexpr (DQK == 64) {
    __shared__ __attribute__((aligned(1024))) char smem[larger(kDkdvSmem<64>, dq_duo::kSmem<64>)];
    if (block < dkdv_blocks) dkdv_body<64>(p, smem, block);
    else dq_duo::body<64, true, __bf16, true>(p, smem, block - dkdv_blocks);
  } else {
    __shared__ __attribute__((aligned(1024))) char smem[larger(kDkdvSmem<DQK>, dq_direct::kSmem<DQK>)];
    if (block < dkdv_blocks) dkdv_body<DQK>(p, smem, block);
    else dq_direct::body<DQK, true, __bf16, true>(p, smem, block - dkdv_blocks);
  }
}

template <int DQK>
void launch_dim(const BwdChunkParams& p, bool one_grid, bool dq_first, unsigned dkdv_blocks, hipStream_t st) {
  const unsigned dq_blocks = (unsigned)(p.q_tiles * p.Hq * p.B);
  if (one_grid) {
    hipLaunchKernelGGL((attn_bwd_pair_chunks_kernel<DQK>), dim3(dkdv_blocks + dq_blocks), dim3(kDkdvThreads<DQK>), 0, st, p, (int)dkdv_blocks, (int)dq_first);
    return;
  }
  hipLaunchKernelGGL((attn_bwd_dkdv_chunks_kernel<DQK>), dim3(dkdv_blocks), dim3(kDkdvThreads<DQK>), 0, st, p);
  hipLaunchKernelGGL((attn_bwd_dq_duo_chunks_kernel<DQK>), dim3(dq_blocks), dim3(dq_duo::kThreads), 0, st, p);
}

}  // namespace

void launch_bwd_chunks(const BwdChunkParams& p, int dqk, bool one_grid, bool dq_first, unsigned dkdv_blocks, hipStream_t st) {
  if (p.ds != nullptr) {
    hipLaunchKernelGGL((attn_bwd_dkdv_chunks_kernel<192, true>), dim3(dkdv_blocks), dim3(kDkdvThreads<192>), 0, st, p);
    launch_dq_from_ds_chunks(p, st);
    return;
  }
  if (dqk == 64) launch_dim<64>(p, one_grid, dq_first, dkdv_blocks, st);
  else if (dqk == 128) launch_dim<128>(p, one_grid, dq_first, dkdv_blocks, st);
  else launch_dim<192>(p, one_grid, dq_first, dkdv_blocks, st);
}

}  // namespace pith
