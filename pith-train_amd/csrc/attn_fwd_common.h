// Declarations shared by the forward kernels.
#pragma once

#include <type_traits>

#include "attn_tiles.h"

namespace pith {

constexpr int kFwdBlockN = 64;            // keys per LDS tile
constexpr float kRescaleLimit = 256.f;    // bound on a P value before the running maximum is refreshed, tested on row sums

struct FwdParams {
  const __bf16* q;
  const __bf16* k;
  const __bf16* v;
  __bf16* o;
  float* lse;
  int Sq, Skv, Hq, Hkv, group;  // group = Hq / Hkv
  int B, m_tiles;
  int through_o;  // O is written through (through_results)
  int chunked;  // tiles from which the heads are taken in chunks (decode_block; 128-row workgroups only)
  int64_t q_bs, k_bs, v_bs, o_bs, lse_bs, lse_hs;
  float kappa;  // scale * log2(e)
  // keys in two parts (k_pe != nullptr): k holds the first 128 features per head, k_pe the last 64,
  // one vector per position shared by all heads (batch / row strides in elements)
  const __bf16* k_pe;
  int64_t k_pe_bs, k_pe_rs;
  // merge with the running result of the rows (prev_o != nullptr; non-causal direct-load kernels only): prev_o is
  // bf16 or fp32 (prev_f32), the merged result goes to o (bf16, may be null then) and / or acc_o (fp32, may be null);
  // lse holds the running LSE on entry and the merged LSE on return
  const void* prev_o;
  int prev_f32;
  int64_t prev_bs;
  float* acc_o;
  int64_t acc_bs;
  int o_r0, o_r1, acc_r0, acc_r1;  // query rows [r0, r1) that receive o / acc_o when merging (multiples of 32, or Sq)
};

// The same over several chunks of keys: k, v, k_pe and Skv of the base are unused, its batch strides hold for every chunk.
struct FwdChunkParams : FwdParams {
  int n_chunks;
  KeyChunk chunk[kMaxChunks];
};

template <bool MULTI>
using FwdArgs = std::conditional_t<MULTI, FwdChunkParams, FwdParams>;
__host__ __device__ __forceinline__ KeyChunk chunk_of(const FwdParams& p, int) { return KeyChunk{p.k, p.v, p.k_pe, p.Skv, 0}; }
__host__ __device__ __forceinline__ const KeyChunk& chunk_of(const FwdChunkParams& p, int i) { return p.chunk[i]; }
__host__ __device__ __forceinline__ int chunk_count(const FwdParams&) { return 1; }
__host__ __device__ __forceinline__ int chunk_count(const FwdChunkParams& p) { return p.n_chunks; }

// Forward with one 8-wave workgroup per compute unit: attn_fwd_direct.hip. dqk = 128, or 192 with half; half = workgroups
// of 128 query rows whose wave pairs split the keys of every tile (see there) instead of 256-row workgroups.
void launch_fwd_direct(const FwdParams& p, int dqk, bool causal, bool half, hipStream_t stream);
void launch_fwd_direct(const FwdChunkParams& p, int dqk, bool causal, bool half, hipStream_t stream);

// attn_fwd_duo.hip. parts = 1: two (64 features: three) 4-wave workgroups of 128 query rows per compute unit; 2 (64
// features) or 4: one 8-wave workgroup of 128 or 64 rows, whose key stream is split in that many parts; 3: two or more 4-wave
// workgroups of 64 rows, whose key stream is split in two.
void launch_fwd_duo(const FwdParams& p, int dqk, int parts, bool causal, hipStream_t stream);
void launch_fwd_duo(const FwdChunkParams& p, int dqk, int parts, bool causal, hipStream_t stream);

}  // namespace pith
