// Key/value-gradient kernel for head dims (64, 64) on gfx950. Same function as the other dK/dV kernels
// (pithtrain/operators/mla/triton.py:130-197, :331-384: P = exp2(kappa*s - lse2) in fp32, masked entries 0, P rounded to
// bf16 for dV += P^T dO, dS = P*(dP - delta) rounded to bf16 for dK += dS^T Q, fp32 accumulation, `scale` applied once).
//
// With 64 features one wave has registers for everything 32 keys need (K, V: 32; dK, dV accumulators: 64; S, dP: 32;
// P, dS fragments: 16), so no pair of waves has to share the work and hand P over through LDS as at 128 features. A
// workgroup is 4 waves = 128 keys of one (batch, kv head) and streams query tiles of 32 rows (of the query heads assigned
// to it); several workgroups share a compute unit and hide each other's vector work, first tiles and epilogue. Per
// interval a wave runs one matrix block
//     dV^T += dO(i-1)^T P(i-1) ;  dK^T += Q(i-1)^T dS(i-1) ;  S(i) = Q(i) K^T ;  dP(i) = dO(i) V^T
// and one vector block P(i), dS(i). Tiles go global -> LDS directly, two intervals ahead, into rings of four; the wait that
// ends an interval lets exactly that interval's loads stay in flight.
// The wave holds -V and starts dP from delta, so that its product yields delta - dP = -(dP - delta) without a subtraction
// per element; the sign goes with the factor -scale on the accumulated dK.
#pragma once

#include "attn_bwd_common.h"

namespace pith {
namespace dkdv_d64 {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kD = 64;
constexpr int kBM = 32;           // query rows per tile
constexpr int kBN = kDkdvBlockN;  // key rows per workgroup
static_assert(kBN == 32 * kWaves, "a wave owns 32 keys");
constexpr int kSlots = 4;         // tiles i-1 and i (in use), i+1 and i+2 (landing); a power of two
constexpr int kAhead = 4;         // fragment reads run this many products ahead in the matrix block
constexpr int kTile = kBM / 2 * kRowBytes128;   // two rows per 256-byte LDS row
constexpr int kStat = 2 * kBM * 4;              // lse[32], delta[32]; every wave keeps its own copy
constexpr int kSlot = 2 * kTile + kWaves * kStat;
constexpr int kTurn = kWaves * kRowsViaLdsBytes<kD / 32>;
constexpr int kSmem = kSlots * kSlot > kTurn ? kSlots * kSlot : kTurn;
constexpr int kLoads = 3;                       // load instructions per wave and tile

template <bool CAUSAL, typename OutT>
__device__ __forceinline__ void body(const BwdParams& p, char* smem, int block, int key_shift = 0) {
  constexpr int KS = kD / 16, DB = kD / 32;

  const int tid = threadIdx.x;
  if (block >= p.main_blocks) {  // workgroups appended to the grid: clear the rows behind the chunk's visible part
    zero_tail_block<OutT>(p, block - p.main_blocks, kD, kD, tid, kThreads);
    return;
  }
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, g = lane >> 5;

  // linear block id -> (key tile, kv head, batch, head part)
  const int per_level = p.Hkv * p.B * p.split;
  int n_tile, pos;
  decode_dkdv_block(block, per_level, p.tiles, n_tile, pos);
  const int part = pos % p.split;
  pos /= p.split;
  const int hk = pos % p.Hkv, b = pos / p.Hkv;
  const int heads_per_part = p.group / p.split;
  const int hq0 = hk * p.group + part * heads_per_part;

  const int kv_wg0 = n_tile * kBN;
  const int kv_wave0 = kv_wg0 + wave * 32;
  const int key = kv_wave0 + c;
  const int q_row_bytes = p.HqT * kD * 2;  // Q and dO rows
  const int64_t kv_row_stride = (int64_t)p.HkvT * kD;

  // Query tiles to visit: all of them, or from the workgroup's diagonal down under the causal mask, head by head.
  const int m_end = (p.Sq + kBM - 1) / kBM;
  const int m_first = CAUSAL ? min(max(kv_wg0 - key_shift, 0) / kBM, m_end) : 0;
  const int n_iter = (m_end - m_first) * heads_per_part;

  DirectPaired64<kBM, kThreads> mover;
  mover.init(q_row_bytes, 0, wave, lane);
  const char* q_base = reinterpret_cast<const char*>(p.q + b * p.q_bs);
  const char* do_base = reinterpret_cast<const char*>(p.dout + b * p.dout_bs);
  int req_h = hq0, req_m = m_first;  // next tile to request
  auto request = [&](int t) __attribute__((always_inline)) {
    char* const slot = smem + (t & (kSlots - 1)) * kSlot;
    const int row0 = req_m * kBM;
    const int64_t off = (int64_t)req_h * kD * 2 + (int64_t)row0 * q_row_bytes;
    mover.issue(q_base + off, p.Sq - row0, slot, wave, lane);
    mover.issue(do_base + off, p.Sq - row0, slot + kTile, wave, lane);
    const int row = min(row0 + c, p.Sq - 1);
    load_lds4((g == 0 ? p.lse : p.delta) + b * p.lse_bs + (int64_t)req_h * p.lse_hs + row, slot + 2 * kTile + wave * kStat);
    if (++req_m == m_end) {
      req_m = m_first;
      ++req_h;
    }
  };
  // stationary fragments: K and -V rows as B operands. Every wave stages its own rows in the ring; the first tiles are
  // requested when all have been read.
  bf16x8 kf[KS], vf[KS];
  {
    static_assert(kWaves * 8192 <= kSmem, "areas of the stationary rows");
    char* const area = smem + wave * 8192;
    const int kv_row_bytes = (int)(kv_row_stride * 2);
    stage_rows32<false>(reinterpret_cast<const char*>(p.k + b * p.k_bs + (int64_t)hk * kD), kv_wave0, p.Skv, kv_row_bytes, area, lane);
    stage_rows32<false>(reinterpret_cast<const char*>(p.v + b * p.v_bs + (int64_t)hk * kD), kv_wave0, p.Skv, kv_row_bytes, area + 4096, lane);
    wait_staged();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kf[ks] = staged_fragment<false>(area, ks, c, g);
      vf[ks] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, staged_fragment<false>(area + 4096, ks, c, g)) ^ 0x80008000u);
    }
    __syncthreads();
  }
  if (n_iter > 0) request(0);
  if (n_iter > 1) request(1);
  if (n_iter > 2) request(2);

  f32x16 dk[DB], dv[DB];  // transposed: this lane's key, 32 features per block
#pragma unroll
  for (int o = 0; o < DB; ++o)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      dk[o][v] = 0.f;
      dv[o][v] = 0.f;
    }

  // per-lane read offsets (LDS row r holds tile row r in pieces 0-7 and r + 16 in pieces 8-15): straight fragment of the
  // tile's 32 rows, contraction step ks; transposed fragment of rows 16j..16j+15, feature block o
  const int s_base = straight_offset128(c & 15, g + 8 * (c >> 4));
  const int t_base[2] = {transposed_offset128(0, 0, 0, lane), transposed_offset128(0, 1, 0, lane)};
  auto s_frag = [&](const char* tile, int ks) __attribute__((always_inline)) {
    return *reinterpret_cast<const bf16x8*>(tile + (s_base ^ (ks << 5)));
  };
  auto t_frag = [&](const char* tile, int j, int o) __attribute__((always_inline)) {
    const int flip = (o << 6) | (j << 7);
    return lds_read_transposed_at(tile + (t_base[0] ^ flip), tile + (t_base[1] ^ flip));
  };

  f32x16 s, dp;             // S and delta - dP of a tile: rows = queries, column = this lane's key
  bf16x8 pf[2], dsf[2];     // P and -dS / scale as B operands, one fragment per 16 queries
  f32x4 lse4[4];

  auto start = [&](const char* slot) __attribute__((always_inline)) {
    const float* stat = reinterpret_cast<const float*>(slot + 2 * kTile + wave * kStat);
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) {
      const f32x4 d = *reinterpret_cast<const f32x4*>(stat + kBM + 8 * b4 + 4 * g);
      lse4[b4] = *reinterpret_cast<const f32x4*>(stat + 8 * b4 + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[4 * b4 + e] = 0.f;
        dp[4 * b4 + e] = d[e];
      }
    }
  };
  auto scores = [&](const char* slot) __attribute__((always_inline)) {
    start(slot);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = mfma32(s_frag(slot, ks), kf[ks], s);
      dp = mfma32(s_frag(slot + kTile, ks), vf[ks], dp);
    }
  };
  auto accumulate = [&](const char* slot) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < DB; ++o) {
        dv[o] = mfma32(t_frag(slot + kTile, j, o), pf[j], dv[o]);
        dk[o] = mfma32(t_frag(slot, j, o), dsf[j], dk[o]);
      }
  };
  auto matrix_block = [&](const char* prev, const char* cur) __attribute__((always_inline)) {
    constexpr int NT = 4 * DB, NS = 2 * KS;
    static_assert(kAhead <= NT, "look-ahead assumes it starts inside the gradient products");
    __builtin_amdgcn_s_setprio(2);
    bf16x8 aq[2][DB], ao[2][DB], bq[KS], bo[KS];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < DB; ++o) {
        ao[j][o] = t_frag(prev + kTile, j, o);
        aq[j][o] = t_frag(prev, j, o);
      }
    start(cur);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      bq[ks] = s_frag(cur, ks);
      bo[ks] = s_frag(cur + kTile, ks);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < DB; ++o) {
        dv[o] = mfma32(ao[j][o], pf[j], dv[o]);
        dk[o] = mfma32(aq[j][o], dsf[j], dk[o]);
      }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = mfma32(bq[ks], kf[ks], s);
      dp = mfma32(bo[ks], vf[ks], dp);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAhead, 0);
#pragma unroll
    for (int m = 0; m < NT - kAhead; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);  // lse and delta of the tile's rows
#pragma unroll
    for (int m = 0; m < NS; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
  };
  // P = exp2(kappa s - lse), masked entries 0; -dS / scale = P * (delta - dP)
  auto make_p_ds = [&](int m_tile) __attribute__((always_inline)) {
    const int q0 = m_tile * kBM;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = __builtin_amdgcn_exp2f(s[v] * p.kappa - lse4[v >> 2][v & 3]);
    if ((CAUSAL && q0 < kv_wave0 - key_shift + 31) || q0 + kBM > p.Sq) {  // wave-uniform: diagonal or ragged tile
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int qrow = q0 + acc_row(v, g);
        if ((CAUSAL && key - key_shift > qrow) || qrow >= p.Sq) s[v] = 0.f;
      }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) dp[v] *= s[v];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      pf[j] = to_bf16x8(s[8 * j], s[8 * j + 1], s[8 * j + 2], s[8 * j + 3], s[8 * j + 4], s[8 * j + 5], s[8 * j + 6], s[8 * j + 7]);
      dsf[j] = to_bf16x8(dp[8 * j], dp[8 * j + 1], dp[8 * j + 2], dp[8 * j + 3], dp[8 * j + 4], dp[8 * j + 5], dp[8 * j + 6], dp[8 * j + 7]);
    }
  };

  if (n_iter > 2) wait_staged<2 * kLoads>();
  else wait_staged();
  __syncthreads();
  if (n_iter > 0) {
    scores(smem);
    make_p_ds(m_first);
    if (n_iter > 2) wait_staged<kLoads>();
    else wait_staged();
    __syncthreads();  // tile 1 is there
    int mt = m_first;
    for (int i = 1; i < n_iter; ++i) {
      if (++mt == m_end) mt = m_first;
      const bool more = i + 2 < n_iter;
      if (more) request(i + 2);
      matrix_block(smem + ((i - 1) & (kSlots - 1)) * kSlot, smem + (i & (kSlots - 1)) * kSlot);
      make_p_ds(mt);
      // tile i + 1 has landed; the loads just requested may stay in flight (they are the wave's last memory operations)
      if (more) __builtin_amdgcn_s_waitcnt(0x0F70 | kLoads);
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    }
    accumulate(smem + ((n_iter - 1) & (kSlots - 1)) * kSlot);
  }
  __syncthreads();  // every wave is done with the rings

  // ---- epilogue: rows turned through LDS, first dV, then dK
  char* const turn = smem + wave * kRowsViaLdsBytes<DB>;
  if (p.split > 1) {  // packed fp32 partials
    const int64_t row_stride = (int64_t)p.Hkv * kD;
    const int64_t at = (((int64_t)part * p.B + b) * p.Skv + kv_wave0) * row_stride + (int64_t)hk * kD;
    store_rows32_via_lds<float, DB>(turn, p.ws_dv + at, row_stride, p.Skv - kv_wave0, dv, 1.f, false, lane);
    store_rows32_via_lds<float, DB>(turn, p.ws_dk + at, row_stride, p.Skv - kv_wave0, dk, -p.scale, false, lane);
  } else {
    const int64_t at = kv_wave0 * kv_row_stride + (int64_t)hk * kD;
    store_rows32_via_lds<OutT, DB>(turn, reinterpret_cast<OutT*>(p.dv) + b * p.dv_bs + at, kv_row_stride, p.Skv - kv_wave0, dv, 1.f, p.accumulate != 0, lane);
    store_rows32_via_lds<OutT, DB>(turn, reinterpret_cast<OutT*>(p.dk) + b * p.dk_bs + at, kv_row_stride, p.Skv - kv_wave0, dk, -p.scale, p.accumulate != 0, lane);
  }
}

}  // namespace dkdv_d64
}  // namespace pith
