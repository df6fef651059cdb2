// Key/value-gradient kernel for head dims (64, 64) on gfx950. Same function as the other dK/dV kernels
// (pithtrain/operators/mla/triton.py:130-197, :331-384: P = exp2(kappa*s - lse2) in fp32, masked entries 0, P rounded to
// bf16 for dV += P^T dO, dS = P*(dP - delta) rounded to bf16 for dK += dS^T Q, fp32 accumulation, `scale` applied once).
//
// With 64 features one wave has registers for everything 32 keys need (K, V: 32; dK, dV accumulators: 64; S, dP: 32;
// P, dS fragments: 16), so no pair of waves has to share the work and hand P over through LDS as at 128 features. A
// workgroup is 4 waves = 128 keys of one (batch, kv head) and streams query tiles of 32 rows (of the query heads assigned
// to it); two workgroups share a compute unit and hide each other's first tiles and epilogue. With 64 features the vector
// work of a tile (76 instructions) takes as long to issue as its 16 products, so the two are woven: step i runs
//     dV^T += dO(i-1)^T P(i-1) ;  dK^T += Q(i-1)^T dS(i-1)      between the exponentials of tile i (P)
//     S(i+1) = Q(i+1) K^T ;  dP(i+1) = dO(i+1) V^T              between the rest of its arithmetic (dS, bf16)
// with the step's three loads spread over the first half (sent back to back they held a wave up for 280 cycles). Tiles go global
// -> LDS directly, three steps ahead, into rings of eight; the wait that ends a step lets exactly its loads stay in flight.
// Against matrix block, then vector block (186 registers, or three workgroups of 168: equal): a step alone on its unit 0.70 ->
// 0.55 us, 1 x 2048 x 4/1 heads causal (both gradients) 52 -> 41 us; with every unit full the chip is at its power limit (1.9
// GHz) and 3 % are left: 1 x 8192 x 16/4 474 -> 459 us.
// The wave holds -V and starts dP from delta, so that its product yields delta - dP = -(dP - delta) without a subtraction
// per element; the sign goes with the factor -scale on the accumulated dK.
#pragma once

#include <type_traits>

#include "attn_bwd_common.h"

namespace pith {
namespace dkdv_d64 {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kD = 64;
constexpr int kBM = 32;           // query rows per tile
constexpr int kBN = kDkdvBlockN;  // key rows per workgroup
static_assert(kBN == 32 * kWaves, "a wave owns 32 keys");
constexpr int kSlots = 8;         // tiles i-1, i and i+1 (in use), i+2 and i+3 (landing); a power of two
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
  decode_dkdv_block(block, per_level, p.tiles, p.chunked, n_tile, pos);
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

  // one load per wave moves a quarter of a tile's rows; a head's last tile may be ragged
  using Mover = DirectPaired64<kBM, kThreads>;
  static_assert(Mover::kPerThread == 1, "one load per wave and tile");
  const int src_full = Mover::source(q_row_bytes, 0, 4 * wave + (lane >> 4), lane, kBM);
  const int src_last = Mover::source(q_row_bytes, 0, 4 * wave + (lane >> 4), lane, p.Sq - (m_end - 1) * kBM);
  // the next tile to request: addresses of its Q and dO rows, of its lse (lanes 0..31) and delta values, rows left from it on
  const int64_t tile_step = (int64_t)kBM * q_row_bytes;
  const int64_t head_step = kD * 2 - (m_end - 1 - m_first) * tile_step;  // from a head's last tile to the first one of the next
  const int64_t stat_head_step = p.lse_hs * 4 - (int64_t)(m_end - 1 - m_first) * kBM * 4;
  const int64_t first_row = (int64_t)m_first * kBM;
  const char* q_next = reinterpret_cast<const char*>(p.q + b * p.q_bs) + (int64_t)hq0 * kD * 2 + first_row * q_row_bytes;
  const char* do_next = reinterpret_cast<const char*>(p.dout + b * p.dout_bs) + (int64_t)hq0 * kD * 2 + first_row * q_row_bytes;
  const char* stat_next = reinterpret_cast<const char*>((g == 0 ? p.lse : p.delta) + b * p.lse_bs + (int64_t)hq0 * p.lse_hs + first_row);
  const int left_first = p.Sq - m_first * kBM;
  int left = left_first;
  // A tile's three requests, one at a time (the address unit takes 16 cycles for each, and a wave that sends them back to back
  // waits for it): parts 0 and 1 its Q and dO rows, part 2 its lse and delta; then on to the next tile.
  auto request_part = [&](int t, int part) __attribute__((always_inline)) {
    char* const slot = smem + (t & (kSlots - 1)) * kSlot;
    if (part < 2) load_lds16(part == 0 ? q_next : do_next, left >= kBM ? src_full : src_last, slot + part * kTile + wave * 1024);
    if (part == 2) {
      load_lds4(stat_next + min(c, left - 1) * 4, slot + 2 * kTile + wave * kStat);
      left -= kBM;
      const bool wrap = left <= 0;
      q_next += wrap ? head_step : tile_step;
      do_next += wrap ? head_step : tile_step;
      stat_next += wrap ? stat_head_step : kBM * 4;
      left = wrap ? left_first : left;
    }
  };
  auto request = [&](int t) __attribute__((always_inline)) {
    for (int part = 0; part < 3; ++part) request_part(t, part);
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

  // S and delta - dP of two tiles: rows = queries, column = this lane's key. One pair is turned into P and dS while the
  // products of the next tile fill the other.
  f32x16 s0, dp0, s1, dp1;
  bf16x8 pf[2], dsf[2];     // P and -dS / scale as B operands, one fragment per 16 queries

  auto slot_of = [&](int t) __attribute__((always_inline)) { return smem + (t & (kSlots - 1)) * kSlot; };
  auto stats = [&](const char* slot) __attribute__((always_inline)) { return reinterpret_cast<const float*>(slot + 2 * kTile + wave * kStat); };
  // fragment m of the gradient products of the tile in `slot`: 16-row step m / 4, feature block m / 2 % 2, dO (for dV) or Q (for dK)
  auto grad_frag = [&](const char* slot, int m) __attribute__((always_inline)) { return t_frag(slot + (m & 1 ? 0 : kTile), m >> 2, m >> 1 & 1); };
  auto grad_product = [&](bf16x8 a, int m) __attribute__((always_inline)) {
    f32x16& acc = m & 1 ? dk[m >> 1 & 1] : dv[m >> 1 & 1];
    acc = mfma32(a, m & 1 ? dsf[m >> 2] : pf[m >> 2], acc);
  };
  // fragment m of its score products: contraction step m / 2, Q (for S) or dO (for dP)
  auto score_frag = [&](const char* slot, int m) __attribute__((always_inline)) { return s_frag(slot + (m & 1 ? kTile : 0), m >> 1); };
  auto start = [&](const char* slot, f32x16& x, f32x16& y) __attribute__((always_inline)) {
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) {
      const f32x4 d = *reinterpret_cast<const f32x4*>(stats(slot) + kBM + 8 * b4 + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[4 * b4 + e] = 0.f;
        y[4 * b4 + e] = d[e];
      }
    }
  };
  // x <- P = exp2(kappa x - lse) of the tile in `slot`, between the gradient products of the tile in `prev` (GRAD)
  // and the requests for tile `ask` (ASK)
  auto make_p = [&](const char* slot, const char* prev, f32x16& x, int ask, auto grad_tag, auto ask_tag) __attribute__((always_inline)) {
    constexpr bool GRAD = decltype(grad_tag)::value, ASK = decltype(ask_tag)::value;
    constexpr int N = 4 * DB;
    f32x4 lse4[4];
    bf16x8 a[N];
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) lse4[b4] = *reinterpret_cast<const f32x4*>(stats(slot) + 8 * b4 + 4 * g);
    if constexpr (GRAD) {
#pragma unroll
      for (int m = 0; m < kAhead; ++m) a[m] = grad_frag(prev, m);
    }
#pragma unroll
    for (int m = 0; m < N; ++m) {
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (GRAD) {
        if (m + kAhead < N) a[m + kAhead] = grad_frag(prev, m + kAhead);
        grad_product(a[m], m);
      }
      if (ASK && m % 2 == 0 && m < 6) request_part(ask, m / 2);
#pragma unroll
      for (int v = 2 * m; v < 2 * m + 2; ++v) x[v] = __builtin_amdgcn_exp2f(x[v] * p.kappa - lse4[v >> 2][v & 3]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // masked entries 0
  auto mask_p = [&](int m_tile, f32x16& x) __attribute__((always_inline)) {
    const int q0 = m_tile * kBM;
    if ((CAUSAL && q0 < kv_wave0 - key_shift + 31) || q0 + kBM > p.Sq) {  // wave-uniform: diagonal or ragged tile
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int qrow = q0 + acc_row(v, g);
        if ((CAUSAL && key - key_shift > qrow) || qrow >= p.Sq) x[v] = 0.f;
      }
    }
  };
  // P and -dS / scale = P * (delta - dP) as fragments, between the score products of the tile in `next` (SCORES), which
  // leave S in nx and delta - dP in ny
  auto make_ds = [&](const char* next, const f32x16& x, const f32x16& y, f32x16& nx, f32x16& ny, auto scores_tag) __attribute__((always_inline)) {
    constexpr bool SCORES = decltype(scores_tag)::value;
    constexpr int N = 2 * KS;
    static_assert(N == 8, "two accumulator values per product");
    bf16x8 a[N];
    u32x4 pu[2], du[2];
    if constexpr (SCORES) {
      start(next, nx, ny);
#pragma unroll
      for (int m = 0; m < kAhead; ++m) a[m] = score_frag(next, m);
    }
#pragma unroll
    for (int m = 0; m < N; ++m) {
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (SCORES) {
        if (m + kAhead < N) a[m + kAhead] = score_frag(next, m + kAhead);
        if (m & 1) ny = mfma32(a[m], vf[m >> 1], ny);
        else nx = mfma32(a[m], kf[m >> 1], nx);
      }
      uint32_t pw = pack_bf16x2(x[2 * m], x[2 * m + 1]), dw = pack_bf16x2(y[2 * m] * x[2 * m], y[2 * m + 1] * x[2 * m + 1]);
      asm volatile("" : "+v"(pw), "+v"(dw));  // formed here, not where they are used
      pu[m >> 2][m & 3] = pw;
      du[m >> 2][m & 3] = dw;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      pf[j] = __builtin_bit_cast(bf16x8, pu[j]);
      dsf[j] = __builtin_bit_cast(bf16x8, du[j]);
    }
  };
  constexpr std::true_type yes;
  constexpr std::false_type no;
  auto first_scores = [&](const char* slot, f32x16& x, f32x16& y) __attribute__((always_inline)) {
    start(slot, x, y);
#pragma unroll
    for (int m = 0; m < 2 * KS; ++m) {
      if (m & 1) y = mfma32(score_frag(slot, m), vf[m >> 1], y);
      else x = mfma32(score_frag(slot, m), kf[m >> 1], x);
    }
  };

  if (n_iter > 2) wait_staged<2 * kLoads>();
  else wait_staged();
  __syncthreads();
  if (n_iter > 0) {
    first_scores(smem, s0, dp0);
    if (n_iter > 2) wait_staged<kLoads>();
    else wait_staged();
    __syncthreads();  // tile 1 is there
    // Step i: the gradient products of tile i - 1 between the exponentials of tile i, then the score products of tile i + 1
    // between the rest of its arithmetic. Tile i + 3 is requested; tile i + 2 has landed when the step ends.
    int mt = m_first;
    auto step = [&](int i, auto grad_tag, auto ask_tag, f32x16& x, f32x16& y, f32x16& nx, f32x16& ny) __attribute__((always_inline)) {
      make_p(slot_of(i), slot_of(i - 1), x, i + 3, grad_tag, ask_tag);
      mask_p(mt, x);
      make_ds(slot_of(i + 1), x, y, nx, ny, yes);
      if (++mt == m_end) mt = m_first;
      // the loads just requested may stay in flight (they are the wave's last memory operations)
      wait_staged<decltype(ask_tag)::value ? kLoads : 0>();
      __syncthreads();
    };
    // the last tile: no scores behind it
    auto last = [&](int i, auto grad_tag, f32x16& x, f32x16& y) __attribute__((always_inline)) {
      make_p(slot_of(i), slot_of(i - 1), x, 0, grad_tag, no);
      mask_p(mt, x);
      make_ds(smem, x, y, s1, dp1, no);
#pragma unroll
      for (int m = 0; m < 4 * DB; ++m) grad_product(grad_frag(slot_of(i), m), m);
    };
    if (n_iter == 1) {
      last(0, no, s0, dp0);
    } else {
      if (n_iter > 3) step(0, no, yes, s0, dp0, s1, dp1);
      else step(0, no, no, s0, dp0, s1, dp1);
      int i = 1;
      for (; i + 4 < n_iter; i += 2) {
        step(i, yes, yes, s1, dp1, s0, dp0);
        step(i + 1, yes, yes, s0, dp0, s1, dp1);
      }
      // one request is left if i + 4 == n_iter; two to four steps without one, and the last tile
      if (i + 3 < n_iter) {
        step(i, yes, yes, s1, dp1, s0, dp0);
        s1 = s0;
        dp1 = dp0;
        ++i;
      }
      for (; i + 1 < n_iter; ++i) {
        step(i, yes, no, s1, dp1, s0, dp0);
        s1 = s0;
        dp1 = dp0;
      }
      last(i, yes, s1, dp1);
    }
  }
  __syncthreads();  // every wave is done with the rings

  // ---- epilogue: rows turned through LDS, first dV, then dK
  char* const turn = smem + wave * kRowsViaLdsBytes<DB>;
  if (p.split > 1) {  // packed fp32 partials
    const int64_t row_stride = (int64_t)p.Hkv * kD;
    const int64_t at = (((int64_t)part * p.B + b) * p.Skv + kv_wave0) * row_stride + (int64_t)hk * kD;
    store_rows32_via_lds<float, DB>(turn, p.ws_dv + at, row_stride, p.Skv - kv_wave0, dv, 1.f, false, lane, p.through_parts);
    store_rows32_via_lds<float, DB>(turn, p.ws_dk + at, row_stride, p.Skv - kv_wave0, dk, -p.scale, false, lane, p.through_parts);
  } else {
    const int64_t at = kv_wave0 * kv_row_stride + (int64_t)hk * kD;
    store_rows32_via_lds<OutT, DB>(turn, reinterpret_cast<OutT*>(p.dv) + b * p.dv_bs + at, kv_row_stride, p.Skv - kv_wave0, dv, 1.f, p.accumulate != 0, lane, p.through_dkv);
    store_rows32_via_lds<OutT, DB>(turn, reinterpret_cast<OutT*>(p.dk) + b * p.dk_bs + at, kv_row_stride, p.Skv - kv_wave0, dk, -p.scale, p.accumulate != 0, lane, p.through_dkv);
  }
}

}  // namespace dkdv_d64
}  // namespace pith
