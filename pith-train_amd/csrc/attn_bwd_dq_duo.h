// Query-gradient kernel for head dims (64, 64), (128, 128) and (192, 128) on gfx950 with SMALL workgroups: 4 wavefronts,
// 128 query rows, two of them per compute unit. Same function and numerics as
// attn_bwd_dq_direct.hip (pithtrain/operators/mla/triton.py:205-266, :392-441: P = exp2(kappa*s - lse2) in fp32, masked
// entries 0, dS = P*(dP - delta) rounded to bf16, fp32 accumulation of dQ += dS K, `scale` applied once at the end).
//
// A wave owns 32 query rows (Q^T, dO^T, lse and delta stationary) and walks key tiles of 32; per interval one matrix block
//     dQ^T += K(i-1)^T dS(i-1)^T ;  S(i)^T = K(i) Q^T ;  dP(i)^T = V(i) dO^T
// and one vector block dS(i). Nothing inside a wave overlaps the two; the two workgroups of a compute unit do (each SIMD
// holds one wave of either), and they also hide each other's first tiles, diagonal and epilogue. Tiles of 32 keys keep S,
// dP and dS at 40 registers, which is what lets 192 features fit; they are requested two intervals ahead into rings of
// four, and the wait that ends an interval counts: it lets exactly the loads of that interval stay in flight.
// Bound by the matrix pipe (three products executed for the one that counts). Measured, executed products: 8192 x 8192 x
// 32 heads of 128 features 1284 TFLOP/s (1242 for the 256-row kernel with interleaved halves it replaces), 2 x 4096 x 16 of 64
// features 1033 (915 register-staged), 4096 x 4096 x 16 of 192 features 1219 (1156 with 128-row workgroups splitting keys).
// At 64 features the two blocks are woven as in attn_bwd_dkdv_d64.h (229 registers; in blocks it took 150, and three workgroups
// to a unit: equal alone, slower beside dK/dV workgroups, see one_grid).
#pragma once

#include "attn_bwd_common.h"

namespace pith {
namespace dq_duo {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kBM = 32 * kWaves;  // query rows per workgroup
constexpr int kBN = 32;           // keys per tile

template <int DQK>
struct DqDuoLayout {
  static constexpr int kDv = DQK == 64 ? 64 : 128;
  // ring depth: tiles i-1 and i (in use), i+1 and i+2 (landing), at 64 features i-1 to i+1 and i+2, i+3; a power of two
  static constexpr int kSlots = DQK == 64 ? 8 : 4;
  static constexpr int kPair = kBN / 2 * kRowBytes128, kFull = kBN * kRowBytes128;  // 64- and 128-feature tiles
  static constexpr int kKTile = DQK == 64 ? kPair : DQK == 128 ? kFull : kFull + kPair;
  static constexpr int kVTile = kDv == 64 ? kPair : kFull;
  static constexpr int kRings = kSlots * (kKTile + kVTile);
  static constexpr int kTurnBlocks = DQK == 192 ? 3 : DQK / 32;  // feature blocks the epilogue turns at a time
  static constexpr int kTurn = kWaves * kRowsViaLdsBytes<kTurnBlocks>;
  static constexpr int kSmem = kRings > kTurn ? kRings : kTurn;
  static constexpr int kLoads = (DQK == 64 ? 1 : DQK == 128 ? 2 : 3) + (kDv == 64 ? 1 : 2);  // load instructions per wave and tile
};

template <int DQK>
constexpr int kSmem = DqDuoLayout<DQK>::kSmem;

template <int DQK, bool CAUSAL, typename OutT, bool MULTI = false>
__device__ __forceinline__ void body(const BwdArgs<MULTI>& p, char* smem, int block) {
  using L = DqDuoLayout<DQK>;
  constexpr int kDv = L::kDv, KS = DQK / 16, VS = kDv / 16, DB = DQK / 32, kSlots = L::kSlots;
  constexpr bool kPaired = DQK == 64;
  constexpr int kAhead = DQK == 192 ? 3 : 4;  // fragment reads run this many products ahead in the matrix block
  char* const kbuf = smem;
  char* const vbuf = smem + kSlots * L::kKTile;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, g = lane >> 5;

  int m_tile, h, b;
  decode_block(block, p.Hq, p.B, p.q_tiles, p.group, m_tile, h, b, p.chunked);
  const int hk = h / p.group;
  const int m0 = m_tile * kBM;
  const int q_wave0 = m0 + wave * 32;
  const int qrow = q_wave0 + c;

  const int64_t q_row_stride = (int64_t)p.HqT * DQK;
  const int64_t do_row_stride = (int64_t)p.HqT * kDv;
  // keys in two parts: K rows hold 128 features per head, the last 64 come from k_pe (no head offset)
  const bool two_part = DQK == 192 && chunk_of(p, 0).k_pe != nullptr;
  const int k_head_elems = two_part ? 128 : DQK;
  const int k_row_bytes = p.HkvT * k_head_elems * 2, v_row_bytes = p.HkvT * kDv * 2;
  const int kx_row_bytes = two_part ? (int)p.k_pe_rs * 2 : k_row_bytes;
  // a chunk's first row in K, in the source of features 128.. and in V
  auto k_rows = [&](int id) __attribute__((always_inline)) {
    return reinterpret_cast<const char*>(chunk_of(p, id).k + b * p.k_bs + (int64_t)hk * k_head_elems);
  };
  auto kx_rows = [&](int id) __attribute__((always_inline)) {
    return two_part ? reinterpret_cast<const char*>(chunk_of(p, id).k_pe + b * p.k_pe_bs) : k_rows(id);
  };
  auto v_rows = [&](int id) __attribute__((always_inline)) {
    return reinterpret_cast<const char*>(chunk_of(p, id).v + b * p.v_bs + (int64_t)hk * kDv);
  };

  const ChunkRange<MULTI, CAUSAL, kBN> range(p, m0 + kBM);
  int n_wg = range.tiles_full, n_wave = range.tiles_full;  // key tiles this workgroup / this wave visits
  if (CAUSAL) {
    const int tiles = (chunk_of(p, range.last).rows + kBN - 1) / kBN;
    n_wg += min(tiles, (m0 + kBM - 1) / kBN + 1);
    n_wave += min(tiles, (q_wave0 + 31) / kBN + 1);
  }
  if (CAUSAL) n_wave = tiles_of_wave(n_wave, q_wave0, p.Sq);
  TileSource<MULTI, CAUSAL, kBN> k_src(p, range, k_row_bytes, k_rows), kx_src(p, range, kx_row_bytes, kx_rows), v_src(p, range, v_row_bytes, v_rows);
  TileMask<MULTI, CAUSAL, kBN> mask(p, range);

  DirectTile128<kBN, kThreads> vmover, kmover;
  DirectPaired64<kBN, kThreads> vpmover, kpmover;
  if constexpr (kPaired) {
    vpmover.init(v_row_bytes, 0, wave, lane);
    kpmover.init(k_row_bytes, 0, wave, lane);
  } else {
    vmover.init(v_row_bytes, wave, lane);
    kmover.init(k_row_bytes, wave, lane);
    if constexpr (DQK == 192) kpmover.init(kx_row_bytes, two_part ? 0 : 256, wave, lane);
  }
  // one operand at a time, without a branch: source offsets formed on the spot, and behind the last tile that one again, into a
  // slot that nobody reads (64 features, one chunk)
  auto request_k = [&](int t) __attribute__((always_inline)) {
    const int at = min(t, n_wg - 1);
    kpmover.issue_clamped(k_src.src(at), k_src.left(at), kbuf + (t & (kSlots - 1)) * L::kKTile, wave, lane);
  };
  auto request_v = [&](int t) __attribute__((always_inline)) {
    const int at = min(t, n_wg - 1);
    vpmover.issue_clamped(v_src.src(at), k_src.left(at), vbuf + (t & (kSlots - 1)) * L::kVTile, wave, lane);
  };
  auto request = [&](int t) __attribute__((always_inline)) {
    char* const ks = kbuf + (t & (kSlots - 1)) * L::kKTile;
    char* const vs = vbuf + (t & (kSlots - 1)) * L::kVTile;
    const char* const ksrc = k_src.src(t);
    const char* const vsrc = v_src.src(t);
    const int left = k_src.left(t);
    if constexpr (kPaired) {
      kpmover.issue(ksrc, left, ks, wave, lane);
      vpmover.issue(vsrc, left, vs, wave, lane);
    } else if constexpr (DQK == 128) {
      kmover.issue(ksrc, left, ks, wave, lane);
      vmover.issue(vsrc, left, vs, wave, lane);
    } else {  // no register to spare for source offsets: reloading a spilled one would wait for the tiles in flight
      kmover.issue_clamped(ksrc, left, ks, wave, lane);
      kpmover.issue_clamped(kx_src.src(t), left, ks + L::kFull, wave, lane);
      vmover.issue_clamped(vsrc, left, vs, wave, lane);
      kx_src.advance(p, range, kx_rows);
    }
    k_src.advance(p, range, k_rows);
    v_src.advance(p, range, v_rows);
  };
  // stationary B operands (column = query row), lse and delta of this lane's row. Every wave stages its own rows in the rings,
  // which they fill exactly; the first tiles are requested when all have been read.
  bf16x8 qf[KS], dof[VS];
  float lse_q, delta_q;
  {
    constexpr int kQArea = kPaired ? 4096 : 8192 + (DQK == 192 ? 4096 : 0), kDoArea = kPaired ? 4096 : 8192;
    static_assert(kWaves * (kQArea + kDoArea) <= L::kSmem, "areas of the query-side rows");
    char* const q_area = smem + wave * (kQArea + kDoArea);
    char* const do_area = q_area + kQArea;
    const int row = qrow < p.Sq ? qrow : p.Sq - 1;
    lse_q = p.lse[b * p.lse_bs + (int64_t)h * p.lse_hs + row];
    delta_q = p.delta[b * p.lse_bs + (int64_t)h * p.lse_hs + row];
    const char* const qsrc = reinterpret_cast<const char*>(p.q + b * p.q_bs + (int64_t)h * DQK);
    const char* const dsrc = reinterpret_cast<const char*>(p.dout + b * p.dout_bs + (int64_t)h * kDv);
    const int q_row_bytes = (int)(q_row_stride * 2), do_row_bytes = (int)(do_row_stride * 2);
    stage_rows32<!kPaired>(qsrc, q_wave0, p.Sq, q_row_bytes, q_area, lane);
    if constexpr (DQK == 192) stage_rows32<false>(qsrc + 256, q_wave0, p.Sq, q_row_bytes, q_area + 8192, lane);
    stage_rows32<!kPaired>(dsrc, q_wave0, p.Sq, do_row_bytes, do_area, lane);
    wait_staged();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = ks < 8 ? staged_fragment<!kPaired>(q_area, ks, c, g) : staged_fragment<false>(q_area + 8192, ks - 8, c, g);
#pragma unroll
    for (int ks = 0; ks < VS; ++ks) dof[ks] = staged_fragment<!kPaired>(do_area, ks, c, g);
    __syncthreads();
  }
  request(0);
  if (n_wg > 1) request(1);
  if (n_wg > 2) request(2);

  // per-lane read offsets. Straight fragment of the tile's 32 keys, contraction step ks; transposed fragment of keys
  // 16j..16j+15, feature block i. A 64-feature tile holds key r in pieces 0-7 and key r + 16 in pieces 8-15 of LDS row r.
  int s_base = straight_offset128(c, g);
  int x_base = straight_offset128(c & 15, g + 8 * (c >> 4));
  int t_base[2] = {transposed_offset128(0, 0, 0, lane), transposed_offset128(0, 1, 0, lane)};
  // 192 and 64 features: one base per tile part lives across the loop, the derived offsets are formed anew in every interval
  // (hoisted out of it they would push accumulators into scratch memory)
  auto refresh_offsets = [&]() __attribute__((always_inline)) {
    if constexpr (DQK != 128) asm volatile("" : "+v"(s_base), "+v"(x_base), "+v"(t_base[0]), "+v"(t_base[1]));
  };
  auto k_frag = [&](const char* kt, int ks) __attribute__((always_inline)) {
    const int off = kPaired ? x_base ^ (ks << 5) : ks < 8 ? s_base ^ (ks << 5) : L::kFull + (x_base ^ ((ks - 8) << 5));
    return *reinterpret_cast<const bf16x8*>(kt + off);
  };
  auto v_frag = [&](const char* vt, int ks) __attribute__((always_inline)) {
    return *reinterpret_cast<const bf16x8*>(vt + ((kPaired ? x_base : s_base) ^ (ks << 5)));
  };
  auto kt_frag = [&](const char* kt, int j, int i) __attribute__((always_inline)) {
    int flip, add;
    if (kPaired) { flip = (i << 6) | (j << 7); add = 0; }
    else if (i < 4) { flip = i << 6; add = j * 16 * kRowBytes128; }
    else { flip = ((i - 4) << 6) | (j << 7); add = L::kFull; }
    return lds_read_transposed_at(kt + (t_base[0] ^ flip) + add, kt + (t_base[1] ^ flip) + add);
  };

  f32x16 acc[DB];
#pragma unroll
  for (int o = 0; o < DB; ++o)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[o][v] = 0.f;
  f32x16 s, dp;
  bf16x8 dsf[2];

  auto start = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = 0.f;
      dp[v] = -delta_q;  // dP starts from -delta: dS = P * (dP - delta) without a subtraction per element
    }
  };
  auto scores = [&](const char* kt, const char* vt) __attribute__((always_inline)) {
    start();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = mfma32(k_frag(kt, ks), qf[ks], s);
      if (ks < VS) dp = mfma32(v_frag(vt, ks), dof[ks], dp);
    }
  };
  auto accumulate = [&](const char* kt) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < DB; ++o) acc[o] = mfma32(kt_frag(kt, j, o), dsf[j], acc[o]);
  };
  // dQ^T += K(prev)^T dS(prev)^T, then S^T and dP^T of the next tile, fragment reads kAhead products ahead
  auto matrix_block = [&](const char* kprev, const char* kt, const char* vt) __attribute__((always_inline)) {
    constexpr int NT = 2 * DB, NS = KS + VS;
    __builtin_amdgcn_s_setprio(2);
    bf16x8 at[2][DB], ak[KS], av[VS];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < DB; ++o) at[j][o] = kt_frag(kprev, j, o);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      ak[ks] = k_frag(kt, ks);
      if (ks < VS) av[ks] = v_frag(vt, ks);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < DB; ++o) acc[o] = mfma32(at[j][o], dsf[j], acc[o]);
    start();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = mfma32(ak[ks], qf[ks], s);
      if (ks < VS) dp = mfma32(av[ks], dof[ks], dp);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAhead, 0);
#pragma unroll
    for (int m = 0; m < NT - kAhead; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
#pragma unroll
    for (int m = 0; m < NS; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
  };
  // P = exp2(kappa s - lse), masked entries 0, dS = P * (dP - delta) -> bf16
  auto make_ds = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = __builtin_amdgcn_exp2f(s[v] * p.kappa - lse_q);
    if (mask.partial(range, t, q_wave0)) {  // wave-uniform
      const int limit = mask.limit(range, qrow), n0 = mask.key0(t);
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (n0 + acc_row(v, g) > limit) s[v] = 0.f;
    }
    mask.advance(p, range);
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] *= dp[v];
#pragma unroll
    for (int j = 0; j < 2; ++j)
      dsf[j] = to_bf16x8(s[8 * j], s[8 * j + 1], s[8 * j + 2], s[8 * j + 3], s[8 * j + 4], s[8 * j + 5], s[8 * j + 6], s[8 * j + 7]);
  };

  if constexpr (kPaired) {
    // ---- 64 features: the vector work of a tile costs as much issue time as its products, so the two are woven. Step i: the
    // gradient products of tile i - 1 and S(i + 1) between the exponentials of tile i, then dP(i + 1) between the rest of its
    // arithmetic. Tile i + 3 is requested; tile i + 2 has landed when the step ends.
    f32x16 s1, dp1;
    auto kslot = [&](int t) __attribute__((always_inline)) { return kbuf + (t & (kSlots - 1)) * L::kKTile; };
    auto vslot = [&](int t) __attribute__((always_inline)) { return vbuf + (t & (kSlots - 1)) * L::kVTile; };
    constexpr std::true_type yes;
    constexpr std::false_type no;
    // product m of the step: gradient products 0..3 (GRAD), then S, 4..7, and dP, 8..11, of the next tile (NEXT)
    auto step = [&](int i, auto grad_tag, auto next_tag, f32x16& x, f32x16& y, f32x16& nx, f32x16& ny) __attribute__((always_inline)) {
      constexpr bool GRAD = decltype(grad_tag)::value, NEXT = decltype(next_tag)::value;
      static_assert(2 * DB == 4 && KS == 4 && VS == 4, "products of a step");
      refresh_offsets();
      const char* const kp = kslot(i - 1);
      const char* const kn = kslot(i + 1);
      const char* const vn = vslot(i + 1);
      auto frag = [&](int m) __attribute__((always_inline)) -> bf16x8 {
        if (m < 4) return GRAD ? kt_frag(kp, m >> 1, m & 1) : bf16x8{};
        return NEXT ? (m < 8 ? k_frag(kn, m - 4) : v_frag(vn, m - 8)) : bf16x8{};
      };
      if constexpr (NEXT && MULTI) request(i + 3);  // (a tile's address takes branches; behind the last tile it is one of the last chunk)
      bf16x8 a[12];
#pragma unroll
      for (int m = 0; m < kAhead; ++m) a[m] = frag(m);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        if (NEXT) nx[v] = 0.f;
        if (NEXT) ny[v] = -delta_q;  // dS = P * (dP - delta) without a subtraction per element
      }
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        __builtin_amdgcn_sched_barrier(0);
        a[m + kAhead] = frag(m + kAhead);
        if (GRAD && m < 4) acc[m & 1] = mfma32(a[m], dsf[m >> 1], acc[m & 1]);
        if (NEXT && m >= 4) nx = mfma32(a[m], qf[m - 4], nx);
        if constexpr (NEXT && !MULTI) {
          if (m == 1) request_k(i + 3);
          if (m == 3) request_v(i + 3);
        }
#pragma unroll
        for (int v = 2 * m; v < 2 * m + 2; ++v) x[v] = __builtin_amdgcn_exp2f(x[v] * p.kappa - lse_q);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (mask.partial(range, i, q_wave0)) {  // wave-uniform
        const int limit = mask.limit(range, qrow), n0 = mask.key0(i);
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (n0 + acc_row(v, g) > limit) x[v] = 0.f;
      }
      mask.advance(p, range);
      u32x4 du[2];
#pragma unroll
      for (int m = 8; m < 12; ++m) {
        __builtin_amdgcn_sched_barrier(0);
        if (NEXT) ny = mfma32(a[m], dof[m - 8], ny);
#pragma unroll
        for (int w = 2 * (m - 8); w < 2 * (m - 8) + 2; ++w) {
          uint32_t dw = pack_bf16x2(x[2 * w] * y[2 * w], x[2 * w + 1] * y[2 * w + 1]);
          asm volatile("" : "+v"(dw));  // formed here, not where it is used
          du[w >> 2][w & 3] = dw;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 2; ++j) dsf[j] = __builtin_bit_cast(bf16x8, du[j]);
      if constexpr (NEXT) {  // (a wave's last tile waits for nothing)
        wait_staged<L::kLoads>();
        __syncthreads();
      }
    };
    if (n_wg > 2) wait_staged<2 * L::kLoads>();
    else wait_staged();
    __syncthreads();
    scores(kbuf, vbuf);
    if (n_wg > 2) wait_staged<L::kLoads>();
    else wait_staged();
    __syncthreads();  // tile 1 is there
    if (n_wave == 1) {
      step(0, no, no, s, dp, s1, dp1);
    } else {
      step(0, no, yes, s, dp, s1, dp1);
      int i = 1;
      for (; i + 2 < n_wave; i += 2) {
        step(i, yes, yes, s1, dp1, s, dp);
        step(i + 1, yes, yes, s, dp, s1, dp1);
      }
      if (i + 1 < n_wave) {
        step(i, yes, yes, s1, dp1, s, dp);
        step(i + 1, yes, no, s, dp, s1, dp1);
      } else {
        step(i, yes, no, s1, dp1, s, dp);
      }
    }
    accumulate(kslot(n_wave - 1));
    for (int i = n_wave - 1; i + 1 < n_wg; ++i) {  // waves above the workgroup's last diagonal block keep moving tiles for the others
      if constexpr (MULTI) {
        request(i + 3);
      } else {
        request_k(i + 3);
        request_v(i + 3);
      }
      wait_staged<L::kLoads>();
      __syncthreads();
    }
    wait_staged();
    __syncthreads();  // every wave is done with the rings, and nothing lands in them any more
  } else {
    if (n_wg > 2) wait_staged<2 * L::kLoads>();
    else wait_staged();
    __syncthreads();
    scores(kbuf, vbuf);
    make_ds(0);
    if (n_wg > 2) wait_staged<L::kLoads>();
    else wait_staged();
    __syncthreads();  // tile 1 is there

    int i = 1;
    for (; i < n_wave; ++i) {
      const bool more = i + 2 < n_wg;
      refresh_offsets();
      if (more) request(i + 2);
      matrix_block(kbuf + ((i - 1) & (kSlots - 1)) * L::kKTile, kbuf + (i & (kSlots - 1)) * L::kKTile, vbuf + (i & (kSlots - 1)) * L::kVTile);
      make_ds(i);
      // tile i + 1 has landed; the loads just requested may stay in flight (they are the wave's last memory operations)
      if (more) __builtin_amdgcn_s_waitcnt(0x0F70 | L::kLoads);
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    }
    accumulate(kbuf + ((n_wave - 1) & (kSlots - 1)) * L::kKTile);
    for (; i < n_wg; ++i) {  // waves above the workgroup's last diagonal block keep moving tiles for the others
      const bool more = i + 2 < n_wg;
      if (more) request(i + 2);
      if (more) __builtin_amdgcn_s_waitcnt(0x0F70 | L::kLoads);
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    }
    __syncthreads();  // every wave is done with the rings
  }

  OutT* rows = reinterpret_cast<OutT*>(p.dq) + b * p.dq_bs + (int64_t)h * DQK + q_wave0 * q_row_stride;
  __bf16* fin = nullptr;  // rows whose gradient is complete with this call go out as bf16
  if (sizeof(OutT) == 4 && p.dq_final != nullptr && q_wave0 >= p.final_r0 && q_wave0 < p.final_r1)
    fin = p.dq_final + b * p.dq_final_bs + (int64_t)h * DQK + q_wave0 * q_row_stride;
  char* const turn = smem + wave * kRowsViaLdsBytes<L::kTurnBlocks>;
#pragma unroll
  for (int o0 = 0; o0 < DB; o0 += L::kTurnBlocks) {
    f32x16 part[L::kTurnBlocks];
#pragma unroll
    for (int o = 0; o < L::kTurnBlocks; ++o) part[o] = acc[o0 + o];
    store_rows32_via_lds<OutT, L::kTurnBlocks>(turn, rows + 32 * o0, q_row_stride, p.Sq - q_wave0, part, p.scale, p.accumulate_dq != 0, lane,
                                               p.through_dq, fin == nullptr ? nullptr : fin + 32 * o0);
  }
}

}  // namespace dq_duo
}  // namespace pith
