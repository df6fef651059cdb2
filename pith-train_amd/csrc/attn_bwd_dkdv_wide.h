// Key/value-gradient kernel for head dims (128, 128) on gfx950 with 256 key rows per workgroup. Same function, numerics, roles
// (wave A of a pair: S, P, dV; wave B one tile behind: dP, dS, dK) and dS images as attn_bwd_dkdv_d128.h, and the same bits for
// the same head split: rows are added up in the same steps of 16.
//
// What bounds the 128-key kernel on long calls is power: the chip lowers its clock to 1.66-1.71 GHz. A fragment read from LDS feeds
// one product there, 1 KB per 32-cycle product and wave, all that LDS can deliver, and in a loop of nothing but reads and products
// (tests/probes/lds_fragment_rate_probe.hip) 1, 2 and 4 products per read run at 1.65, 1.77 and 1.80 PFLOP/s, at 1.64, 1.76 and 1.79
// GHz. Here a wave owns two 32-key blocks, so that every fragment
// of Q and dO feeds two products, and a tile requested serves twice as many keys. The accumulators (128 registers) and the
// stationary fragments (64) then leave room for tiles of 32 query rows, two fragments read ahead and five of eight steps'
// stationary fragments; the other three stay in LDS (22 reads per 32 products instead of 32; 24 with a third fragment ahead
// were 1 % slower, and one step more in registers spills without a mask: 8-12 % slower).
// Measured, dK/dV with the sums over head parts, dS handed over, 128 -> 256 keys, us: 8192 x 4096 x 32/4 heads 1084 -> 1034, 16384 x
// 8192 x 16/1 2110 -> 2040, 8192 x 16 1096 -> 1029, causal 4 x 4096 x 16 631 -> 606, 8 x 2048 x 16 376 -> 351. Which calls: wide().
// Counters of the kernel alone at 8192 x 4096 x 32/4: 6.72e7 -> 4.42e7 LDS instructions, 1.71 -> 1.79 GHz, pipe busy 58 -> 60 %, 1055 ->
// 976 us; no dS 1.66 -> 1.77 GHz, 68 -> 65 % of 4 % more cycles, 929 -> 907 us.
// Tried: the first fragments of a matrix block read before the barrier that starts it, 0.5 % slower; no s_setprio, 20 % slower.
#pragma once

#include <type_traits>

#include "attn_bwd_common.h"
#include "attn_bwd_dkdv_d128.h"

namespace pith {
namespace dkdv_wide {

constexpr int kThreads = 512;
constexpr int kBM = 32;             // query rows per tile
constexpr int kBN = kDkdvWideN;     // key rows per workgroup
constexpr int KB = 2;               // 32-key blocks per wave
constexpr int kD = 128;
constexpr int kStages = 3;          // tiles i-1, i (in use) and i+1 (landing)
constexpr int kAhead = 2;           // fragment reads run this many fragments (two products each) ahead
constexpr int kTile = kBM * kRowBytes128;        // 8 KB
constexpr int kStat = 2 * kBM * 4;               // lse[32], delta[32]
constexpr int kStage = 2 * kTile + kStat;        // Q tile, dO tile, stats
constexpr int kExchPair = kBM * 64 * 4;          // one 32 x 64 fp32 P tile
constexpr int kStatRows = KB * 8192;             // stationary rows of a wave, while they are staged (over everything but tile 0)
constexpr int kLdsKs = 3;           // contraction steps whose stationary fragments stay in LDS
constexpr int kOffStatLds = kStages * kStage + 4 * kExchPair;
constexpr int kStatLds = kLdsKs * KB * 1024;     // per wave
constexpr int kTurnBlocks = 2;       // 32-feature blocks the epilogue turns at a time
constexpr int kTurn = 8 * kRowsViaLdsBytes<kTurnBlocks>;
constexpr int larger(int a, int b) { return a > b ? a : b; }
constexpr int kSmem = larger(larger(kOffStatLds + 8 * kStatLds, kStage + 8 * kStatRows), kTurn);
static_assert(kSmem <= 160 * 1024, "one workgroup per compute unit");
// dS hand-over: vector-memory stores a B wave issues per interval (one 16-byte store per lane, 16-row step and key block).
// The wait that ends an interval lets exactly this many operations stay in flight, which is right only while they are the LAST
// vector-memory operations the wave issued.
constexpr int kDsStoresPerInterval = KB * kBM / 16;
static_assert(kDsStoresPerInterval < 16, "the vmcnt immediate below has a 4-bit low field");

using dkdv_d128::TileCursor;

template <bool CAUSAL, typename OutT, bool DESC>
__device__ __forceinline__ void body(const BwdParams& p, char* smem, int block) {
  constexpr int KS = kD / 16, DB = kD / 32;

  const int tid = threadIdx.x;
  if (block >= p.main_blocks) {  // workgroups appended to the grid: clear the rows behind the chunk's visible part
    zero_tail_block<OutT>(p, block - p.main_blocks, kD, kD, tid, kThreads);
    return;
  }
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, g = lane >> 5;
  const int pair = wave & 3;
  const bool role_b = wave >= 4;

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
  const int kv_pair0 = kv_wg0 + pair * (32 * KB);

  const int q_row_bytes = p.HqT * kD * 2;  // Q and dO rows
  const int64_t kv_row_stride = (int64_t)p.HkvT * kD;

  // Query tiles to visit: all of them, or from the diagonal down under the causal mask.
  const int m_end = (p.Sq + kBM - 1) / kBM;
  const int m_first = CAUSAL ? min(kv_wg0 / kBM, m_end) : 0;
  const int n_iter = (m_end - m_first) * heads_per_part;

  // ---- requests: issued by the four B waves only (their vector block, dS, is the shorter one)
  DirectTile128<kBM, kThreads / 2> mover;
  mover.init(q_row_bytes, pair, lane);
  const char* q_base = reinterpret_cast<const char*>(p.q + b * p.q_bs);
  const char* do_base = reinterpret_cast<const char*>(p.dout + b * p.dout_bs);
  using Cursor = TileCursor<DESC>;
  const int hq_end = hq0 + heads_per_part;
  Cursor req = Cursor::first(hq0, m_first, m_end);
  // The lane number, formed anew: what follows from it is then not kept across the loop, where registers are spilled for it and
  // a reload waits for the dS stores in flight.
  auto fresh_lane = [&]() __attribute__((always_inline)) {
    int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
    asm volatile("" : "+v"(l));
    return l;
  };
  auto request = [&](char* stage) __attribute__((always_inline)) {
    const int row0 = req.mt * kBM, ln = fresh_lane();
    const int64_t head_off = (int64_t)req.hq * kD * 2 + (int64_t)row0 * q_row_bytes;
    mover.issue_clamped(q_base + head_off, p.Sq - row0, stage, pair, ln);
    mover.issue_clamped(do_base + head_off, p.Sq - row0, stage + kTile, pair, ln);
    if (pair == 0) {  // the tile's 32 lse and 32 delta values
      int row = row0 + (ln & 31);
      row = row < p.Sq ? row : p.Sq - 1;
      load_lds4((ln < 32 ? p.lse : p.delta) + b * p.lse_bs + (int64_t)req.hq * p.lse_hs + row, stage + 2 * kTile);
    }
    req.advance(m_first, m_end, hq0, hq_end);
  };
  // stationary fragments: K rows for wave A, V rows for wave B
  constexpr int KSR = KS - kLdsKs;  // steps held in registers
  bf16x8 stat[KB][KSR];
  char* const stat_lds = smem + kOffStatLds + wave * kStatLds + lane * 16;
  char* const stat_area = smem + kStage + wave * kStatRows;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
    stage_rows32<true>(reinterpret_cast<const char*>((role_b ? p.v + b * p.v_bs : p.k + b * p.k_bs) + (int64_t)hk * kD), kv_pair0 + 32 * kb, p.Skv,
                       (int)(kv_row_stride * 2), stat_area + kb * 8192, lane);
  if (n_iter > 0 && role_b) request(smem);
  f32x16 acc[KB][DB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[kb][i][v] = 0.f;

  // per-lane read offsets inside a tile; the others follow by XOR (the swizzle is an XOR of the piece index): straight
  // fragment of contraction step ks = s_base ^ (ks << 5), transposing read of feature block o = t_base[hh] ^ (o << 6)
  int s_base = straight_offset128(c, g);
  int t_base[2] = {transposed_offset128(0, 0, 0, lane), transposed_offset128(0, 1, 0, lane)};

  // Called once per interval: the compiler must take the bases as new values each time, or it would compute all derived offsets
  // once, keep them in registers across the loop and spill others.
  auto refresh_offsets = [&]() __attribute__((always_inline)) { asm volatile("" : "+v"(s_base), "+v"(t_base[0]), "+v"(t_base[1])); };
  auto stat_frag = [&](int kb, int ks) __attribute__((always_inline)) {
    return ks < KSR ? stat[kb][ks < KSR ? ks : 0] : *reinterpret_cast<const bf16x8*>(stat_lds + ((ks - KSR) * KB + kb) * 1024);
  };

  // Within a stage wave A reads Q straight and dO transposed, wave B dO straight and Q transposed.
  const int straight_tile = role_b ? kTile : 0;
  const int transposed_tile = role_b ? 0 : kTile;
  char* const exch = smem + kStages * kStage + pair * kExchPair;

  f32x16 x[KB];        // [key block] A: S, then P of the current tile. B: delta - dP, kept into the next interval
  bf16x8 frag[KB][2];  // [key block][16-row step] A: P(i) as B operand of dV(i) in the next interval. B: -dS(i-1) for dK(i-1)

  auto straight_frag = [&](const char* stage, int ks) __attribute__((always_inline)) {
    return *reinterpret_cast<const bf16x8*>(stage + straight_tile + (s_base ^ (ks << 5)));
  };
  auto transposed_frag = [&](const char* stage, int j, int o) __attribute__((always_inline)) {
    const char* base = stage + transposed_tile + j * 16 * kRowBytes128;
    return lds_read_transposed_at(base + (t_base[0] ^ (o << 6)), base + (t_base[1] ^ (o << 6)));
  };
  // x starts from 0 in wave A and from the delta values of the tile's rows in wave B
  auto start_x = [&](const char* stage, auto role_tag) __attribute__((always_inline)) {
    if constexpr (decltype(role_tag)::value) {
      const float* delta_s = reinterpret_cast<const float*>(stage + 2 * kTile) + kBM;
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4) {
        const f32x4 d = *reinterpret_cast<const f32x4*>(delta_s + 8 * b4 + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) x[kb][4 * b4 + e] = d[e];
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int v = 0; v < 16; ++v) x[kb][v] = 0.f;
    }
  };
  // score-type product of the tile in `stage`: x = T1 * stat^T
  auto straight_product = [&](const char* stage, auto role_tag) __attribute__((always_inline)) {
    start_x(stage, role_tag);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bf16x8 a = straight_frag(stage, ks);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) x[kb] = mfma32(a, stat_frag(kb, ks), x[kb]);
    }
  };
  // gradient-type product with the tile in `stage`: acc^T += T2^T * frag
  auto transposed_product = [&](const char* stage) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < DB; ++o) {
        const bf16x8 a = transposed_frag(stage, j, o);
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) acc[kb][o] = mfma32(a, frag[kb][j], acc[kb][o]);
      }
  };
  // both (gradient product of `stage_prev`, then score product of `stage_cur`), with the fragment reads kAhead fragments ahead
  auto matrix_block = [&](const char* stage_prev, const char* stage_cur, auto role_tag) __attribute__((always_inline)) {
    constexpr int NT = 2 * DB, NS = KS;
    static_assert(kAhead <= NT, "look-ahead assumes it starts inside the gradient product");
    __builtin_amdgcn_s_setprio(2);  // the wave that owns the matrix pipe issues first
    bf16x8 at[2][DB], as[KS], sl[KS][KB];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < DB; ++o) at[j][o] = transposed_frag(stage_prev, j, o);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      as[ks] = straight_frag(stage_cur, ks);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) sl[ks][kb] = stat_frag(kb, ks);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < DB; ++o)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) acc[kb][o] = mfma32(at[j][o], frag[kb][j], acc[kb][o]);
    start_x(stage_cur, role_tag);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) x[kb] = mfma32(as[ks], sl[ks][kb], x[kb]);
    // a transposed fragment takes two LDS reads, a straight one a single read
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAhead, 0);
#pragma unroll
    for (int m = 0; m < NT - kAhead; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, KB, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    // wave B: the reads of delta, the start of x, follow the last fragment of the gradient product
    if constexpr (decltype(role_tag)::value) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int m = 0; m < KSR; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, KB, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
#pragma unroll
    for (int m = KSR; m < NS; ++m) {  // with the stationary fragments that are not in registers
      __builtin_amdgcn_sched_group_barrier(0x008, KB, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1 + KB, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, KB * kAhead, 0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
  };
  // Where dS is handed on, the nonexistent keys of a 32-key block that also holds real ones must read 0: dQ's last step reads them.
  // Nobody reads what lies behind (such keys have accumulator columns of their own, which are not stored), and a workgroup that masks
  // them in every tile is what a grid of one round ends on. Backward against 128 keys per workgroup, before -> now: 1664 x 32 heads, full,
  // +7 -> 0 %, 1920 x 32 +5 -> 0 %, 8064 x 8 +5 -> -1 %, 2432 x 24 +5 -> 0 %, 2 x 3000 x 896 x 32 +1 -> -4 %.
  const bool mask_keys = p.ds != nullptr && (p.Skv & 31) != 0 && kv_pair0 < p.Skv && kv_pair0 + 32 * KB > p.Skv;
  // A: x = S of query tile mt -> P, left in the exchange buffer (fp32) and in frag (bf16).
  // Rows of the tile are queries q0 + acc_row(v, g); this lane's columns are keys kv_pair0 + 32*kb + c.
  auto make_p = [&](const char* stage, int mt) __attribute__((always_inline)) {
    const float* lse_s = reinterpret_cast<const float*>(stage + 2 * kTile);
    const int q0 = mt * kBM;
    // tile on the diagonal, ragged last tile, or mask_keys (wave-uniform)
    const bool masked = (CAUSAL && q0 < kv_pair0 + 32 * KB - 1) || q0 + kBM > p.Sq || mask_keys;
    f32x4 l4[4];
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) l4[b4] = *reinterpret_cast<const f32x4*>(lse_s + 8 * b4 + 4 * g);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
      for (int v = 0; v < 16; ++v) x[kb][v] = __builtin_amdgcn_exp2f(x[kb][v] * p.kappa - l4[v >> 2][v & 3]);
      if (masked) {
        const int key = kv_pair0 + 32 * kb + c;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int qrow = q0 + acc_row(v, g);
          if ((CAUSAL && key > qrow) || qrow >= p.Sq || key >= p.Skv) x[kb][v] = 0.f;
        }
      }
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4) {
        const f32x4 pr = {x[kb][4 * b4], x[kb][4 * b4 + 1], x[kb][4 * b4 + 2], x[kb][4 * b4 + 3]};
        *reinterpret_cast<f32x4*>(exch + ((kb * 4 + b4) * 64 + lane) * 16) = pr;
      }
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
        frag[kb][jj] = to_bf16x8(x[kb][8 * jj], x[kb][8 * jj + 1], x[kb][8 * jj + 2], x[kb][8 * jj + 3],
                                 x[kb][8 * jj + 4], x[kb][8 * jj + 5], x[kb][8 * jj + 6], x[kb][8 * jj + 7]);
    }
  };
  // B: x = delta - dP of the tile in `stage`, P from the exchange buffer -> -dS / scale in frag (bf16), also
  // stored as images of query tile `tile` where dS is handed on. Returns whether it stored. (One instance for both: with the
  // stores compiled out the register allocator spilled 40 registers.)
  const int key_block = kv_pair0 >> 7;  // of 128 keys: the unit in which images are kept
  char* const ds_pair = p.ds + (int64_t)(kv_pair0 >> 5) * 4096;
  auto make_ds = [&](const Cursor& tile) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      f32x4 pr[4];
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4) pr[b4] = *reinterpret_cast<const f32x4*>(exch + ((kb * 4 + b4) * 64 + lane) * 16);
#pragma unroll
      for (int v = 0; v < 16; ++v) x[kb][v] = pr[v >> 2][v & 3] * x[kb][v];  // x = delta - dP
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
        frag[kb][jj] = to_bf16x8(x[kb][8 * jj], x[kb][8 * jj + 1], x[kb][8 * jj + 2], x[kb][8 * jj + 3],
                                 x[kb][8 * jj + 4], x[kb][8 * jj + 5], x[kb][8 * jj + 6], x[kb][8 * jj + 7]);
    }
    const int t64 = tile.mt >> 1;
    if (p.ds == nullptr || key_block >= (CAUSAL ? (t64 >> 1) + 1 : p.ds_kb)) return false;  // no room is kept for what nobody reads
    char* img = ds_pair + (int64_t)(b * p.Hq + tile.hq) * p.ds_hs + ds_tile_start<CAUSAL>(t64, p.ds_kb) * kDsBlockBytes + (tile.mt & 1) * 2048;
    const int ln = fresh_lane(), lg = ln >> 5;
    const int off = (lg << 9) + (((ln & 31) ^ (lg << 3)) << 4);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        store16_through(img + kb * 4096 + j * 1024, off ^ (j << 6), frag[kb][j]);
    return true;
  };

  wait_staged();  // everything issued so far: tile 0, stationary rows
  // wave B works with -V: its score-type product then starts from delta and yields delta - dP, i.e. -(dP - delta) without a
  // subtraction per element; the sign is undone with the factor -scale on the accumulated dK (and by the reader of the dS images)
  const unsigned sign = role_b ? 0x80008000u : 0u;
  auto staged = [&](int kb, int ks) __attribute__((always_inline)) {
    return __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, staged_fragment<true>(stat_area + kb * 8192, ks, c, g)) ^ sign);
  };
  bf16x8 rest[KB][kLdsKs];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
    for (int ks = 0; ks < KSR; ++ks) stat[kb][ks] = staged(kb, ks);
#pragma unroll
    for (int ks = KSR; ks < KS; ++ks) rest[kb][ks - KSR] = staged(kb, ks);
  }
  __syncthreads();  // every wave has read its rows: their place becomes ring, exchange and stationary fragments
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int i = 0; i < kLdsKs; ++i) *reinterpret_cast<bf16x8*>(stat_lds + (i * KB + kb) * 1024) = rest[kb][i];

  // Interval i = 0 .. n_iter touches tiles i-1 and i; tile -1 and tile n_iter do not exist, so the
  // first and the last interval are peeled and the loop body in between is straight-line code.
  // Under the causal mask a tile that lies entirely above a pair's diagonal is processed like any
  // other: its P is all zeros (at most one tile per query head and pair).
  // Ring stages rotate: prev <- cur <- next <- (the stage prev used to be).
  auto run = [&](auto role_tag) __attribute__((always_inline)) {
    constexpr bool ROLE_B = decltype(role_tag)::value;
    Cursor cur = Cursor::first(hq0, m_first, m_end), done = cur;  // tiles i and i-1 of interval i
    int off_prev = 2 * kStage, off_cur = 0, off_next = kStage;
    auto end_interval = [&](bool stored) __attribute__((always_inline)) {
      // the tile requested in this interval has landed. Vector memory operations complete in issue
      // order, and where wave B issued its four dS stores after the request (every interval but the
      // first) they may stay in flight.
      if (ROLE_B && stored) __builtin_amdgcn_s_waitcnt(0x0F70 | kDsStoresPerInterval);
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
      done = cur;
      cur.advance(m_first, m_end, hq0, hq_end);
      const int t = off_prev;
      off_prev = off_cur;
      off_cur = off_next;
      off_next = t;
    };
    // interval 0
    if (!ROLE_B) {
      straight_product(smem + off_cur, role_tag);
      __syncthreads();
      make_p(smem + off_cur, cur.mt);
    } else {
      if (n_iter > 1) request(smem + off_next);
      __syncthreads();
      straight_product(smem + off_cur, role_tag);
    }
    end_interval(false);
    for (int i = 1; i < n_iter; ++i) {
      refresh_offsets();
      const char* stage_cur = smem + off_cur;
      const char* stage_prev = smem + off_prev;
      const bool will_request = i + 1 < n_iter;
      bool stored = false;
      if (!ROLE_B) {
        matrix_block(stage_prev, stage_cur, role_tag);
        __syncthreads();  // B has read P(i-1); the matrix pipe passes to B
        make_p(stage_cur, cur.mt);
      } else {
        if (will_request) request(smem + off_next);
        stored = make_ds(done);
        __syncthreads();
        matrix_block(stage_prev, stage_cur, role_tag);
      }
      end_interval(stored);
    }
    // interval n_iter
    if (!ROLE_B) {
      transposed_product(smem + off_prev);
      __syncthreads();
    } else {
      make_ds(done);
      __syncthreads();
      transposed_product(smem + off_prev);
    }
  };
  // Both roles pass the same barriers; separate code keeps each loop body straight-line.
  if (n_iter > 0) {
    if (!role_b) run(std::false_type{});
    else run(std::true_type{});
  }

  // ---- epilogue: wave A stores dV, wave B stores dK (it accumulated -dK / scale); a lane holds one key row, turned through
  // LDS so that the stores cover whole rows, 64 features at a time
  __syncthreads();  // every wave is done with the ring
  char* const turn = smem + wave * kRowsViaLdsBytes<kTurnBlocks>;
  const float factor = role_b ? -p.scale : 1.f;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int o0 = 0; o0 < DB; o0 += kTurnBlocks) {
      f32x16 part_acc[kTurnBlocks];
#pragma unroll
      for (int o = 0; o < kTurnBlocks; ++o) part_acc[o] = acc[kb][o0 + o];
      const int key0 = kv_pair0 + 32 * kb, rows_valid = p.Skv - key0;
      if (p.split > 1) {
        // the partials are packed: exactly the Hkv heads of this call per row
        const int64_t row_stride = (int64_t)p.Hkv * kD;
        float* ws = (role_b ? p.ws_dk : p.ws_dv) + (((int64_t)part * p.B + b) * p.Skv + key0) * row_stride + (int64_t)hk * kD + 32 * o0;
        store_rows32_via_lds<float, kTurnBlocks>(turn, ws, row_stride, rows_valid, part_acc, factor, false, lane, p.through_parts);
      } else {
        OutT* out = reinterpret_cast<OutT*>(role_b ? p.dk : p.dv) + b * (role_b ? p.dk_bs : p.dv_bs) + key0 * kv_row_stride + (int64_t)hk * kD + 32 * o0;
        store_rows32_via_lds<OutT, kTurnBlocks>(turn, out, kv_row_stride, rows_valid, part_acc, factor, p.accumulate != 0, lane, p.through_dkv);
      }
    }
}

}  // namespace dkdv_wide
}  // namespace pith
