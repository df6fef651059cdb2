// Chunk attention forward for head dims (64, 64), (128, 128) and (192, 128) on gfx950 with SMALL workgroups: 4 wavefronts,
// 128 query rows (PARTS = 1), two of them per compute unit (three at 64 features). Same function, numerics and tile layouts as
// attn_fwd_direct.hip (pithtrain/operators/mla/triton.py:32-93, :274-323): a wave owns 32 query rows and all 64 keys of a
// tile, per interval one matrix block [O^T += V(i)^T P(i)^T ; S(i+1)^T = K(i+1) Q^T] and one softmax.
//
// What bounds launches of a few rounds of workgroups is not the loop but everything around it: with one 8-wave workgroup
// per compute unit nothing runs while it fetches its first tiles, waits for its slowest wave at the diagonal and writes its
// rows (9-15 us per round). Two independent workgroups hide each other's: 3 x 1999 rows x 32 heads causal 131 -> 105 us
// (128-row workgroups with split keys before), 8 x 512 x 32 47 -> 32 us, 2 x 2048 x 16 heads of 64 features 42 -> 31 us.
// The waves that share a SIMD belong to different workgroups, so no role split keeps their matrix and vector phases apart;
// measured, the workgroups drift apart by themselves: fixed or alternating wave priorities by wave slot were 2-10 %
// slower, and so was asking for the tiles behind the matrix block (0-4 %).
// 64 features: a K or V tile packs two rows per 256-byte LDS row (see DirectPaired64), and the softmax of 32 x 64 scores
// costs as much vector time as its products cost matrix time, so three workgroups per compute unit share the pipes.
//
// PARTS = 3 (SMALL): 64 rows; the two waves that share 32 rows take half a tile's keys each and merge through LDS. An interval has
// half the products and half the vector work of a wave, and the grid twice the workgroups, where those of 128 rows leave a SIMD little more
// than one wave that does one thing at a time (2 x 2048 x 16/4 heads of 64: 0.97 waves per SIMD, matrix pipe 18 % busy): 33.3 -> 27.3
// us, 2 x 1024 x 16/4 16.5 -> 13.1, 256 x 8/2 of 128 8.5 -> 7.3, 2 x 512 x 32/4 13.9 -> 11.6.
// PARTS = 2, 4: two such teams of 4 waves in one workgroup, each with its own rings, taking every second tile; the results are
// merged through LDS. For grids that leave units idle or a heavy workgroup alone on its unit, where the length of a stream
// counts. PARTS = 2: 128 rows as above. PARTS = 4: 64 rows, the two waves of a team that share rows take half a tile's keys
// each: twice the requests per product, on units that have nothing else to do. Measured against the split-key workgroups of
// attn_fwd_direct.hip (64 features: against one team), inputs from memory: 1 x 1021 x 16 heads of 192 25.9 -> 24.0 us, its
// ring share of 3 chunks 60.0 -> 47.7, 1 x 4096 x 4 of 192 70 -> 62, 1 x 2048 x 8 of 128 30.5 -> 26.4, 1 x 8192 x 4 of 64
// 98 -> 70 (4 parts); 1 x 4096 x 16 of 64 57 -> 53, 1 x 4096 x 8 of 64 52 -> 43 (2 parts, 64 features only). More at
// pick_split.
//
// LDS: rings of two K and two V tiles; interval i reads V(i) and K(i+1) while V(i+1) and K(i+2) land in the slots that
// interval i-1 released.
#include "attn_fwd_common.h"

namespace pith {
namespace {

constexpr int kTeamWaves = 4;                 // waves that share a stream of tiles
constexpr int kTeamThreads = kTeamWaves * 64;
constexpr int kBN = kFwdBlockN;   // keys per tile
constexpr int kAhead = 4;         // fragment reads run this many products ahead in the matrix block
// Intervals of a workgroup from which the two teams of 64-row workgroups (128 and 192 features) take turns (run_halves). The tiles of such a workgroup, 40 KB
// per team and interval at 192 features, are what bounds it: without its loads 1021 x 3063 keys x 16 heads takes 33 us, loads alone 45, and with everything
// landed at the end of each interval 54. Rows of few tiles lose the half interval by which the second team ends later. One
// barrier an interval / turns, us, inputs from memory, full: 512 x 512 x 16 of 192 (4 intervals) 12.4 / 12.9, 768 (6) 15.3 / 15.2, 1024 18.1 / 17.2, 2048 32.6 /
// 28.6, 3063 53.2 / 45.6, 1021 x 3063 54.1 / 47.5; of 128 512 11.0 / 11.7, 1024 15.6 / 15.3, 2048 24.5 / 22.2, 3063 45.3 / 37.9; causal 1021 x 16 of
// 192 17.9 / 17.1, 2048 x 8 28.4 / 25.1, 4096 x 4 47.8 / 41.1, 8192 x 4 122 / 110, of 128 1021 x 16 15.3 / 15.1, 4096 x 4 41.0 / 36.2, 8192 x 4 104 / 91;
// shares, 4 ranks: 1021 x 16 of 192 in two parts 44.3 / 41.4, 2048 x 16 115.6 / 107.0, 1024 x 16 55.0 / 48.6. 64 features lose at any length (4096 x 16 48.8 / 49.7).
constexpr int kHalvesFrom = 8;

template <int DQK, int PARTS>
struct DuoLayout {
  static constexpr int kTeams = PARTS == 1 || PARTS == 3 ? 1 : 2;
  static constexpr int kParts = PARTS == 3 ? 2 : PARTS;  // waves that share 32 query rows
  static constexpr int kThreads = kTeams * kTeamThreads;
  static constexpr int kRowBlocks = PARTS >= 3 ? 2 : 4;  // of 32 query rows
  static constexpr int kBM = 32 * kRowBlocks;            // query rows per workgroup
  static constexpr int kDv = DQK == 64 ? 64 : 128;
  static constexpr int kKTile = DQK == 64 ? kExtraTileBytes : DQK == 128 ? kBN * kRowBytes128 : kBN * kRowBytes128 + kExtraTileBytes;
  static constexpr int kVTile = kDv == 64 ? kExtraTileBytes : kBN * kRowBytes128;
  static constexpr int kRings = 2 * (kKTile + kVTile);   // of one team
  static constexpr int kTurn = kRowsViaLdsBytes<kDv / 32>;
  static constexpr int kAfter = kRowBlocks * (PARTS == 1 ? 1 : kParts - 1) * kTurn;  // the epilogue's use of the rings
  static constexpr int kSmem = kTeams * kRings > kAfter ? kTeams * kRings : kAfter;
};

template <int DQK, int PARTS, bool CAUSAL, bool MULTI>
__global__ __launch_bounds__((DuoLayout<DQK, PARTS>::kThreads), 2) void attn_fwd_duo_kernel(FwdArgs<MULTI> p) {
  using L = DuoLayout<DQK, PARTS>;
  constexpr int kDv = L::kDv, KS = DQK / 16, DVB = kDv / 32, kBM = L::kBM, kTeams = L::kTeams;
  constexpr int KVB = PARTS >= 3 ? 1 : 2;  // 32-key blocks of a tile this wave owns
  constexpr bool kPaired = DQK == 64;  // tiles hold two rows per 256-byte LDS row
  constexpr int kTile = kBN * kRowBytes128;
  constexpr bool kHalves = PARTS == 4 && DQK != 64;  // see kHalvesFrom
  __shared__ __attribute__((aligned(1024))) char smem[L::kSmem];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wg_wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wg_wave & (kTeamWaves - 1);              // within its team
  const int team = kTeams == 1 ? 0 : wg_wave / kTeamWaves;  // takes the tiles t with t % kTeams == team
  const int row_block = wave & (L::kRowBlocks - 1);
  const int kvb0 = PARTS >= 3 ? wave >> 1 : 0;              // first 32-key block of a tile this wave owns
  const int part = PARTS == 4 ? 2 * team + kvb0 : PARTS == 3 ? kvb0 : team;  // of its 32 rows' keys
  char* const kbuf = smem + team * L::kRings;
  char* const vbuf = kbuf + 2 * L::kKTile;
  const int c = lane & 31, g = lane >> 5;

  int m_tile, h, b;
  decode_block(blockIdx.x, p.Hq, p.B, p.m_tiles, p.group, m_tile, h, b, p.chunked);
  const int hk = h / p.group;
  const int m0 = m_tile * kBM;
  const int q_wave0 = m0 + row_block * 32;
  const int qrow = q_wave0 + c;

  const int64_t q_row_stride = (int64_t)p.Hq * DQK;
  const int64_t o_row_stride = (int64_t)p.Hq * kDv;
  // keys in two parts: K rows hold 128 features per head, the last 64 come from k_pe (no head offset)
  const bool two_part = DQK == 192 && chunk_of(p, 0).k_pe != nullptr;
  const int k_head_elems = two_part ? 128 : DQK;
  const int k_row_bytes = p.Hkv * k_head_elems * 2, v_row_bytes = p.Hkv * kDv * 2;
  const __bf16* qh = p.q + b * p.q_bs + (int64_t)h * DQK;
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

  // Number of key tiles this workgroup / this wavefront has to visit.
  const ChunkRange<MULTI, CAUSAL, kBN> range(p, m0 + kBM);
  int n_tiles_wg = range.tiles_full, n_tiles_wave = range.tiles_full;
  if (CAUSAL) {
    const int tiles = (chunk_of(p, range.last).rows + kBN - 1) / kBN;
    n_tiles_wg += min(tiles, (m0 + kBM - 1) / kBN + 1);
    n_tiles_wave += min(tiles, (q_wave0 + 31) / kBN + 1);
  }
  if constexpr (PARTS != 2) n_tiles_wave = tiles_of_wave(n_tiles_wave, q_wave0, p.Sq);
  const int intervals = (n_tiles_wg + kTeams - 1) / kTeams;  // of the workgroup
  if constexpr (kTeams > 1) {  // from here on a team's own tiles (the second team of a single tile has none)
    n_tiles_wg = (n_tiles_wg + 1 - team) >> 1;
    n_tiles_wave = (n_tiles_wave + 1 - team) >> 1;
  }
  auto tile = [&](int t) __attribute__((always_inline)) { return kTeams * t + team; };  // in the workgroup's stream
  TileSource<MULTI, CAUSAL, kBN> k_src(p, range, k_row_bytes, k_rows), kx_src(p, range, kx_row_bytes, kx_rows),
      v_src(p, range, v_row_bytes, v_rows);
  TileMask<MULTI, CAUSAL, kBN> mask(p, range);
  if (team == 1) {
    k_src.advance(p, range, k_rows);
    if constexpr (DQK == 192) kx_src.advance(p, range, kx_rows);
    v_src.advance(p, range, v_rows);
    mask.advance(p, range);
  }

  DirectTile128<kBN, kTeamThreads> vmover, kmover;
  DirectPaired64<kBN, kTeamThreads> vpmover, kpmover;  // 64-feature tiles, and features 128..191 of a 192-feature key
  if constexpr (kPaired) {
    vpmover.init(v_row_bytes, 0, wave, lane);
    kpmover.init(k_row_bytes, 0, wave, lane);
  } else {
    vmover.init(v_row_bytes, wave, lane);
    kmover.init(k_row_bytes, wave, lane);
    if constexpr (DQK == 192) kpmover.init(kx_row_bytes, two_part ? 0 : 256, wave, lane);
  }
  // (tiles are requested strictly in order, so the sources just move on)
  auto issue_k = [&](int t) __attribute__((always_inline)) {
    char* slot = kbuf + (t & 1) * L::kKTile;
    const int at = tile(t);
    if constexpr (kPaired) {
      kpmover.issue(k_src.src(at), k_src.left(at), slot, wave, lane);
    } else {
      kmover.issue(k_src.src(at), k_src.left(at), slot, wave, lane);
      if constexpr (DQK == 192) {
        kpmover.issue(kx_src.src(at), kx_src.left(at), slot + kTile, wave, lane);
        for (int n = 0; n < kTeams; ++n) kx_src.advance(p, range, kx_rows);
      }
    }
    for (int n = 0; n < kTeams; ++n) k_src.advance(p, range, k_rows);
  };
  auto issue_v = [&](int t) __attribute__((always_inline)) {
    char* slot = vbuf + (t & 1) * L::kVTile;
    const int at = tile(t);
    if constexpr (kPaired) vpmover.issue(v_src.src(at), v_src.left(at), slot, wave, lane);
    else vmover.issue(v_src.src(at), v_src.left(at), slot, wave, lane);
    for (int n = 0; n < kTeams; ++n) v_src.advance(p, range, v_rows);
  };
  // Query rows first: nothing can start without them. PARTS = 1: every wave stages its own in slots of tiles that are requested
  // behind them (K 1 and V 1, two waves each; at 192 features the fourth wave takes V 0). Several parts: the waves of a row
  // block share the loads and an area in the V 1 slots (small workgroups of 192 features: in V 1 and K 1).
  constexpr int kQArea = kPaired ? 4096 : 8192 + (DQK == 192 ? 4096 : 0);
  constexpr bool kDelayV0 = PARTS == 1 && DQK == 192, kDelayK1 = PARTS == 3 && DQK == 192;
  static_assert(PARTS == 1   ? 2 * kQArea <= L::kKTile && (kDelayV0 ? kQArea : 2 * kQArea) <= L::kVTile
                : PARTS == 3 ? (kDelayK1 ? kQArea <= L::kKTile && kQArea <= L::kVTile : 2 * kQArea <= L::kVTile)
                             : kQArea * L::kRowBlocks / 2 <= L::kVTile, "query areas");
  char* const k1 = kbuf + L::kKTile;
  char* const v0 = vbuf;
  char* const v1 = vbuf + L::kVTile;
  char* q_area;
  if constexpr (PARTS == 1) q_area = wave < 2 ? k1 + wave * kQArea : kDelayV0 ? (wave == 2 ? v1 : v0) : v1 + (wave - 2) * kQArea;
  else if constexpr (PARTS == 3) q_area = row_block == 0 ? v1 : kDelayK1 ? k1 : v1 + kQArea;
  else if constexpr (PARTS == 2) q_area = smem + (row_block >> 1) * L::kRings + 2 * L::kKTile + L::kVTile + (row_block & 1) * kQArea;
  else q_area = smem + row_block * L::kRings + 2 * L::kKTile + L::kVTile;
  {
    constexpr int kShare = L::kParts;
    const char* const qsrc = reinterpret_cast<const char*>(qh);
    const int q_row_bytes = (int)(q_row_stride * 2);
    if constexpr (!kPaired) stage_rows32<true, 8 / kShare>(qsrc, q_wave0, p.Sq, q_row_bytes, q_area, lane, part * (8 / kShare));
    if constexpr (DQK != 128)
      stage_rows32<false, 4 / kShare>(qsrc + (kPaired ? 0 : 256), q_wave0, p.Sq, q_row_bytes, q_area + (kPaired ? 0 : 8192), lane, part * (4 / kShare));
  }
  if (kTeams == 1 || n_tiles_wg > 0) {
    issue_k(0);
    if constexpr (!kDelayV0) issue_v(0);
  }
  if (PARTS > 1 && !kDelayK1 && n_tiles_wg > 1) issue_k(1);
  constexpr int kLoadsK = kPaired ? 2 : DQK == 192 ? 6 : 4, kLoadsV = kPaired ? 2 : 4;  // load instructions of a wave per tile
  bf16x8 qf[KS];  // Q^T fragments (B operand): column = query row, slots = 8 consecutive features
  auto read_q = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = kPaired ? staged_fragment<false>(q_area, ks, c, g) : ks < 8 ? staged_fragment<true>(q_area, ks, c, g)
                                                                           : staged_fragment<false>(q_area + 8192, ks - 8, c, g);
  };

  // per-lane read offsets (see attn_fwd_direct.hip): one base per tile part, the rest by XOR
  // (KVB = 1: the wave's key block sits in the bases)
  const int k_base = straight_offset128(c, g) + kvb0 * 32 * kRowBytes128, x_base = straight_offset128(c, g) ^ (kvb0 << 7);
  int v_base[2] = {transposed_offset128(0, 0, 0, lane), transposed_offset128(0, 1, 0, lane)};
  for (int& v : v_base) v = kPaired ? v ^ (kvb0 << 7) : v + kvb0 * 32 * kRowBytes128;
  auto k_frag = [&](const char* ktile, int ks, int kvb) __attribute__((always_inline)) {
    int off;
    if (kPaired) off = x_base ^ (ks << 5) ^ (kvb << 7);
    else if (ks < 8) off = (k_base ^ (ks << 5)) + kvb * 32 * kRowBytes128;
    else off = kTile + (x_base ^ ((ks - 8) << 5) ^ (kvb << 7));
    return *reinterpret_cast<const bf16x8*>(ktile + off);
  };
  // 16 keys j of the wave's, feature block i
  auto v_frag = [&](const char* vtile, int j, int i) __attribute__((always_inline)) {
    const int add = kPaired ? (j & 1) * 16 * kRowBytes128 : j * 16 * kRowBytes128;
    const int flip = kPaired ? (i << 6) | ((j >> 1) << 7) : i << 6;
    return lds_read_transposed_at(vtile + (v_base[0] ^ flip) + add, vtile + (v_base[1] ^ flip) + add);
  };

  f32x16 oacc[DVB];
#pragma unroll
  for (int i = 0; i < DVB; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[i][v] = 0.f;
  float m_run = -INFINITY;
  // A row that sees nothing of the first chunks has no maximum until its own, and would have the whole workgroup take that of every tile anew: in a zigzag share's
  // 64-row workgroup across the first row that sees the other chunks, whose teams it made wait for each other. Any finite start below all scores spares that (the
  // first key that a row sees exceeds the limit and sets its maximum; nothing has been added up by then). Rank 0 of four, 1514 x 16/4 heads of 128 85.5 us before the teams took
  // turns, 89.4 since, 72.4 without these maxima, of eight 960 x 32/4 116 / 123 / 96, 2260 x 8/2 255 / 265 / 205, 1008 x 16 of 192 67.8 / 68.0 / 58.2.
  if constexpr (MULTI && PARTS == 4)
    if (qrow < chunk_of(p, range.first()).q_row0) m_run = -1e38f / fmaxf(p.kappa, 1.f);  // (times kappa finite, too)
  float l_run = 0.f;  // this lane's share of the row sum (the partner lane holds the rest)
  f32x16 s[KVB];       // S^T of one tile: 32 x 32 tiles [keys] x [queries]
  bf16x8 pf[2 * KVB];  // P^T as B operand, one fragment per 16 keys

  // ---- S^T = K Q^T
  auto scores = [&](const char* ktile) __attribute__((always_inline)) {
#pragma unroll
    for (int kvb = 0; kvb < KVB; ++kvb)
#pragma unroll
      for (int v = 0; v < 16; ++v) s[kvb][v] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kvb = 0; kvb < KVB; ++kvb) s[kvb] = mfma32(k_frag(ktile, ks, kvb), qf[ks], s[kvb]);
  };

  // ---- mask, online softmax of the next tile in order (one query column per lane pair), P^T fragments
  auto softmax = [&](int t) __attribute__((always_inline)) {
    const int at = tile(t);
    if (mask.partial(range, at, q_wave0)) {
      const int limit = mask.limit(range, qrow);
#pragma unroll
      for (int kvb = 0; kvb < KVB; ++kvb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = mask.key0(at) + (kvb0 + kvb) * 32 + acc_row(v, g);
          if (key > limit) s[kvb][v] = -INFINITY;
        }
    }
    for (int n = 0; n < kTeams; ++n) mask.advance(p, range);
    f32x16 e[KVB];
    float rs = 0.f;
    // lazily refreshed running maximum, tested on the row sum (attn_fwd_direct.hip)
    const bool fresh = m_run == -INFINITY;
    float mk = fresh ? 0.f : m_run * p.kappa;
#pragma unroll
    for (int kvb = 0; kvb < KVB; ++kvb)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        e[kvb][v] = __builtin_amdgcn_exp2f(s[kvb][v] * p.kappa - mk);
        rs += e[kvb][v];
      }
    if (__builtin_amdgcn_ballot_w64(fresh || !(rs <= kRescaleLimit)) != 0) {
      float x = s[0][0];
#pragma unroll
      for (int kvb = 0; kvb < KVB; ++kvb)
#pragma unroll
        for (int v = 0; v < 16; ++v) x = fmaxf(x, s[kvb][v]);
      const float m_new = fmaxf(m_run, pair_max(x));
      const float alpha = (m_new == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f((m_run - m_new) * p.kappa);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < DVB; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) oacc[i][v] *= alpha;
      mk = (m_run == -INFINITY) ? 0.f : m_run * p.kappa;
      rs = 0.f;
#pragma unroll
      for (int kvb = 0; kvb < KVB; ++kvb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          e[kvb][v] = __builtin_amdgcn_exp2f(s[kvb][v] * p.kappa - mk);
          rs += e[kvb][v];
        }
    }
    l_run += rs;
#pragma unroll
    for (int kvb = 0; kvb < KVB; ++kvb)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const f32x16& x16 = e[kvb];
        pf[2 * kvb + jj] = to_bf16x8(x16[8 * jj], x16[8 * jj + 1], x16[8 * jj + 2], x16[8 * jj + 3], x16[8 * jj + 4],
                                     x16[8 * jj + 5], x16[8 * jj + 6], x16[8 * jj + 7]);
      }
  };

  // ---- O^T += V^T P^T
  auto accumulate = [&](const char* vtile) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2 * KVB; ++j)
#pragma unroll
      for (int i = 0; i < DVB; ++i) oacc[i] = mfma32(v_frag(vtile, j, i), pf[j], oacc[i]);
  };

  // both products of an interval, with the fragment reads pinned kAhead products ahead of their use
  auto matrix_block = [&](const char* vtile, const char* ktile) __attribute__((always_inline)) {
    constexpr int NPV = 2 * KVB * DVB, NQK = KVB * KS;
    __builtin_amdgcn_s_setprio(2);
    bf16x8 av[2 * KVB][DVB], ak[KS][KVB];
#pragma unroll
    for (int j = 0; j < 2 * KVB; ++j)
#pragma unroll
      for (int i = 0; i < DVB; ++i) av[j][i] = v_frag(vtile, j, i);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kvb = 0; kvb < KVB; ++kvb) ak[ks][kvb] = k_frag(ktile, ks, kvb);
#pragma unroll
    for (int j = 0; j < 2 * KVB; ++j)
#pragma unroll
      for (int i = 0; i < DVB; ++i) oacc[i] = mfma32(av[j][i], pf[j], oacc[i]);
#pragma unroll
    for (int kvb = 0; kvb < KVB; ++kvb)
#pragma unroll
      for (int v = 0; v < 16; ++v) s[kvb][v] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kvb = 0; kvb < KVB; ++kvb) s[kvb] = mfma32(ak[ks][kvb], qf[ks], s[kvb]);
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAhead, 0);
#pragma unroll
    for (int m = 0; m < NPV - kAhead; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
#pragma unroll
    for (int m = 0; m < NQK; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
  };

  if constexpr (PARTS == 1) {
    wait_staged<kLoadsK + (kDelayV0 ? 0 : kLoadsV)>();
    read_q();
    wait_staged<kDelayV0 ? 0 : kLoadsV>();
    __syncthreads();  // K tile 0 is there, and every wave has read its query rows: their slots may be filled
    if constexpr (kDelayV0) issue_v(0);
    if (n_tiles_wg > 1) issue_k(1);
  } else {
    if (kDelayK1) wait_staged<kLoadsV>();
    else if (n_tiles_wg > 1) wait_staged<kLoadsV + kLoadsK>();
    else wait_staged();
    __syncthreads();
    read_q();
    if constexpr (kDelayK1) {
      __syncthreads();
      if (n_tiles_wg > 1) issue_k(1);
    }
  }
  const bool any = kTeams == 1 || n_tiles_wave > 0;
  if (any) scores(kbuf);
  if (team == 0) softmax(0);
  wait_staged();
  __syncthreads();  // K tile 0 (and the query rows) has been read: its slot may be refilled; V 0 and K 1 are there

  // interval i: O += V(i)^T P(i), S(i+1) = K(i+1) Q^T, P(i+1); K(i+2) and V(i+1) are requested meanwhile. The second team
  // takes the softmax first (of S(i)): the two waves of a SIMD are in different phases.
  auto run = [&](auto second_tag) __attribute__((always_inline)) {
    constexpr bool SECOND = decltype(second_tag)::value;
    int i = 0;
    for (; i + 1 < n_tiles_wave; ++i) {
      if (i + 2 < n_tiles_wg) issue_k(i + 2);
      issue_v(i + 1);
      if constexpr (SECOND) {
        softmax(i);
        __builtin_amdgcn_sched_barrier(0);
      }
      matrix_block(vbuf + (i & 1) * L::kVTile, kbuf + ((i + 1) & 1) * L::kKTile);
      if constexpr (!SECOND) softmax(i + 1);
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    }
    for (; i < intervals; ++i) {
      if (i + 2 < n_tiles_wg) issue_k(i + 2);
      if (i + 1 < n_tiles_wg) issue_v(i + 1);
      if (i < n_tiles_wave) {
        if constexpr (SECOND) softmax(i);
        accumulate(vbuf + (i & 1) * L::kVTile);
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    }
  };
  // Long streams (kHalvesFrom): a team's interval is its products of V(i) and K(i+1), a barrier, the softmax of tile i+1, a barrier, and
  // the second team is half an interval behind. Slots are requested anew as soon as the products have read them, V(i+2) and K(i+3),
  // which then have the softmax and a whole interval to land, instead of one interval that ends with everything landed.
  auto run_halves = [&]() __attribute__((always_inline)) {
    auto request = [&](int i) __attribute__((always_inline)) {
      if (i + 2 < n_tiles_wg) issue_v(i + 2);
      if (i + 3 < n_tiles_wg) issue_k(i + 3);
    };
    request(-1);
    if (team == 1) {
      if (any) softmax(0);
      __syncthreads();
    }
    int i = 0;
    for (; i + 3 < n_tiles_wg && i + 1 < n_tiles_wave; ++i) {
      matrix_block(vbuf + (i & 1) * L::kVTile, kbuf + ((i + 1) & 1) * L::kKTile);
      __syncthreads();
      request(i);
      softmax(i + 1);
      wait_staged<kLoadsV + kLoadsK>();  // V(i+1) and K(i+2) are there, what has just been requested may be on its way
      __syncthreads();
    }
    for (; i < intervals; ++i) {
      if (i + 1 < n_tiles_wave) matrix_block(vbuf + (i & 1) * L::kVTile, kbuf + ((i + 1) & 1) * L::kKTile);
      else if (i < n_tiles_wave) accumulate(vbuf + (i & 1) * L::kVTile);
      __syncthreads();
      request(i);
      if (i + 1 < n_tiles_wave) softmax(i + 1);
      if (i + 3 < n_tiles_wg) wait_staged<kLoadsV + kLoadsK>();
      else if (i + 2 < n_tiles_wg) wait_staged<kLoadsV>();
      else wait_staged();
      __syncthreads();
    }
    if (team == 0) __syncthreads();
  };
  if (kHalves && intervals >= kHalvesFrom) run_halves();
  else if (kTeams == 1 || team == 0) run(std::false_type{});
  else run(std::true_type{});

  // ---- several parts: the other waves of a row block hand accumulator, maximum and sum to its first one, which rescales
  // all to the common maximum and adds them. The rings are free (every wave passed the barrier behind the last interval).
  if constexpr (PARTS > 1) {
    constexpr int kExch = L::kTurn;  // DVB * 16 accumulator values and (m, l) per lane
    static_assert(kExch == DVB * 4 * 64 * 16 + 64 * 8, "exchange area");
    auto area = [&](int from) __attribute__((always_inline)) { return smem + ((from - 1) * L::kRowBlocks + row_block) * kExch; };
    if (part > 0) {
      char* const exch = area(part);
#pragma unroll
      for (int i = 0; i < DVB; ++i)
#pragma unroll
        for (int b4 = 0; b4 < 4; ++b4) {
          const f32x4 v4 = {oacc[i][4 * b4], oacc[i][4 * b4 + 1], oacc[i][4 * b4 + 2], oacc[i][4 * b4 + 3]};
          *reinterpret_cast<f32x4*>(exch + ((i * 4 + b4) * 64 + lane) * 16) = v4;
        }
      const f32x2 ml = {m_run, l_run};
      *reinterpret_cast<f32x2*>(exch + DVB * 4 * 64 * 16 + lane * 8) = ml;
    }
    __syncthreads();
    if (part > 0) return;
    f32x2 ml[L::kParts - 1];
    float m_new = m_run;
#pragma unroll
    for (int n = 0; n < L::kParts - 1; ++n) {
      ml[n] = *reinterpret_cast<const f32x2*>(area(n + 1) + DVB * 4 * 64 * 16 + lane * 8);
      m_new = fmaxf(m_new, ml[n][0]);
    }
    // a part that saw no key has m = -inf, l = 0 and a zero accumulator: weight 0
    const float w0 = (m_run == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((m_run - m_new) * p.kappa);
    m_run = m_new;
    l_run *= w0;
#pragma unroll
    for (int i = 0; i < DVB; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) oacc[i][v] *= w0;
#pragma unroll
    for (int n = 0; n < L::kParts - 1; ++n) {
      const float w = (ml[n][0] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((ml[n][0] - m_new) * p.kappa);
      l_run += ml[n][1] * w;
#pragma unroll
      for (int i = 0; i < DVB; ++i)
#pragma unroll
        for (int b4 = 0; b4 < 4; ++b4) {
          const f32x4 v4 = *reinterpret_cast<const f32x4*>(area(n + 1) + ((i * 4 + b4) * 64 + lane) * 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) oacc[i][4 * b4 + e] += v4[e] * w;
        }
    }
  }

  // ---- epilogue: normalise, store O (bf16) and LSE2; the rings are free (every wave passed the last barrier)
  __bf16* oh = p.o + b * p.o_bs + (int64_t)h * kDv;
  float* lse = p.lse + b * p.lse_bs + (int64_t)h * p.lse_hs;
  const float l = pair_sum(l_run);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  char* const turn = smem + row_block * L::kTurn;
  if constexpr (!CAUSAL && kDv == 128) {
    if (p.prev_o != nullptr) {  // merge with the running result of the rows, as in attn_fwd_direct.hip
      const float lse_new = l > 0.f ? __builtin_amdgcn_logf(l) + m_run * p.kappa : -INFINITY;
      const float lse_old = qrow < p.Sq ? lse[qrow] : -INFINITY;
      const float big = fmaxf(lse_old, lse_new);
      const float w_old = big == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(lse_old - big);
      const float w_new = big == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(lse_new - big);
      const float den = w_old + w_new;
      const float rden = den > 0.f ? 1.f / den : 0.f;
      const int64_t prev_rs = o_row_stride;
      const char* prev = reinterpret_cast<const char*>(p.prev_o) +
                         (b * p.prev_bs + (int64_t)h * kDv + q_wave0 * prev_rs) * (p.prev_f32 ? 4 : 2);
      const bool to_o = p.o && q_wave0 >= p.o_r0 && q_wave0 < p.o_r1;
      const bool to_acc = p.acc_o && q_wave0 >= p.acc_r0 && q_wave0 < p.acc_r1;
      merge_rows32_via_lds<DVB>(turn, prev, p.prev_f32 != 0, prev_rs, to_o ? oh + q_wave0 * o_row_stride : nullptr, o_row_stride,
                                to_acc ? p.acc_o + b * p.acc_bs + (int64_t)h * kDv + q_wave0 * o_row_stride : nullptr,
                                o_row_stride, p.Sq - q_wave0, oacc, w_new * inv * rden, w_old * rden, lane);
      if (qrow < p.Sq && g == 0) lse[qrow] = den > 0.f ? big + __builtin_amdgcn_logf(den) : -INFINITY;
      return;
    }
  }
  store_rows32_via_lds<__bf16, DVB>(turn, oh + q_wave0 * o_row_stride, o_row_stride, p.Sq - q_wave0, oacc, inv, false, lane, p.through_o);
  if (qrow < p.Sq && g == 0) lse[qrow] = (l > 0.f) ? __builtin_amdgcn_logf(l) + m_run * p.kappa : -INFINITY;
}

// Tiles from which the heads are taken in chunks (decode_block). Taken level by level (every head's tile t before any tile
// t-1), the workgroups in flight stream K and V of all heads, which costs nothing while the last-level cache (256 MB) holds
// them; once it does not, every level reads them from memory, and with 128-row workgroups half as many rows share a stream as
// with 256-row ones. So the line is the size of K and V, however many the tiles; under the mask a row sees half of the keys
// and heaviest-first over the whole grid is worth something, hence a higher one. From 192 heads on a chunk's tiles are in flight
// together and read its K and V through one L2: without a mask, chunks for any size. Level by level / in chunks, us:
//   d192 full    4096 x 64 heads (160 MiB) 588 / 601     8192 x 40 (200) 1381 / 1432    16384 x 24 (240) 3240 / 3300
//                4096 x 96 (240) 932 / 899               6144 x 64 (240) 1278 / 1260    8192 x 64 (320) 2484 / 2249
//                4096 x 128 (320) 1437 / 1189            6144 x 128 (480) 3385 / 2533   1024 x 256 (160) 207 / 179
//                768 x 256 (120) 123 / 104               512 x 384 (120) 91 / 80        384 x 512 of 64 features 35.4 / 32.5
//        causal  8192 x 24 (120) 441 / 475               8192 x 40 (200) 718 / 765      9216 x 40 (225) 898 / 947
//                4096 x 104 (260) 523 / 546              32768 x 16 (320) 4280 / 4319   2 x 16384 x 16 (320) 2230 / 2202
//                4096 x 128 (320) 682 / 671              4096 x 256 (640) 1679 / 1292   2048 x 224 (280) 366 / 345
//   d64  full    8192 x 64 (128) 1081 / 1079             8192 x 128 (256) 2266 / 2116   1024 x 512 (128) 173 / 158
//        causal  8192 x 32 (64) 276 / 303                16384 x 64 (256) 2190 / 2249   16 x 4096 x 32 (512) 1582 / 1243
// A walk over several chunks of keys has them one after the other: what counts is the size of one, and it takes many heads;
// otherwise the line of many tiles stands. 4 ranks, d192, level by level / in chunks: 4096 x 128 heads (320 MiB a chunk) 2735 /
// 2431 and 4830 / 4101; 3072 x 128 (240) 1425 / 1402 and 2533 / 2255; 2048 x 128 (160) 659 / 680 and 1152 / 1060; 4096 x 64
// (160) 1149 / 1177 and 2004 / 2002; 6144 x 64 (240) 2675 / 2708; 8192 x 32 (160) 2278 / 2234 and 4014 / 3833.
template <int DQK, bool MULTI>
int chunked_tiles(const FwdArgs<MULTI>& p, bool causal) {
  const bool two_part = DQK == 192 && chunk_of(p, 0).k_pe != nullptr;
  const int64_t keys = chunk_of(p, chunk_count(p) - 1).rows, heads = (int64_t)p.B * p.Hkv;  // (the last chunk is a whole one)
  const int64_t mib = keys * heads * ((two_part ? 128 : DQK) + (DQK == 64 ? 64 : 128)) * 2 >> 20;
  if (MULTI) return heads >= 96 && mib >= 200 ? 1 : kChunkedTiles;
  const int64_t line = causal ? (DQK != 64 && heads >= 208 ? 240 : 288) : heads >= 192 ? 0 : heads >= 64 ? 200 : 256;
  return mib >= line ? 1 : 0x7fffffff;
}

template <int DQK, int PARTS, bool MULTI>
void launch_one(FwdArgs<MULTI> p, bool causal, hipStream_t st) {
  using L = DuoLayout<DQK, PARTS>;
  p.m_tiles = (p.Sq + L::kBM - 1) / L::kBM;
  p.chunked = chunked_tiles<DQK, MULTI>(p, causal);
  const dim3 grid((unsigned)(p.m_tiles * p.Hq * p.B)), block(L::kThreads);
  if constexpr (MULTI) {  // the last chunk is seen under the mask
    hipLaunchKernelGGL((attn_fwd_duo_kernel<DQK, PARTS, true, true>), grid, block, 0, st, p);
  } else {
    if (causal) hipLaunchKernelGGL((attn_fwd_duo_kernel<DQK, PARTS, true, false>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((attn_fwd_duo_kernel<DQK, PARTS, false, false>), grid, block, 0, st, p);
  }
}

template <int DQK, bool MULTI>
void launch_parts(const FwdArgs<MULTI>& p, int parts, bool causal, hipStream_t st) {
  if (parts == 1) launch_one<DQK, 1, MULTI>(p, causal, st);
  else if (parts == 3) launch_one<DQK, 3, MULTI>(p, causal, st);
  else if (parts == 4) launch_one<DQK, 4, MULTI>(p, causal, st);
  else if constexpr (DQK == 64) launch_one<DQK, 2, MULTI>(p, causal, st);
}

template <bool MULTI>
void launch_dim(const FwdArgs<MULTI>& p, int dqk, int parts, bool causal, hipStream_t st) {
  if (dqk == 64) launch_parts<64, MULTI>(p, parts, causal, st);
  else if (dqk == 128) launch_parts<128, MULTI>(p, parts, causal, st);
  else launch_parts<192, MULTI>(p, parts, causal, st);
}

}  // namespace

void launch_fwd_duo(const FwdParams& p, int dqk, int parts, bool causal, hipStream_t st) { launch_dim<false>(p, dqk, parts, causal, st); }

void launch_fwd_duo(const FwdChunkParams& p, int dqk, int parts, bool causal, hipStream_t st) { launch_dim<true>(p, dqk, parts, causal, st); }

}  // namespace pith
