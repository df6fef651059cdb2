// Entry points of the key/value-gradient step of one chunk attention backward for gfx950, against an external
// (ring-combined) base-2 LSE and delta = rowsum(O*dO): argument checks, the head split and its reduction kernel. The
// kernels are attn_bwd_dkdv_d64.hip, attn_bwd_dkdv_d128.hip, attn_bwd_dkdv_wide.hip and attn_bwd_dkdv_d192.hip.
//
// With grouped-query attention the heads of a group may be cut into `split` parts handled by
// different workgroups (more parallelism when there are few key tiles); the parts leave fp32
// partial results in a caller-provided workspace and a second kernel adds them in a fixed
// order, so the result does not depend on scheduling.
#include <algorithm>
#include <mutex>

#include "attn_bwd_common.h"
#include "handover_rows.h"

namespace pith {
namespace {

constexpr int kBN = kDkdvBlockN;  // key rows per workgroup (128 features: or kDkdvWideN)

// out[b, s, h, :] (+)= sum over parts of ws[part][b][s][h][:], parts added in index order; blockIdx.y picks the item (dK and
// dV of a call, or those of all its chunks).
struct ReduceItem {
  const float* ws;
  void* out;
  int64_t part_stride, row_elems, out_bs, n4;
  int64_t out_row_elems;  // elements between consecutive rows of `out` (>= row_elems: a head range of a wider tensor)
  int64_t rows_per_batch;
};
template <int N>
struct ReduceParams {
  ReduceItem item[N];
  int parts, accumulate;
};

// Bound by latency where the parts are many and small: the sum over 16 heads of the two-part keys of three 1021-row chunks 6.3 us with one
// load at a time and 64-bit divisions, 4.0 with three in flight (seven: 4.7; loads that are not non-temporal 4.6). Large sums
// (four parts of 8.4 MB each) run at copy rate either way, 13.5-13.9.
constexpr int kInFlight = 3;
__device__ __forceinline__ f32x4 load_part(const float* src) { return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(src)); }

template <typename OutT, int N>
__global__ __launch_bounds__(256) void reduce_parts_kernel(ReduceParams<N> p) {
  const ReduceItem& r = p.item[blockIdx.y];
  const float* __restrict__ ws = r.ws;
  OutT* out = reinterpret_cast<OutT*>(r.out);
  const int64_t part_stride = r.part_stride, n4 = r.n4;
  auto sum_rows = [&](auto index_tag) {
    using Index = decltype(index_tag);  // 32 bits where they do: a 64-bit division is a hundred instructions
    const Index row_elems = (Index)r.row_elems, per_batch = (Index)r.rows_per_batch * row_elems, end = (Index)n4;
    for (Index i = (Index)blockIdx.x * blockDim.x + threadIdx.x; i < end; i += (Index)gridDim.x * blockDim.x) {
      const Index e = i * 4;
      const float* src = ws + e;
      f32x4 s = load_part(src);
      int left = p.parts - 1;
      for (; left >= kInFlight; left -= kInFlight) {
        f32x4 x[kInFlight];
#pragma unroll
        for (int j = 0; j < kInFlight; ++j) x[j] = load_part(src += part_stride);
#pragma unroll
        for (int j = 0; j < kInFlight; ++j) s += x[j];
      }
      for (; left > 0; --left) s += load_part(src += part_stride);
      const Index bb = e / per_batch;
      const Index in_batch = e - bb * per_batch;
      const Index row = in_batch / row_elems;
      OutT* dst = out + bb * r.out_bs + row * r.out_row_elems + (in_batch - row * row_elems);
      store4<OutT>(dst, s[0], s[1], s[2], s[3], p.accumulate != 0);
    }
  };
  if (n4 <= 1 << 28) sum_rows(uint32_t{});
  else sum_rows(int64_t{});
}

// A launch of the above, item by item.
template <int N>
struct Reduction {
  ReduceParams<N> p;
  int n = 0;
  int64_t max_n4 = 0;

  void add(const float* ws, void* out, int64_t out_bs, int64_t batch, int64_t rows, int64_t row_elems, int64_t out_row_elems) {
    ReduceItem& r = p.item[n++];
    r.ws = ws; r.out = out; r.out_bs = out_bs;
    r.row_elems = row_elems; r.out_row_elems = out_row_elems; r.rows_per_batch = rows;
    r.part_stride = batch * rows * row_elems;
    r.n4 = r.part_stride / 4;
    if (r.n4 > max_n4) max_n4 = r.n4;
  }
  void launch(int parts, bool accumulate, bool f32, hipStream_t st) {
    p.parts = parts;
    p.accumulate = accumulate;
    const int64_t blocks = (max_n4 + 255) / 256;
    const dim3 grid((unsigned)(blocks < 8192 ? blocks : 8192), n);
    if (f32) hipLaunchKernelGGL((reduce_parts_kernel<float, N>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((reduce_parts_kernel<__bf16, N>), grid, dim3(256), 0, st, p);
  }
};

// The head split doubles until the workgroups wanted are there, which leaves up to twice as many. Whether half of those do better, a
// round of them without a mask, one to two (W workgroups per unit) under it: they leave half of the partial sums, which make a round
// trip through memory, and spend half as often what a workgroup spends around its products (7 us). Long walks (rows x heads of a part) lose, the
// sooner the fewer workgroups are there to even them out: in a call that hands dS over nothing else fills the units. Forward + backward, more / half,
// us, 32/4 heads unless others are named:
//   causal d128, handing over, by W and walk
//                1.0         2080 13 x 520 x 16/4 155 / 147, 3072 11 x 768 x 16/4 198 / 187; 4160 13 x 520 265 / 273, 5472 3 x 1368 254 / 278, 12288 11 x 768 x 64/4 647 / 692
//                1.12-1.17   4096 9 x 1024 x 16/4 235 / 225, 5120 15 x 640 350 / 331; 6000 3 x 1500 294 / 313, 10624 12 x 664 x 64/4 603 / 648
//                1.2-1.3     6000 7 x 1500 x 16/4 335 / 325, 6144 13 x 768 394 / 375, 3600 5 x 900 231 / 234; 7200 5 x 900 x 64/4 411 / 424, 11344 13 x 709 x 64/4 744 / 752
//                1.38-1.5    7200 11 x 900 456 / 439, 9216 5 x 1152 x 64/4 557 / 551, 12288 15 x 768 x 64/4 858 / 836; 7200 3 x 1800 392 / 399, 14400 3 x 1800 x 64/4 746 / 763,
//                            21888 8 x 1368 x 64/4 1223 / 1256
//                1.55-1.9    3600 2 x 1800 281 / 258, 9216 11 x 1152 616 / 593, 16384 13 x 1024 x 64/4 1151 / 1119, 18432 11 x 1152 x 64/4 1199 / 1186, 28800 equal
//                not         1.0 11 x 709 x 8/2 118 / 107, 1.12 2304 239 / 224, 9 x 400 x 16/4 104 / 89, 1.4 2 x 1368 201 / 185, 1.5 3 x 900 172 / 157; 3000 x 64/4 600 / 617
//                short rows  24 x 128 112 / 92, 20 x 160 111 / 97, 10 x 200 x 64/4 143 / 125
//   full   d128  1100 134.7 / 119.6, 1300 162 / 150, 1790 253 / 242, 3 x 700 155 / 145, 3 x 1408 x 8/2 153 / 140, 2 x 2100 x 8/2 209 / 188, 2700 566 / 530; rows that
//                do not hand over 4 x 520 133.7 / 125.8, 4 x 600 x 64/4 290 / 268, 9 x 560 x 16/4 154 / 135, 20 x 160 119.6 / 103.8, 40 x 100 113 / 96, 33 x 100 110 /
//                91; 5000 x 8/2 442 / 462, 3500 x 64/4 1509 / 1523. Calls that hand dS over leave at most a quarter of the units idle (ds_handover_pays).
//   d64          causal 9 x 1100 x 32/8 303 / 280, 5 x 1290 x 32/8 236 / 216, 4300 x 32/8 369 / 361, 20 x 250 x 32/8 95 / 84, 3 x 2200 x 16/4 equal;
//                full 10 x 600 x 16/4 114 / 106, 4 x 1290 x 32/8 305 / 295, 2600 x 32/8 281 / 274, 2200 x 32/8 equal
// Several chunks, whose workgroups are unequal, in one grid with more than one dQ workgroup per unit to even them out: four ranks, 1100 contiguous
// rank 3 392 / 371, 2 x 900 zigzag 328 / 310, 600 x 64/4 173 / 163, 2 x 2400 x 8/2 500 / 459, 5000 x 8/2 contiguous 1177 / 1117, 8200 x 8/2 2497 / 2430, 3300
// equal. Not with fewer (2 x 1314 x 8/2 188 / 195, eight ranks 900 335 / 342) nor with more than four, where the two differ by -2 to +2 % (one grid 2300 x 64/4
// 1439 / 1426, 2 x 1200 x 64/4 887 / 885, 2500 x 64/4 contiguous 2894 / 2847, 2050 x 64/4 2058 / 2100), two ranks 3348 x 64/4 1529 / 1689.
// half: the parts there would be
bool half_as_many(const pith_attn_bwd_args* a, int64_t tiles, int half, bool chunks) {
  const int64_t cus = compute_units_or_default(), wgs = tiles * a->Hkv * a->B * half;
  if (chunks) {
    const int64_t q_wgs = (a->Sq + 127) / 128 * a->Hq * a->B;
    return a->Dqk == 128 && q_wgs > cus && q_wgs <= 4 * cus;
  }
  if (a->Dqk == 192) return false;
  if (a->Dqk == 64) return a->Sq <= 5120;
  const bool hands_over = handover_rows_pay(a->B, a->Sq, a->Hq, a->causal != 0, cus);
  if (!a->causal) return a->Sq <= 2816 && (!hands_over || 4 * wgs >= 3 * cus);
  if (a->Sq > (5 * wgs >= 8 * cus ? 4096 : 2304)) return false;
  const int64_t walk = a->Sq * (a->Hq / a->Hkv / half);
  return !hands_over || walk <= (8 * wgs <= 9 * cus ? 4096 : 8 * wgs < 11 * cus ? 6144 : 2 * wgs <= 3 * cus ? 12288 : 24576);
}

// tiles: key tiles of the launch, over all of its chunks
int pick_split(const pith_attn_bwd_args* a, int64_t tiles, bool chunks = false) {
  const int64_t group = a->Hq / a->Hkv;
  const int64_t base = tiles * a->Hkv * a->B;
  int split = 1;
  // Workgroups wanted. Without a causal mask all of them carry the same work, so one full round is ideal; under the mask
  // two rounds (heaviest first) balance better. At 64 features two workgroups share a compute unit and twice as many are
  // wanted (8192 rows x 32 heads causal: 757 us with 512 workgroups, 560 us with 1024; without a mask 512 and 1024 are
  // within 2 %).
  const int64_t want = (a->causal ? 2 : 1) * (a->Dqk == 64 ? 2 : 1) * (int64_t)compute_units_or_default();
  while (split < group && base * split < want && group % (split * 2) == 0) split *= 2;
  if (split > 1 && base * split > want && half_as_many(a, tiles, split / 2, chunks)) split /= 2;
  return split;
}

// Workspace layout: [head-split partial dK | partial dV] (split > 1), then the per-head gradients of a
// shared k_pe [Hkv][B][Skv][64] (keys in two parts).
int64_t split_bytes_for(const pith_attn_bwd_args* a, int split) {
  if (split <= 1) return 0;
  return (int64_t)split * a->B * a->Skv * a->Hkv * (a->Dqk + a->Dv) * (int64_t)sizeof(float);
}
int64_t dkpe_bytes_for(const pith_attn_bwd_args* a) {
  return a->k_pe ? a->Hkv * a->B * a->Skv * 64 * (int64_t)sizeof(float) : 0;
}
int64_t workspace_bytes_for(const pith_attn_bwd_args* a, int split) { return split_bytes_for(a, split) + dkpe_bytes_for(a); }

// How a dK/dV call is cut: key rows per workgroup and head parts. A pair in one grid with dQ has workgroups of kBN rows.
struct Plan {
  int rows, split;
};
Plan plan_for(const pith_attn_bwd_args* a, int rows) { return {rows, pick_split(a, (a->Skv + rows - 1) / rows)}; }
int64_t workgroups(const pith_attn_bwd_args* a, const Plan& p) { return (a->Skv + p.rows - 1) / p.rows * a->Hkv * a->B * p.split; }

// Whether a call of 128 features and not too few rows, launched alone, goes to the workgroups of kDkdvWideN keys (attn_bwd_dkdv_wide.h), which are
// 4-7 % faster per product. Half as many workgroups cost
//   - without a mask, a longer last round: the rounds are compared (5000 x 16 heads, 320 workgroups of 256 keys: +17 %);
//   - under it, balance, below two workgroups per unit (8192 x 8/8 +34 %, 12288 x 8/8, 1.5 per unit, +5 %), and the products of
//     256 instead of 128 keys with rows that see none of them, so not for short rows;
//   - a finer head split, whose partial sums make a round trip: each part needs work for it. dK/dV + sums, 128 -> 256 keys, us,
//     (mean rows per key) x (heads of a part) behind it: causal 4096 x 32/4 293 -> 311 (2048), 6144 x 32/4 651 -> 668 (3072),
//     4096 x 64/4 600 -> 585 (4096), 8192 x 32/4 1141 -> 1100 (8192); full 3072 x 32/4 339 -> 344 (3072), 2 x 2048 x 32/4 267 ->
//     268 (4096 in short rows), 4096 x 32/4 529 -> 514 (8192), 8192 x 4096 x 32/4 1061 -> 1018, 16384 x 8192 x 16/1 2077 -> 1992.
// Without a finer split: full 16 x 1024 x 16 333 -> 309, 8192 x 16 1064 -> 1013; causal 16 x 1024 x 16 221 -> 215, 2 x 8192 x 8
// 579 -> 545 (all handing dS over; recomputing 0-7 % faster). A call that fits the built-in scratch of pith_attn_bwd_dkdv_static
// with 128 keys has to fit it with 256, too, so that both entry points add up in the same order. This keeps two of the measured
// calls above on 128 keys, causal 4096 x 64/4 and 8192 x 32/4 (64 MB of partial sums, 128 with 256 keys), and the causal steps of
// shares of 16384 x 64/4 (none, 128 MB).
bool wide(const pith_attn_bwd_args* a, const Plan& n, const Plan& w) {
  const int64_t cus = compute_units_or_default(), narrow_wgs = workgroups(a, n), wide_wgs = workgroups(a, w);
  const int64_t narrow_heads = a->Hq / a->Hkv / n.split, wide_heads = a->Hq / a->Hkv / w.split;
  if (w.split > 1 && (a->Sq < 4096 || (a->causal ? a->Sq / 2 : a->Sq) * wide_heads < 4096)) return false;
  const int64_t fits = PITH_DKDV_STATIC_SCRATCH_BYTES;
  if (workspace_bytes_for(a, w.split) > fits && workspace_bytes_for(a, n.split) <= fits) return false;
  if (a->causal) return wide_wgs >= 2 * cus;
  return (wide_wgs + cus - 1) / cus * 2 * wide_heads <= (narrow_wgs + cus - 1) / cus * narrow_heads;
}
// `n`: the plan with kBN rows
Plan pick_plan(const pith_attn_bwd_args* a, const Plan& n) {
  if (a->Dqk != 128 || a->Sq < (a->causal ? 1024 : 512)) return n;
  const Plan w = plan_for(a, kDkdvWideN);
  return wide(a, n, w) ? w : n;
}

constexpr int64_t kWalkDescBytes = 192ll << 20;

// with_dq: dQ of the pair in the same grid (p prepared for it)
template <int DQK, int DV>
void launch_dkdv(BwdParams p, const pith_attn_bwd_args* a, int rows, bool with_dq, hipStream_t st) {
  p.tiles = (int)((a->Skv + rows - 1) / rows);
  p.accumulate = a->accumulate_dkv;
  p.main_blocks = (int)(p.tiles * a->Hkv * a->B * p.split);
  p.zero_tail = a->accumulate_dkv ? 0 : (int)a->dkv_zero_tail;  // rows that are added to keep what they hold
  const unsigned grid = (unsigned)(p.main_blocks + (p.zero_tail + kZeroTailRows - 1) / kZeroTailRows);
  const bool f32 = a->dkv_dtype == PITH_F32;
  if (with_dq) {
    launch_bwd_pair(p, DQK, a->causal != 0, f32, a->dq_dtype == PITH_F32, grid, st);
  } else if constexpr (DQK == 128 && DV == 128) {
    // descending walk under the mask when Q and dO together exceed what the last-level cache (256 MB) keeps
    p.walk_desc = a->causal != 0 && (int64_t)a->B * a->Sq * a->Hq * (DQK + DV) * 2 > kWalkDescBytes;
    if (rows == kDkdvWideN) launch_dkdv_wide(p, a->causal != 0, f32, grid, st);
    else launch_dkdv_d128(p, a->causal != 0, f32, grid, st);
  } else if constexpr (DQK == 192 && DV == 128) {
    launch_dkdv_d192(p, a->causal != 0, f32, grid, st);
  } else {
    launch_dkdv_d64(p, a->causal != 0, f32, grid, st);
  }
  if (p.k_pe) {  // dk_pe (+)= sum over heads, in head order
    Reduction<2> r;
    r.add(p.ws_dkpe, a->dk_pe, a->dk_pe_bs, a->B, a->Skv, 64, 64);
    r.launch((int)a->Hkv, a->accumulate_dkv, f32, st);
  }
  if (p.split > 1) {
    Reduction<2> r;
    r.add(p.ws_dk, a->dk, a->dk_bs, a->B, a->Skv, a->Hkv * a->Dqk, p.HkvT * a->Dqk);
    r.add(p.ws_dv, a->dv, a->dv_bs, a->B, a->Skv, a->Hkv * a->Dv, p.HkvT * a->Dv);
    r.launch(p.split, a->accumulate_dkv, f32, st);
  }
}

// Whether dK/dV and dQ go out as one grid (no dS handed over). At 128 and 192 features the dQ workgroups are then the
// split-key ones (the two kernels must agree on the workgroup size), which is what grids of up to one workgroup per compute
// unit want anyway. Beyond, one grid pays where either kernel alone would leave its last round half empty, against what the
// two-workgroup dQ kernel is faster by; W = dQ workgroups per compute unit, apart -> together, inputs from memory, us:
//   d128 causal   W 1.5: 1 x 2304 x 16 108 -> 91, 1 x 6144 x 8/2 289 -> 265, 6 x 512 x 16/4 68 -> 61; 1.75: 1 x 1792 x 32/4
//                 122 -> 121; 2: 1 x 2048 x 32/4 154 -> 150, 1 x 8192 x 8/2 446 -> 449; 2.25: 1 x 2304 x 32/4 191 -> 181
//        full     W 1.5: 1 x 1536 x 32/4 157 -> 145; 1.7: 1 x 3456 x 16 307 -> 329; 2: 1 x 4096 x 16 412 -> 422;
//                 2.2: 1 x 4480 x 16 628 -> 520, 1 x 2304 x 32/4 383 -> 289
//   d192 causal   W 1.1: 1 x 4608 x 8 246 -> 198; 1.5: 1 x 3072 x 16 193 -> 186; 1.7: 1 x 3456 x 16
//                 227 -> 227; 2: 1 x 2048 x 32 171 -> 175; 2.2: 1 x 2560 x 28 233 -> 242
// and with the forward, since the head split halves (half_as_many). These calls recompute; from two thirds of a device of query rows on (about W 2.8) most hand dS over and have
// two launches in any case, so that the upper lines hold for those which do not: up to 256 rows, unmasked 513 to 639, more than 16384 of few heads, groups of an odd number of
// heads, fp32 results, no room for the buffer.
//   d128 causal   W 1.6: 13 x 500 x 8/2 86.5 -> 80.7; 2: 2 x 1000 x 32/4 128 -> 125, 4 x 500 x 32/4 97.6 -> 96.3, 4 x 512 98.4 -> 97.5, 2 x 900 117.2 -> 111.5; 2.25-2.8: 3 x 768 x 32/4 116.4 ->
//                 107.4, 3 x 700 108.4 -> 100.3, 6 x 384 89 -> 86, 5 x 450 101 -> 98, 1 x 2700 322 -> 309, 1 x 1500 x 60/4 546 -> 505, 3 x 1000 x 30/2 386 ->
//                 352, 3 x 1900 x 16 234 -> 231; 2.9-3.3: 1 x 6000 x 16 652 -> 629, 1 x 3000 x 32/4 369 -> 361, 1 x 3300 423 -> 410, 1 x 13000 x 8/2 1461
//                 -> 1429, 1 x 3100 x 34/2 1209 -> 1121; 3.5: 1 x 3500 x 32/4 456 -> 459, 7 x 900 x 16 equal; 5: 20 x 160 x 32/4 99 -> 107
//        full     W 1.75-2: 1 x 1700 x 32/4 227 -> 235, 2 x 900 148 -> 153; 2.6-3.1: 3 x 900 x 28/4 257 -> 214, 1 x 1400 x 62/2 989 -> 917, 1 x 2816 x 32/4 578
//                 -> 561, 1 x 6000 x 16 and 1 x 12500 x 8/2 equal; 3.25-3.5: 1 x 3300 x 32/4 763 -> 772, 7 x 900 x 16 263 -> 267
//   d192 causal   W 1.1-1.4: 2 x 1100 x 16 109.6 -> 95.6, 2 x 1400 x 16 139 -> 128, 1 x 1300 x 32 129 -> 119, 3 x 800 x 16 92.7 -> 89.2, 3 x 384 x 32 81 -> 78;
//                 1.5: 3 x 1024 x 16 120 -> 116, 1 x 1500 x 32 equal; 2.25: 9 x 400 x 16 99 -> 105
// Several chunks, whose dK/dV workgroups are more unequal, gain 1-5 % up to two per unit (2048 x 32/4 of 128, 4 ranks,
// zigzag, rank 0: 525 -> 498 us; 4096 x 16 of 192, rank 3: 1099 -> 1081). 128 features: up to four, where two launches lost
// even to one pair of them per ring step (in brackets): 4096 x 32/4, 4 ranks, rank 0 1889 -> 1728 (1724); 9216 x 8/2, 8
// ranks, contiguous 5439 -> 4593 (4746); 12288 x 8/2, rank 0 4120 -> 3875 (3878), rank 1 4040 -> 3721 (3930); 3584 x 32/4,
// rank 3 1286 -> 1295 (1417). 192 features with three lose (6144 x 16: 2385 -> 2413). 128 features also up to eight where a share
// is more than a whole chunk beside its own (forward + backward, 4 ranks, apart -> together): 4.2 17000 x 8/2 10670 -> 9880; 4.5 2300 x 64/4
// 1588 -> 1488; 5 2 x 1200 x 64/4 974 -> 882, 5120 x 32/4 3272 -> 3232; 6 6144 x 32/4 4866 -> 4590; 7 2 x 1700 x 64/4 contiguous 1994 -> 1928; 8 8 x 1024 x 32/4
// equal; 9 to 11 9216 x 32/4 10400 -> 10540, 11264 x 32/4 15150 -> 15480; two ranks 2 x 3000 x 32/4 contiguous 1733 -> 1749.
// At 64 features both kernels fit two workgroups to a unit, and one grid is faster for chunk pairs and most shares: forward +
// backward, apart -> together, 1 x 32768 x 8/2 heads causal 4808 -> 4660 us, 1 x 16384 x 16/4 2423 -> 2359, 16 x 1024 x 32/8 415 ->
// 404, 1 x 16384 x 16/4 without a mask 4684 -> 4630; shares, zigzag, 4096 x 64/8, 4 ranks, rank 0 2740 -> 2543, 8192 x 32/8 rank 1
// 5084 -> 4972, 5120 x 32/8 rank 0 2284 -> 2135, 12288 x 16/4 rank 1 5771 -> 5615, 32768 x 8/2, 2 ranks, rank 0 10660 -> 10224, 16384 x
// 32/8, 2 ranks 10091 -> 9983. Not where few long dQ walks start beside the last dK/dV workgroups and either kernel is whole
// rounds (three or more of dK/dV, up to four of dQ, from 12288 rows on), so that nothing is left to fill: 12288 x 16/4, 4 ranks, rank 0
// 5805 -> 5994, 16384 x 16/4 10106 -> 10295, 24576 x 8/2 11896 -> 12077, contiguous 16384 x 16/4 rank 2 12525 -> 12699, 12288 x 16/4 rank 3
// 9957 -> 10027. Whole rounds of more or shorter ones: 10240, 12288, 16384 x 32/8 7642 -> 7543, 10879 -> 10763, 19213 -> 18984, 3 x 4096 x
// 16/4 1983 -> 1964; dQ first: 16384 x 16 10221 -> 10018. Together they have to be a grid that the runtime launches (2^32 threads
// are refused), which either of them may be where both are not (65535 x 1 row x 130 heads).
bool one_grid(const pith_attn_bwd_args* a, int64_t dkdv_wgs, bool chunks) {
  if (ds_usable(a) || (a->dkv_dtype == PITH_F32 && a->dq_dtype != PITH_F32)) return false;
  const int64_t cus = compute_units_or_default();
  const int64_t q_wgs = ((a->Sq + 127) / 128) * a->Hq * a->B;
  if (a->Dqk == 64) return (q_wgs + dkdv_wgs) * 256 < (1ll << 32);
  if (chunks) return q_wgs <= (a->Dqk == 128 ? (a->Skv > 2 * a->Sq ? 8 : 4) : 2) * cus;
  if (q_wgs <= cus) return true;
  if (a->Dqk == 192) return 2 * q_wgs <= 3 * cus && a->Skv >= (a->causal ? 256 : 1536);
  if (2 * q_wgs <= 3 * cus) return true;
  return a->causal ? 3 * q_wgs <= 10 * cus && a->Skv >= 384 : q_wgs > 2 * cus && 10 * q_wgs <= 31 * cus;
}

// Workgroups of the dQ kernel that reads handed-over dS.
int64_t dq_ds_workgroups(const pith_attn_bwd_args* a) {
  const int rows = dq_ds_rows((int)a->Dqk);
  return (a->Sq + rows - 1) / rows * a->Hq * a->B;
}

}  // namespace
}  // namespace pith

using namespace pith;

extern "C" int64_t pith_attn_bwd_dkdv_workspace_bytes(const pith_attn_bwd_args* a) {
  if (!a || a->Hkv <= 0 || a->Hq <= 0 || a->Hq % a->Hkv != 0 || a->B <= 0 || a->Skv <= 0) return 0;
  // of the call alone or in one grid with dQ
  const Plan narrow = plan_for(a, kBN);
  return workspace_bytes_for(a, std::max(pick_plan(a, narrow).split, narrow.split));
}

extern "C" int pith_attn_bwd_plan(const pith_attn_bwd_args* a, pith_attn_bwd_plan_t* plan) {
  const char* who = "pith_attn_bwd_plan";
  if (!a || !plan) return fail(PITH_ERR_NULL_POINTER, "%s: %s is NULL", who, a ? "plan" : "args");
  if (a->Hkv <= 0 || a->Hq <= 0 || a->Hq % a->Hkv != 0 || a->B <= 0 || a->Sq <= 0 || a->Skv <= 0)
    return fail(PITH_ERR_BAD_SHAPE, "%s: bad shape", who);
  const Plan chosen = pick_plan(a, plan_for(a, kBN));
  plan->dkdv_rows = chosen.rows;
  plan->dkdv_split = chosen.split;
  plan->dq_ds_pairs = a->causal && ds_bytes_for(a) > 0 && dq_ds_pairs(dq_ds_workgroups(a));
  pith_attn_bwd_args bf16 = *a;
  bf16.ds = nullptr;
  bf16.dq_dtype = bf16.dkv_dtype = PITH_BF16;
  plan->one_grid = one_grid(&bf16, workgroups(a, plan_for(a, kBN)), false);
  return PITH_OK;
}

namespace {

// Keys in two parts: what the dK/dV side asks of them.
int validate_dk_pe(const pith_attn_bwd_args* a, const char* who) {
  if (!a->k_pe) return PITH_OK;
  if (a->Hq != a->Hkv)
    return fail(PITH_ERR_UNSUPPORTED, "%s: keys in two parts need Hq == Hkv (got %lld, %lld)", who, (long long)a->Hq, (long long)a->Hkv);
  if (!a->dk_pe) return fail(PITH_ERR_NULL_POINTER, "%s: dk_pe is NULL", who);
  if (!aligned16(a->dk_pe) || a->dk_pe_bs % 8) return fail(PITH_ERR_MISALIGNED, "%s: dk_pe pointer / batch stride must keep 16-byte alignment", who);
  return PITH_OK;
}

// Runs the kernels with the head-split partials in `workspace` (NULL: no head split).
int run_dkdv(const pith_attn_bwd_args* a, const Plan& plan, void* workspace, hipStream_t st, const char* who, bool with_dq = false) {
  const int split = plan.split;
  // the grid of this kernel runs over key tiles (validate_bwd bounded the query-side grid)
  if (((a->Skv + kBN - 1) / kBN) * a->Hkv * a->B * (int64_t)split > 0x7fffffffLL)
    return fail(PITH_ERR_UNSUPPORTED, "%s: Skv=%lld x Hkv=%lld x B=%lld exceeds the launch grid limit", who,
                (long long)a->Skv, (long long)a->Hkv, (long long)a->B);
  BwdParams p = make_bwd_params(a);
  if (with_dq)
    if (const int rc = prepare_dq(a, &p, who)) return rc;
  if (a->k_pe) {
    if (const int rc = validate_dk_pe(a, who)) return rc;
    if (!workspace) return fail(PITH_ERR_BAD_SHAPE, "%s: keys in two parts need a workspace of %lld bytes", who, (long long)dkpe_bytes_for(a));
    p.ws_dkpe = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + split_bytes_for(a, split));
  }
  begin_launch();
  p.through_parts = through_results(workspace_bytes_for(a, workspace ? split : 1));
  if (split > 1 && workspace) {
    p.split = split;
    p.ws_dk = reinterpret_cast<float*>(workspace);
    p.ws_dv = p.ws_dk + (int64_t)split * a->B * a->Skv * a->Hkv * a->Dqk;
  }
  // dS hand-over to the dQ call: only when the buffer is usable (otherwise the call behaves as without it)
  if (ds_usable(a)) {
    if ((uintptr_t)a->ds % 256) return fail(PITH_ERR_MISALIGNED, "%s: ds must be 256-byte aligned", who);
    p.ds = reinterpret_cast<char*>(a->ds);
  }
  if (a->Dqk == 128) launch_dkdv<128, 128>(p, a, plan.rows, with_dq, st);
  else if (a->Dqk == 192) launch_dkdv<192, 128>(p, a, plan.rows, with_dq, st);
  else launch_dkdv<64, 64>(p, a, plan.rows, with_dq, st);
  return check_launch(who);
}

// Scratch of pith_attn_bwd_dkdv_static: device memory that belongs to the library's code object
// (one copy per GPU, held until the process ends). Host code never uses this name as an address;
// it asks the runtime for the array's device address once per device and passes that on.
constexpr int64_t kStaticScratchBytes = PITH_DKDV_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device; resolved at the first call on that device.
int static_scratch(void** out, const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(PITH_ERR_LAUNCH, "%s: hipGetDevice: %s", who, hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(PITH_ERR_UNSUPPORTED, "%s: device index %d beyond %d", who, dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(PITH_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch) on device %d: %s", who, dev, hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return PITH_OK;
}

}  // namespace

namespace {

int bwd_dkdv(const pith_attn_bwd_args* a, pith_stream_t stream, const char* who, bool with_dq) {
  const int rc = validate_bwd(a, who, false, true);
  if (rc != PITH_OK) return rc;
  // Head groups are split only when the caller brought a workspace that is large enough.
  const Plan narrow = plan_for(a, kBN);
  const auto fits = [&](const Plan& plan) { return plan.split == 1 || (a->workspace && a->workspace_bytes >= workspace_bytes_for(a, plan.split)); };
  Plan plan = with_dq ? narrow : pick_plan(a, narrow);
  if (!fits(plan)) plan = narrow;
  if (!fits(plan)) plan.split = 1;
  if (a->workspace && !aligned16(a->workspace)) return fail(PITH_ERR_MISALIGNED, "%s: workspace must be 16-byte aligned", who);
  if (a->k_pe && (!a->workspace || a->workspace_bytes < workspace_bytes_for(a, plan.split)))
    return fail(PITH_ERR_BAD_SHAPE, "%s: keys in two parts need a workspace of %lld bytes, %lld given", who,
                (long long)workspace_bytes_for(a, plan.split), (long long)(a->workspace ? a->workspace_bytes : 0));
  return run_dkdv(a, plan, a->workspace, (hipStream_t)stream, who, with_dq);
}

}  // namespace

extern "C" int pith_attn_bwd_dkdv(const pith_attn_bwd_args* a, pith_stream_t stream) {
  return bwd_dkdv(a, stream, "pith_attn_bwd_dkdv", false);
}

extern "C" int pith_attn_bwd(const pith_attn_bwd_args* a, pith_stream_t stream) {
  const char* who = "pith_attn_bwd";
  if (const int rc = validate_bwd(a, who, true, true)) return rc;
  if (one_grid(a, workgroups(a, plan_for(a, kBN)), false)) return bwd_dkdv(a, stream, who, true);
  // what the second call would reject is rejected before the first has written (or added to) anything
  BwdParams dq;
  if (const int rc = prepare_dq(a, &dq, who)) return rc;
  if (const int rc = pith_attn_bwd_dkdv(a, stream)) return rc;
  return pith_attn_bwd_dq(a, stream);
}

extern "C" int pith_attn_bwd_dkdv_static(const pith_attn_bwd_args* a, pith_stream_t stream) {
  const char* who = "pith_attn_bwd_dkdv_static";
  const int rc = validate_bwd(a, who, false, true);
  if (rc != PITH_OK) return rc;
  const Plan plan = pick_plan(a, plan_for(a, kBN));
  const int64_t need = workspace_bytes_for(a, plan.split);
  if (need > kStaticScratchBytes)
    return fail(PITH_ERR_UNSUPPORTED,
                "%s: the head-split partial sums of this shape need %lld bytes, the built-in scratch holds %lld "
                "(use pith_attn_bwd_dkdv with a caller-provided workspace)",
                who, (long long)need, (long long)kStaticScratchBytes);
  void* ws = nullptr;
  if (need > 0) {
    const int src = static_scratch(&ws, who);
    if (src != PITH_OK) return src;
  }
  return run_dkdv(a, plan, ws, (hipStream_t)stream, who);
}

// ---------------------------------------------------------------------------------------------
// Several chunks of keys in one call

namespace {

// The call as one against all keys of its chunks together: what the rules for launches look at. False: malformed.
bool merged_call(const pith_attn_bwd_args* args, const pith_key_chunk* chunks, int64_t n, pith_attn_bwd_args* a, int64_t* tiles) {
  if (!args || !chunks || n < 1 || n > kMaxChunks) return false;
  *a = *args;
  a->Skv = 0;
  *tiles = 0;
  int64_t seen = 0;  // (query row, key) pairs
  for (int64_t i = 0; i < n; ++i) {
    const pith_key_chunk& c = chunks[i];
    if (c.rows <= 0 || c.rows > (1 << 24) || c.q_row0 < 0 || c.q_row0 >= args->Sq) return false;
    a->Skv += c.rows;
    *tiles += (c.rows + kBN - 1) / kBN;
    seen += i == n - 1 ? c.rows * args->Sq / 2 : c.rows * (args->Sq - c.q_row0);
  }
  a->k_pe = chunks[0].k_pe;
  a->ds = nullptr;
  a->causal = 10 * seen <= 7 * a->Skv * args->Sq;  // rows as unequal as under a mask (see pith_attn_fwd_chunks)
  return a->B > 0 && a->Hkv > 0 && a->Hq > 0 && a->Hq % a->Hkv == 0;
}

// Bytes of a chunk's dS images per (batch, query head).
int64_t chunk_ds_head_bytes(int64_t sq, const pith_key_chunk& c, bool diagonal) {
  const int qt = (int)((sq - c.q_row0 + 63) / 64), kb = (int)((c.rows + kBN - 1) / kBN);
  return (diagonal ? ds_tile_start<true>(qt, kb) : ds_tile_start<false>(qt, kb)) * kDsBlockBytes;
}

int pick_chunks_split(pith_attn_bwd_args a, int64_t tiles) {
  a.causal = 1;  // the chunks' workgroups are unequal in any case
  return pick_split(&a, tiles, true);
}

// The launches of a call of several chunks: one grid or two, and which kind goes first in one.
struct ChunkGrids {
  bool one, dq_first;
};
ChunkGrids chunk_grids(const pith_attn_bwd_args* all, int64_t tiles, int split, int64_t dkdv_blocks) {
  const int64_t cus = compute_units_or_default(), q_wgs = ((all->Sq + 127) / 128) * all->Hq * all->B;
  // In one grid the longer workgroups go first: dQ's cost 3 products per key of all chunks, dK/dV's 4 per query row and head
  // of the part. With more than a workgroup of either per compute unit the dK/dV ones, unequal over the chunks, come first in
  // any case (128 and 192 features): 2048 x 32/4 of 128, rank 0: 498 us, dQ first 518; 4096 x 16 of 192, rank 3: 1081 and 1084.
  const bool few = all->Dqk == 64 || q_wgs <= cus;
  const bool dq_first = few && 3 * all->Skv > 4 * all->Sq * (all->Hq / all->Hkv / split);
  // (64 features: see one_grid)
  const int64_t round = 2 * cus, dkdv_wgs = tiles * all->Hkv * all->B * split;
  const bool whole = q_wgs > 2 * round && q_wgs <= 4 * round && q_wgs % round == 0 && dkdv_wgs >= 3 * round && dkdv_wgs % round == 0;
  return {one_grid(all, dkdv_blocks, true) && !(all->Dqk == 64 && !dq_first && all->Sq >= 12288 && whole), dq_first};
}

}  // namespace

extern "C" int pith_attn_bwd_chunks_plan(const pith_attn_bwd_args* args, const pith_key_chunk* chunks, int64_t n, pith_attn_bwd_plan_t* plan) {
  const char* who = "pith_attn_bwd_chunks_plan";
  pith_attn_bwd_args all;
  int64_t tiles;
  if (!plan || !merged_call(args, chunks, n, &all, &tiles)) return fail(PITH_ERR_BAD_SHAPE, "%s: plan is NULL or bad shape", who);
  if (n == 1) {
    all.Skv = chunks[0].rows;
    all.causal = 1;
    return pith_attn_bwd_plan(&all, plan);
  }
  all.dq_dtype = all.dkv_dtype = PITH_BF16;
  plan->dkdv_rows = kBN;
  plan->dkdv_split = pick_chunks_split(all, tiles);
  plan->dq_ds_pairs = pith_attn_bwd_chunks_ds_bytes(args, chunks, n) > 0 && dq_ds_pairs(dq_ds_workgroups(args));
  plan->one_grid = chunk_grids(&all, tiles, plan->dkdv_split, tiles * all.Hkv * all.B * plan->dkdv_split).one;
  return PITH_OK;
}

extern "C" int64_t pith_attn_bwd_chunks_workspace_bytes(const pith_attn_bwd_args* args, const pith_key_chunk* chunks, int64_t n) {
  pith_attn_bwd_args a;
  int64_t tiles;
  if (!merged_call(args, chunks, n, &a, &tiles)) return 0;
  if (n == 1) {  // goes out as pith_attn_bwd, whose head split is another one (with less than it asks for there is none: 1 x 3200 x 32/4 399 -> 617 us)
    a.causal = 1;
    return pith_attn_bwd_dkdv_workspace_bytes(&a);
  }
  return workspace_bytes_for(&a, pick_chunks_split(a, tiles));
}

extern "C" int64_t pith_attn_bwd_chunks_ds_bytes(const pith_attn_bwd_args* args, const pith_key_chunk* chunks, int64_t n) {
  pith_attn_bwd_args a;
  int64_t tiles, bytes = 0;
  if (n < 2 || !merged_call(args, chunks, n, &a, &tiles) || a.Dqk != 192 || a.Dv != 128 || a.Sq <= dq_ds_rows(192) / 2) return 0;
  for (int64_t i = 0; i < n; ++i) {
    if (chunks[i].q_row0 % 64) return 0;  // a 64-row tile that sees the chunk in part would lie across two of its images
    bytes += a.B * a.Hq * chunk_ds_head_bytes(a.Sq, chunks[i], i == n - 1);
  }
  return bytes;
}

namespace {

int run_bwd_chunks(const pith_attn_bwd_args* args, const pith_key_chunk* chunks, int64_t n, void* ds, int64_t ds_bytes, pith_stream_t stream, const char* who) {
  if (!args || !chunks) return fail(PITH_ERR_NULL_POINTER, "%s: args or chunks is NULL", who);
  pith_attn_bwd_args all;
  int64_t tiles;
  if (!merged_call(args, chunks, n, &all, &tiles))
    return fail(PITH_ERR_BAD_SHAPE, "%s: 1..%d chunks, each of 1..2^24 rows and seen from a query row on, and Hq a multiple of Hkv", who, kMaxChunks);
  if (args->dq_dtype != PITH_BF16 || args->dkv_dtype != PITH_BF16 || args->accumulate_dq || args->accumulate_dkv || args->dq_final)
    return fail(PITH_ERR_UNSUPPORTED, "%s: gradients are written, once, in bf16", who);
  if (n == 1) {
    pith_attn_bwd_args a = *args;
    const pith_key_chunk& c = chunks[0];
    a.k = c.k; a.v = c.v; a.k_pe = c.k_pe; a.dk = c.dk; a.dv = c.dv; a.dk_pe = c.dk_pe;
    a.Skv = c.rows; a.causal = 1; a.dkv_zero_tail = c.zero_tail; a.ds = nullptr;
    return pith_attn_bwd(&a, stream);
  }
  const int split = pick_chunks_split(all, tiles);
  const int64_t need = workspace_bytes_for(&all, split);
  if (need > 0 && (!args->workspace || args->workspace_bytes < need || !aligned16(args->workspace)))
    return fail(PITH_ERR_BAD_SHAPE, "%s: a 16-byte aligned workspace of %lld bytes is needed", who, (long long)need);
  const int64_t ds_need = pith_attn_bwd_chunks_ds_bytes(args, chunks, n);
  const bool hand_over = ds && ds_need > 0 && ds_bytes >= ds_need;
  if (hand_over && (uintptr_t)ds % 256) return fail(PITH_ERR_MISALIGNED, "%s: ds must be 256-byte aligned", who);
  BwdChunkParams p;
  unsigned blocks = 0;
  int64_t rows_before = 0, ds_off = 0;
  for (int64_t i = 0; i < n; ++i) {
    const pith_key_chunk& c = chunks[i];
    const bool diagonal = i == n - 1;
    if ((diagonal && c.q_row0) || (i > 0 && !diagonal && c.q_row0 < chunks[i - 1].q_row0))
      return fail(PITH_ERR_BAD_SHAPE, "%s: chunk %lld: q_row0=%lld (chunks sorted by it, the queries' own, 0, last)", who, (long long)i, (long long)c.q_row0);
    pith_attn_bwd_args a = *args;
    a.k = c.k; a.v = c.v; a.k_pe = c.k_pe; a.dk = c.dk; a.dv = c.dv; a.dk_pe = c.dk_pe;
    a.Skv = c.rows; a.causal = diagonal; a.dkv_zero_tail = c.zero_tail; a.ds = nullptr;
    if (!c.k_pe != !chunks[0].k_pe) return fail(PITH_ERR_UNSUPPORTED, "%s: keys in two parts in some chunks only", who);
    if (const int rc = validate_bwd(&a, who, true, true)) return rc;
    if (const int rc = validate_dk_pe(&a, who)) return rc;
    if (i == 0) static_cast<BwdParams&>(p) = make_bwd_params(&a);
    BwdChunk& ch = p.chunk[i];
    ch.key = KeyChunk{(const __bf16*)c.k, (const __bf16*)c.v, (const __bf16*)c.k_pe, (int)c.rows, (int)c.q_row0};
    ch.dk = (__bf16*)c.dk; ch.dv = (__bf16*)c.dv; ch.dk_pe = (__bf16*)c.dk_pe;
    ch.tiles = (int)((c.rows + kBN - 1) / kBN);
    ch.zero_tail = (int)c.zero_tail;
    ch.first_block = (int)blocks;
    ch.rows_before = (int)rows_before;
    ch.ds_off = ds_off;
    ch.ds_hs = chunk_ds_head_bytes(a.Sq, c, diagonal);
    ch.ds_kb = ch.tiles;
    ds_off += a.B * a.Hq * ch.ds_hs;
    const int64_t next = blocks + (int64_t)ch.tiles * a.Hkv * a.B * split + (c.zero_tail + kZeroTailRows - 1) / kZeroTailRows;
    rows_before += c.rows;
    if (next > 0x3fffffff || rows_before > 0x3fffffff) return fail(PITH_ERR_UNSUPPORTED, "%s: the chunks exceed the launch grid limit", who);
    blocks = (unsigned)next;
  }
  p.n_chunks = (int)n;
  p.chunked = kChunkedTiles;  // (rows unequal, as under the mask)
  p.through_dkv = through_results(rows_before * all.B * all.Hkv * (all.Dqk + all.Dv) * 2);
  p.dk_pe_bs = args->dk_pe_bs;
  p.split = split;
  const int dq_rows = hand_over ? dq_ds_rows(192) : 128;
  p.q_tiles = (p.Sq + dq_rows - 1) / dq_rows;
  if (hand_over) p.ds = reinterpret_cast<char*>(ds);
  p.ws_dk = reinterpret_cast<float*>(need > 0 ? args->workspace : nullptr);
  p.ws_dv = p.ws_dk + (split > 1 ? (int64_t)split * all.B * all.Skv * all.Hkv * all.Dqk : 0);
  p.ws_dkpe = reinterpret_cast<float*>(reinterpret_cast<char*>(p.ws_dk) + split_bytes_for(&all, split));
  p.through_parts = through_results(need);
  hipStream_t st = (hipStream_t)stream;
  begin_launch();
  const ChunkGrids grids = chunk_grids(&all, tiles, split, blocks);
  launch_bwd_chunks(p, (int)all.Dqk, grids.one, grids.dq_first, blocks, st);
  if (all.k_pe || split > 1) {  // (never both: keys in two parts have no head groups to split)
    Reduction<2 * kMaxChunks> r;
    for (int64_t i = 0; i < n; ++i) {
      const pith_key_chunk& c = chunks[i];
      const int64_t at = p.chunk[i].rows_before * all.B * all.Hkv;
      if (all.k_pe) {
        r.add(p.ws_dkpe + at * 64, c.dk_pe, args->dk_pe_bs, all.B, c.rows, 64, 64);
      } else {
        r.add(p.ws_dk + at * split * all.Dqk, c.dk, args->dk_bs, all.B, c.rows, all.Hkv * all.Dqk, p.HkvT * all.Dqk);
        r.add(p.ws_dv + at * split * all.Dv, c.dv, args->dv_bs, all.B, c.rows, all.Hkv * all.Dv, p.HkvT * all.Dv);
      }
    }
    r.launch(all.k_pe ? (int)all.Hkv : split, false, false, st);
  }
  return check_launch(who);
}

}  // namespace

extern "C" int pith_attn_bwd_chunks(const pith_attn_bwd_args* args, const pith_key_chunk* chunks, int64_t n, pith_stream_t stream) {
  return run_bwd_chunks(args, chunks, n, nullptr, 0, stream, "pith_attn_bwd_chunks");
}

extern "C" int pith_attn_bwd_chunks_handover(const pith_attn_bwd_args* args, const pith_key_chunk* chunks, int64_t n, void* ds, int64_t ds_bytes,
                                             pith_stream_t stream) {
  return run_bwd_chunks(args, chunks, n, ds, ds_bytes, stream, "pith_attn_bwd_chunks_handover");
}
