// Entry point of the chunk attention forward for gfx950: O = softmax(scale * Q K^T [+causal]) V, base-2 LSE, argument
// checks and the choice of a kernel. Numerics of all kernels follow pithtrain/operators/mla/triton.py:32-93 (causal) and
// :274-323 (non-causal): fp32 scores from bf16 MFMA, P = exp2(kappa*(s - m)) in fp32, row sum from the fp32 P, P rounded
// to bf16 for P V, O = acc / l rounded to bf16, LSE2 = log2(l) + kappa*m, kappa = scale*log2(e).
// One deviation in rounding only: the running maximum m is refreshed (and O, l rescaled) only when a row's P values
// would exceed 2^8; P, l and O stay consistent with whichever m is in force, so O and LSE2 are the same function of the
// inputs.
#include "attn_fwd_common.h"

namespace pith {
namespace {

// Work splits (attn_fwd_direct.hip, attn_fwd_duo.hip):
//   FULL   one 256-row workgroup of 8 waves per compute unit: the fewest K/V tile requests per product;
//   DUO    two 128-row workgroups of 4 waves per compute unit: twice the requests, but one's prologue, epilogue and last
//          tiles overlap the other's loop, and the diagonal wastes half as much;
//   HALF   one 128-row workgroup of 8 waves per compute unit, wave pairs splitting the keys of every tile;
//   TEAMS  one 128-row workgroup of 8 waves per compute unit, two teams of 4 waves taking every second tile (64 features);
//   QUARTER  one 64-row workgroup of 8 waves: two teams, and wave pairs of a team splitting the keys of its tile.
// FULL and DUO when every compute unit has work for its whole time; the others when workgroups are few or (under the mask)
// so unequal that a heavy one would run alone on its unit. Kernels measured on one box, microseconds, with inputs that
// rotate over 500 MB (the tiles come from memory, as in a training step; the prefetch depth counts then: TEAMS at 192
// features, two tiles per ring, beat HALF by 2-8 % on inputs in the last-level cache and lost 4-9 % here)
// (QUARTER before its teams took turns on streams of 1024 keys and more, 3-17 % faster since: kHalvesFrom in attn_fwd_duo.hip):
//                                                       FULL    DUO   HALF  TEAMS QUARTER
//   d128 causal   1 x 16384 x 8 heads (cached)           454    470    507    515    643
//                 3 x 1999 x 32 (cached)                 109    107    133    131    187
//                 1 x 4096 x 8  (256 WGs of 128 rows)   82.1   76.6   61.4   68.2   64.2
//                 1 x 4096 x 6  (192 WGs)               79.5   71.1   57.0   64.5   50.9
//                 1 x 8192 x 4  (256 WGs)                150    137    109    123    108
//                 1 x 2048 x 8  (128 WGs)               43.4   37.8   30.5   33.7   26.4
//                 1 x 384 x 8 / 320 x 8 (cached)               11.2 / 9.5           10.9 / 10.3
//   d192 causal   1 x 8192 x 16 (1024 WGs, cached)              298    339    331    430
//                 1 x 4096 x 16 (512 WGs)                       112    100    110    152
//                 1 x 4096 x 8  (256 WGs)                      85.6   74.2   84.2   78.2
//                 1 x 1021 x 16 (128 WGs)                      27.3   25.9   28.8   24.0
//   d64  causal   1 x 4096 x 20 (640 WGs, cached)              62.4          69.7   78.0
//                 1 x 4096 x 16 (512 WGs)                      57.2          52.9   65.0
//                 2 x 2048 x 16 (512 WGs)                      32.0          32.4   44.4
//                 1 x 4096 x 8  (256 WGs)                      52.4          42.7   43.6
//                 1 x 1024 x 16 (128 WGs)                      16.4          15.2   11.8
//        full     1 x 2048 x 16 (256 WGs)                      30.3          27.4   39.9
//   ring shares, 4 ranks, zigzag: d192 4096 rows x 16 rank 0 / 3    416 / 323   367 / 342   385 / 330   530 / 460
//                                      2048 rows x 16 rank 0 / 2    180 / 136   142 / 113   149 / 117   130 / 121
//                                 d128 4096 rows x 8/2 rank 0       281         218         239         195
// No FULL at 192 features: its register budget left no room for the row-sum test of the running maximum. Such a kernel, ms,
// against DUO, tiles from memory; the two are within what one machine differs from the next (32768 x 128 on three of them:
// 36.0 / 36.4, 35.6 / 35.2, 35.7 / 37.4), and shorter streams are DUO's:
//   causal   32768 x 128 heads 36.0 / 36.4   x 120 33.9 / 33.3   x 64 18.1 / 17.9   x 16 4.58 / 4.53   16384 x 64  4.67 / 4.59
//            8192 x 128        2.59 / 2.39   x 16  0.345 / 0.298                    4096 x 128 0.692 / 0.663
//   full     32768 x 16        8.89 / 8.96   16384 x 64 8.91 / 9.05   8192 x 128 4.87 / 4.58   x 16 0.565 / 0.567   4096 x 128 1.24 / 1.17
enum class Split { kFull, kDuo, kHalf, kTeams, kQuarter };

// `mean` = mean length of the rows' key streams in percent of the longest (a masked chunk: 50).
Split pick_split(const pith_attn_fwd_args* a, int mean) {
  const int64_t cus = compute_units_or_default();
  const int64_t wgs = ((a->Sq + 127) / 128) * a->Hq * a->B, wgs64 = ((a->Sq + 63) / 64) * a->Hq * a->B;  // of 128 and 64 rows
  const bool d64 = a->Dqk == 64, unequal = mean <= 70;  // HALF is 3 % slower than DUO at 0.75, 5-10 % above
  // few rows: below 6 tiles (64 features: 5) the merge costs more than the shorter streams save
  if (wgs64 <= cus && a->Skv > (d64 ? 256 : 320)) return Split::kQuarter;
  // more 64-row workgroups than compute units: heavy ones first, then light ones, as long as the streams are long. HALF / QUARTER, causal,
  // us, inputs from memory, rounds of 64-row workgroups: 192 features, 1.1 1024 x 18 21.7 / 17.5, 1536 x 12 28.6 / 21.1; 1.5 1024 x 24 23.5 / 23.0, 1536 x
  // 16 31.0 / 27.0; 1.75-2 1536 x 20 32.2 / 32.5, 2048 x 14 38.8 / 36.1, x 16 40.6 / 39.7, 3072 x 10 54.2 / 49.4, 4096 x 7 69.0 / 58.8, x 8 71.2 /
  // 64.0; 128, 1.1 1024 x 18 18.0 / 16.1, 1536 x 12 23.4 / 19.5; 1.5 1024 x 24 18.2 / 19.3, 1536 x 16 23.6 / 22.4; 1.75-2 1536 x 20 26.8 / 28.3, 2048 x 14
  // 31.0 / 30.6, x 16 33.7 / 34.6, 3072 x 10 43.8 / 40.7, 4096 x 7 53.6 / 46.9, x 8 57.8 / 53.6. Without a mask HALF, 1024 x 2048 x 32 45.8 / 62.0 and 37.6 / 52.9.
  if (!d64 && unequal && wgs64 <= 2 * cus && a->Skv >= (4 * wgs64 <= 5 * cus ? 1024 : 2 * wgs64 <= 3 * cus ? 1536 : a->Dqk == 192 ? 2048 : 3072)) return Split::kQuarter;
  const Split key_split = d64 ? Split::kTeams : Split::kHalf;
  if (wgs <= cus && a->Skv > (d64 ? 1024 : 512)) return key_split;
  if (unequal && wgs <= 2 * cus && a->Skv > (d64 ? 2048 : 1535)) return key_split;
  // FULL under the mask also for shorter rows of many heads whose K and V outgrow the last-level cache (half the streams in
  // flight; 2048 x 256 heads 355 -> 314 us, 2048 x 224 293 -> 276, 1024 x 512 221 -> 207, 2048 x 192 (192 MiB) 231 -> 235; not
  // for rows of a few workgroups: 8 x 512 x 128 155 -> 167)
  const bool many_heads = a->Sq >= 1024 && a->Skv == a->Sq && a->B * a->Skv * a->Hkv * (a->Dqk + a->Dv) * 2 >= 224ll << 20;
  if (a->Dqk == 128 && (unequal ? (a->Sq >= 3072 || many_heads) && wgs > 2 * cus : a->Skv > 1024 && wgs > cus)) return Split::kFull;
  return Split::kDuo;
}

}  // namespace
}  // namespace pith

using namespace pith;

namespace {

// Argument checks and everything the kernels' parameters take from the arguments.
int prepare(const pith_attn_fwd_args* a, FwdParams& p) {
  if (!a) return fail(PITH_ERR_NULL_POINTER, "pith_attn_fwd: args is NULL");
  if (!a->q || !a->k || !a->v || !a->lse || (!a->o && !(a->prev_o && a->acc_o)))
    return fail(PITH_ERR_NULL_POINTER, "pith_attn_fwd: NULL tensor pointer");
  if (a->B <= 0 || a->Sq <= 0 || a->Skv <= 0 || a->Hq <= 0 || a->Hkv <= 0)
    return fail(PITH_ERR_BAD_SHAPE, "pith_attn_fwd: B=%lld Sq=%lld Skv=%lld Hq=%lld Hkv=%lld must all be positive",
                (long long)a->B, (long long)a->Sq, (long long)a->Skv, (long long)a->Hq, (long long)a->Hkv);
  if (a->Hq % a->Hkv != 0)
    return fail(PITH_ERR_BAD_SHAPE, "pith_attn_fwd: Hq=%lld is not a multiple of Hkv=%lld", (long long)a->Hq,
                (long long)a->Hkv);
  if (!(a->scale > 0.f) || !(a->scale < INFINITY))
    return fail(PITH_ERR_BAD_SHAPE, "pith_attn_fwd: scale=%g must be positive and finite", (double)a->scale);
  if (a->causal && a->Sq != a->Skv)
    return fail(PITH_ERR_UNSUPPORTED, "pith_attn_fwd: causal needs Sq == Skv (got %lld, %lld)", (long long)a->Sq,
                (long long)a->Skv);
  if (a->Sq > (1 << 24) || a->Skv > (1 << 24) || a->Hq > 65535 || a->B > 65535 ||
      ((a->Sq + 63) / 64) * a->Hq * a->B > 0x7fffffffLL)
    return fail(PITH_ERR_UNSUPPORTED, "pith_attn_fwd: sequence, head or batch count beyond the launch grid limits");
  if (!aligned16(a->q) || !aligned16(a->k) || !aligned16(a->v) || !aligned16(a->o) || a->q_bs % 8 || a->k_bs % 8 ||
      a->v_bs % 8 || a->o_bs % 8)
    return fail(PITH_ERR_MISALIGNED, "pith_attn_fwd: tensor pointers / batch strides must keep 16-byte alignment");

  p.q = (const __bf16*)a->q; p.k = (const __bf16*)a->k; p.v = (const __bf16*)a->v;
  p.o = (__bf16*)a->o; p.lse = a->lse;
  p.Sq = (int)a->Sq; p.Skv = (int)a->Skv; p.Hq = (int)a->Hq; p.Hkv = (int)a->Hkv; p.group = (int)(a->Hq / a->Hkv);
  p.B = (int)a->B; p.m_tiles = 0; p.through_o = through_results(a->B * a->Sq * a->Hq * a->Dv * 2); p.chunked = kChunkedTiles;
  p.q_bs = a->q_bs; p.k_bs = a->k_bs; p.v_bs = a->v_bs; p.o_bs = a->o_bs; p.lse_bs = a->lse_bs; p.lse_hs = a->lse_hs;
  p.kappa = a->scale * 1.44269504088896340736f;
  p.k_pe = (const __bf16*)a->k_pe; p.k_pe_bs = a->k_pe_bs; p.k_pe_rs = a->k_pe_rs;
  if (a->k_pe) {
    if (a->Dqk != 192 || a->Dv != 128)
      return fail(PITH_ERR_UNSUPPORTED, "pith_attn_fwd: keys in two parts (k_pe) need head dims (192, 128), got (%lld, %lld)",
                  (long long)a->Dqk, (long long)a->Dv);
    if (!aligned16(a->k_pe) || a->k_pe_bs % 8 || a->k_pe_rs % 8 || a->k_pe_rs < 64)
      return fail(PITH_ERR_MISALIGNED, "pith_attn_fwd: k_pe pointer / strides must keep 16-byte alignment (row stride >= 64)");
  }
  p.prev_o = a->prev_o; p.prev_f32 = a->prev_o_dtype == PITH_F32; p.prev_bs = a->prev_o_bs;
  p.acc_o = a->prev_o ? a->acc_o : nullptr; p.acc_bs = a->acc_o_bs;
  p.o_r0 = p.o_r1 = p.acc_r0 = p.acc_r1 = 0;
  if (a->prev_o) {
    if (a->prev_o_dtype != PITH_BF16 && a->prev_o_dtype != PITH_F32)
      return fail(PITH_ERR_BAD_DTYPE, "pith_attn_fwd: prev_o_dtype %d is not bf16/fp32", a->prev_o_dtype);
    if (a->causal || a->Dv != 128 || (a->Dqk != 128 && a->Dqk != 192))
      return fail(PITH_ERR_UNSUPPORTED, "pith_attn_fwd: merging with a running result needs a non-causal call with head dims "
                  "(128,128) or (192,128); run pith_attn_fwd and pith_combine instead");
    if (!aligned16(a->prev_o) || a->prev_o_bs % 8 || (a->acc_o && (!aligned16(a->acc_o) || a->acc_o_bs % 8)))
      return fail(PITH_ERR_MISALIGNED, "pith_attn_fwd: prev_o / acc_o pointers and batch strides must keep 16-byte alignment");
    const int64_t* ranges[2] = {a->o_rows, a->acc_o_rows};
    int* dst[2][2] = {{&p.o_r0, &p.o_r1}, {&p.acc_r0, &p.acc_r1}};
    for (int i = 0; i < 2; ++i) {
      int64_t r0 = ranges[i][0], r1 = ranges[i][1];
      if (r0 == 0 && r1 == 0) r1 = a->Sq;
      if (r0 < 0 || r1 < r0 || r1 > a->Sq || r0 % 32 || (r1 % 32 && r1 != a->Sq))
        return fail(PITH_ERR_BAD_SHAPE, "pith_attn_fwd: %s = [%lld, %lld) must lie within the %lld query rows on multiples of 32",
                    i ? "acc_o_rows" : "o_rows", (long long)ranges[i][0], (long long)ranges[i][1], (long long)a->Sq);
      *dst[i][0] = (int)r0;
      *dst[i][1] = (int)r1;
    }
  }
  const bool dims_ok = (a->Dqk == 64 && a->Dv == 64) || ((a->Dqk == 128 || a->Dqk == 192) && a->Dv == 128);
  if (!dims_ok)
    return fail(PITH_ERR_UNSUPPORTED, "pith_attn_fwd: head dims (Dqk=%lld, Dv=%lld) not in {(64,64),(128,128),(192,128)}",
                (long long)a->Dqk, (long long)a->Dv);
  return PITH_OK;
}

template <typename P>
int launch(const P& p, const pith_attn_fwd_args* a, Split split, pith_stream_t stream, const char* who) {
  hipStream_t st = (hipStream_t)stream;
  begin_launch();
  const int dqk = (int)a->Dqk;
  const bool causal = a->causal != 0;
  if (split == Split::kFull || split == Split::kHalf) launch_fwd_direct(p, dqk, causal, split == Split::kHalf, st);
  else launch_fwd_duo(p, dqk, split == Split::kDuo ? 1 : split == Split::kTeams ? 2 : 4, causal, st);
  return check_launch(who);
}

}  // namespace

extern "C" int pith_attn_fwd(const pith_attn_fwd_args* a, pith_stream_t stream) {
  FwdParams p;
  if (const int rc = prepare(a, p)) return rc;
  return launch(p, a, pick_split(a, a->causal ? 50 : 100), stream, "pith_attn_fwd");
}

extern "C" int pith_attn_fwd_chunks(const pith_attn_fwd_args* args, const pith_key_chunk* chunks, int64_t n, pith_stream_t stream) {
  const char* who = "pith_attn_fwd_chunks";
  if (!args || !chunks) return fail(PITH_ERR_NULL_POINTER, "%s: args or chunks is NULL", who);
  if (n < 1 || n > kMaxChunks) return fail(PITH_ERR_BAD_SHAPE, "%s: %lld chunks, not 1..%d", who, (long long)n, kMaxChunks);
  if (args->prev_o) return fail(PITH_ERR_UNSUPPORTED, "%s: no merging with a running result", who);
  pith_attn_fwd_args a = *args;
  FwdChunkParams p;
  int64_t keys = 0, seen = 0;  // in the chunks; (query row, key) pairs
  for (int64_t i = 0; i < n; ++i) {
    const pith_key_chunk& c = chunks[i];
    const bool diagonal = i == n - 1;
    if (c.q_row0 < 0 || c.q_row0 >= args->Sq || (diagonal && c.q_row0) || (i > 0 && !diagonal && c.q_row0 < chunks[i - 1].q_row0))
      return fail(PITH_ERR_BAD_SHAPE, "%s: chunk %lld: q_row0=%lld (chunks sorted by it, the queries' own, 0, last)", who, (long long)i, (long long)c.q_row0);
    a.k = c.k; a.v = c.v; a.k_pe = c.k_pe; a.Skv = c.rows; a.causal = diagonal;
    if (!c.k_pe != !chunks[0].k_pe) return fail(PITH_ERR_UNSUPPORTED, "%s: keys in two parts in some chunks only", who);
    if (const int rc = prepare(&a, p)) return rc;
    p.chunk[i] = KeyChunk{(const __bf16*)c.k, (const __bf16*)c.v, (const __bf16*)c.k_pe, (int)c.rows, (int)c.q_row0};
    keys += c.rows;
    seen += diagonal ? c.rows * args->Sq / 2 : c.rows * (args->Sq - c.q_row0);
  }
  p.n_chunks = (int)n;
  // The split goes by the whole stream and by how unequal the rows' streams are.
  a.Skv = keys;
  const Split split = pick_split(&a, (int)(100 * seen / (keys * args->Sq)));
  a.causal = 1;
  if (n == 1) return launch<FwdParams>(p, &a, split, stream, who);
  return launch(p, &a, split, stream, who);
}
