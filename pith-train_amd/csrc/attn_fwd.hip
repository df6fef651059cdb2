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
//   QUARTER  one 64-row workgroup of 8 waves: two teams, and wave pairs of a team splitting the keys of its tile;
//   SMALL  two (64 features: four) 64-row workgroups of 4 waves, wave pairs splitting the keys of every tile: an interval of half the length, and
//          more workgroups than any other split that hide each other's first tiles and epilogues.
// FULL and DUO when every compute unit has work for its whole time; the others when workgroups are few or (under the mask)
// so unequal that a heavy one would run alone on its unit. Kernels measured on one box, microseconds, with inputs that
// rotate over 500 MB (the tiles come from memory, as in a training step; the prefetch depth counts then: TEAMS at 192
// features, two tiles per ring, beat HALF by 2-8 % on inputs in the last-level cache and lost 4-9 % here)
//                                                       FULL    DUO   HALF  TEAMS QUARTER  SMALL
//   d128 causal   1 x 16384 x 8 heads                    451    461    494            597    544
//                 3 x 1999 x 32                          108    106    126            187    130
//                 1 x 4096 x 8  (256 WGs of 128 rows)   83.6   76.9   57.4           52.6   60.0
//                 1 x 4096 x 6  (192 WGs)               82.0   74.5   55.1           42.9   57.2
//                 1 x 8192 x 4  (256 WGs)                159    147    106           88.7    113
//                 1 x 2048 x 8  (128 WGs)               44.2   39.1   30.7           25.0   30.0
//   d192 causal   1 x 8192 x 16 (1024 WGs)                      291    333            380    344
//                 1 x 4096 x 16 (512 WGs)                       103   90.9            112   94.1
//                 1 x 4096 x 8  (256 WGs)                      89.0   74.7           59.8   70.6
//                 1 x 1021 x 16 (128 WGs)                      26.1   23.1           19.7   20.7
//   d64  causal   1 x 4096 x 20 (640 WGs)                      63.8          74.4    84.1   56.2
//                 1 x 4096 x 16 (512 WGs)                      60.5          54.9    68.9   49.5
//                 2 x 2048 x 16 (512 WGs)                      33.7          32.8    42.1   27.5
//                 1 x 4096 x 8  (256 WGs)                      55.4          44.8    37.7   44.0
//                 1 x 1024 x 16 (128 WGs)                      16.8          15.0    11.9   13.8
//        full     1 x 2048 x 16 (256 WGs)                      32.0          27.9    35.6   27.6
//   ring shares, 4 ranks, zigzag: d192 4096 rows x 16 rank 0 / 3    371 / 313   323 / 322           442 / 393   368 / 363
//                                      2048 rows x 16 rank 0 / 2    180 / 142   142 / 114           126 / 112   149 / 112
//                                 d128 4096 rows x 8/2 rank 0       299         216                 175         222
// No FULL at 192 features: its register budget left no room for the row-sum test of the running maximum. Such a kernel, ms,
// against DUO, tiles from memory; the two are within what one machine differs from the next (32768 x 128 on three of them:
// 36.0 / 36.4, 35.6 / 35.2, 35.7 / 37.4), and shorter streams are DUO's:
//   causal   32768 x 128 heads 36.0 / 36.4   x 120 33.9 / 33.3   x 64 18.1 / 17.9   x 16 4.58 / 4.53   16384 x 64  4.67 / 4.59
//            8192 x 128        2.59 / 2.39   x 16  0.345 / 0.298                    4096 x 128 0.692 / 0.663
//   full     32768 x 16        8.89 / 8.96   16384 x 64 8.91 / 9.05   8192 x 128 4.87 / 4.58   x 16 0.565 / 0.567   4096 x 128 1.24 / 1.17
// Where workgroups are few, by W = 64-row workgroups per compute unit, us, DUO / HALF (64 features: TEAMS) / QUARTER / SMALL, inputs from memory:
//   d64 causal   W 1         2 x 256 x 32 7.3 / 7.6 / 6.7 / 6.2, 1024 x 16 15.9 / 14.1 / 10.8 / 12.1, 4096 x 4 50.4 / 39.8 / 27.3 / 35.4
//                W 2         4 x 256 x 32 7.6 / 7.9 / 9.8 / 6.4, 1024 x 32 16.4 / 14.5 / 13.8 / 12.5, 2048 x 16 27.6 / 23.0 / 19.7 / 20.6,
//                            4096 x 8 50.4 / 40.0 / 31.1 / 36.9
//                W 3 - 4     8 x 256 x 24 7.7 / 12.9 / 13.1 / 7.2, 2 x 1024 x 32 17.7 / 19.9 / 24.7 / 14.9, 2048 x 24 28.7 / 24.2 / 29.0 / 22.6,
//                            2048 x 32 30.1 / 28.6 / 35.3 / 25.1, 2 x 2048 x 16 30.1 / 28.6 / 35.1 / 25.0, 4096 x 16 55.9 / 47.8 / 57.8 / 47.1
//                W 4.1 - 6   3 x 1346 x 16 22.4 / 28.2 / 31.3 / 19.0, 3 x 1596 x 16 26.5 / 34.1 / 36.6 / 25.5, 4404 x 16 61.8 / 60.8 / 68.2 / 52.2,
//                            4 x 1024 x 20 18.5 / 27.3 / 30.4 / 20.3, 2 x 2048 x 20 33.3 / 40.6 / 44.5 / 32.4, 12 x 512 x 16 14.4 / 23.4 / 28.2 / 15.9
//   d64 full     W 1         2 x 256 x 32 6.9 / 7.8 / 6.8 / 6.2, 1024 x 16 15.8 / 14.6 / 11.2 / 12.2
//                W 2         4 x 192 x 43 8.1 / 14.4 / 14.7 / 8.1, 1024 x 32 16.6 / 15.4 / 19.2 / 13.9, 2 x 512 x 32 10.3 / 10.3 / 13.3 / 9.1
//                W 3 - 4     2048 x 24 33.6 / 45.3 / 43.3 / 35.0
//   d128 causal  W 1         4 x 128 x 32 7.1 / 7.9 / 7.9 / 6.7, 2 x 256 x 32 9.0 / 9.1 / 9.0 / 8.1, 512 x 32 13.0 / 12.1 / 11.0 / 10.8,
//                            1024 x 16 20.9 / 17.7 / 15.3 / 16.2
//                W 1.1 - 1.5 1024 x 18 21.2 / 18.2 / 16.0 / 16.7, 1536 x 12 28.9 / 23.5 / 19.2 / 22.1, 2 x 512 x 24 13.3 / 12.4 / 16.0 / 11.3,
//                            1024 x 24 21.3 / 18.0 / 19.1 / 16.9, 1536 x 16 29.0 / 23.4 / 21.7 / 22.3
//                W 2         2 x 512 x 32 13.6 / 12.6 / 16.8 / 11.7, 1024 x 32 21.8 / 18.7 / 21.2 / 17.8, 2048 x 16 37.5 / 30.0 / 30.1 / 29.5,
//                            3072 x 10 53.6 / 42.0 / 39.0 / 42.1, 4096 x 8 69.4 / 53.2 / 47.1 / 53.4
//                W 2.5 - 3   8 x 256 x 20 10.1 / 15.1 / 20.5 / 13.2, 2 x 1024 x 20 23.2 / 19.9 / 29.8 / 19.1, 2 x 1024 x 24 23.6 / 22.6 / 31.6 / 22.7
//   d128 full    W 1         2 x 256 x 32 9.2 / 9.0 / 9.4 / 8.2, 512 x 32 13.4 / 11.8 / 11.6 / 10.9
//                W 2         4 x 256 x 32 10.5 / 10.1 / 17.3 / 10.3, 2 x 512 x 32 14.8 / 13.1 / 21.1 / 13.7, 1024 x 2048 x 32 40.8 / 35.4 / 47.1 / 37.9
//   d192 causal  W 1         2 x 256 x 32 10.5 / 10.4 / 10.2 / 9.2, 512 x 32 15.2 / 14.0 / 12.6 / 12.4, 1024 x 16 24.6 / 21.6 / 17.2 / 18.5
//                W 1.1 - 1.5 8 x 128 x 24 9.9 / 11.3 / 16.7 / 10.4, 2 x 512 x 24 16.7 / 16.1 / 19.4 / 15.2, 1024 x 24 25.8 / 23.6 / 23.2 / 22.2,
//                            1409 x 16 32.7 / 28.5 / 24.8 / 26.6
//                W 2         2 x 512 x 32 17.0 / 16.1 / 20.4 / 15.3, 2048 x 16 45.3 / 38.5 / 36.3 / 37.7, 4096 x 8 82.3 / 69.7 / 58.3 / 67.5
//                W 2.5 - 3   2 x 1024 x 20 27.5 / 24.4 / 35.6 / 24.6
//   d192 full    W 1         2 x 256 x 32 10.5 / 10.4 / 10.7 / 9.5, 512 x 32 15.3 / 13.9 / 13.3 / 12.9
//                W 2         4 x 256 x 32 12.8 / 14.4 / 21.2 / 14.0, 2 x 512 x 32 18.2 / 17.2 / 26.5 / 19.3, 1024 x 2048 x 32 50.5 / 44.6 / 60.5 / 54.9
// Zigzag shares above W 1.5 take QUARTER while the workgroups of their longer half are one round, HALF / QUARTER: 224 to 256 of them 896 x 32/4 of 128, eight ranks,
// rank 0 164 / 81, four 78 / 49, 960 x 32/4 rank 2 116 / 95, 2 x 1024 x 16/4 117 / 98, 3 x 1204 x 8/2 143 / 115, 960 x 32 of 192 194 / 138; 260 to 288 1022 x 32/4 rank
// 2 124 / 156, 1530 x 20/5 179 / 219, 3 x 1270 x 8/2 148 / 187, 1300 x 24/3 240 / 260, 1022 x 32 of 192 144 / 185.
// Where the other half is not short (mean 2/3) 128 and 192 features wait for 3072 keys from W 1.2 and for 6144 from W 1.3 on: 1024 x 20 of 192, two ranks, rank 1, 33.3 / 35.7, 1280 x
// 16/4 of 128 32.6 / 33.6; 678 x 32 of 192 rank 2 46 / 50, 3 x 2510 x 4 74 / 78, 4 x 1504 x 4/1 of 128 40.6 / 41.7, but W 1.25 1240 x 16 of 192 rank 2 70 / 58, W 1.5 3 x 2074 x 4
// 118 / 110, eight ranks, rank 4 1352 x 16 156 / 137. 64 features for 2048 from W 1.4, and above 1.5 for 1536 rows: 3 x 256 x 32/8 24.7 / 26.4, 3 x 552 x 16/4
// 26.8 / 29.0, 1280 x 24/6 27.8 / 29.1, 3 x 2152 x 4 39.9 / 37.3.
enum class Split { kFull, kDuo, kHalf, kTeams, kQuarter, kSmall };

// Calls against one chunk a little above a whole round of 128-row workgroups, W of them per compute unit (a ragged length is enough): the
// last round of FULL, DUO or HALF would hold few of them, which a split with more or shorter ones spreads. us, by W:
//   causal d128  HALF / QUARTER   8448 x 4 (1.03) 100.6 / 91.6, 9000 x 4 (1.11) 115.7 / 106.3, 9984 x 4 (1.22) 124.6 / 128.6, 4224 x 8 (1.03) 53.9 / 54.0
//                FULL / HALF      4220 x 16 (2.06) 88.9 / 80.6, 4400 x 16 (2.19) 94.6 / 88.4, 4700 x 16 (2.31) 102.4 / 99.3, 5100 x 16 (2.5) 116.4 / 114.9,
//                                 8400 x 8 (2.06) 169.7 / 145.0, 16640 x 4 (2.03) 327.7 / 267.5, 10200 x 8 (2.5) 222.9 / 215.8, 20900 x 4 (2.56) 450.9 /
//                                 435.7, 12300 x 8 (3.03) 292.6 / 300.8; 2100 x 32 (2.12) DUO 46.4 / 49.1
//          d192  HALF / QUARTER   4224 x 8 (1.03) 71.4 / 62.3, 4600 x 8 (1.12) 78.2 / 74.1, 5000 x 8 (1.25) 86.1 / 85.4, 5400 x 8 (1.34) 93.9 / 95.8, 8448 x 4 (1.03)
//                                 134.0 / 108.6, 9984 x 4 (1.22) 165.4 / 152.7, 10700 x 4 (1.31) 179.0 / 171.1, 2112 x 16 (1.06) 37.9 / 40.5
//                HALF / SMALL     1100 x 32 (1.12) 24.7 / 23.5, 1250 x 32 (1.25) 27.8 / 27.1, 2300 x 16 (1.12) 42.6 / 41.2, 2560 x 16 (1.25) 47.7 / 46.9
//                DUO / HALF       4220 x 16 (2.06) 106.3 / 100.6, 4400 x 16 (2.19) 111.4 / 111.0, 8400 x 8 (2.06) 201.9 / 180.5, 8900 x 8 (2.19) 219.5 / 206.5,
//                                 16640 x 4 (2.03) 390.4 / 340.4, 18400 x 4 (2.25) 450.3 / 426.6, 9500 x 8 (2.34) 240.6 / 237.5, 2100 x 32 (2.12) 56.9 / 59.0
//          d64   TEAMS, to 6144 keys SMALL / QUARTER  4224 x 8 (1.03) 39.5 / 36.2, 4600 x 8 (1.12) 42.3 / 42.3, 8448 x 4 (1.03) 77.7 / 62.3, 9984 x 4 (1.22) 91.6 / 85.8,
//                                 10700 x 4 (1.31) 98.3 / 97.3, 2112 x 16 (1.06) 21.6 / 22.9
//                DUO / SMALL      8400 x 8 (2.06) 112.4 / 93.3, 10200 x 8 (2.5) 144.9 / 126.9, 20900 x 4 (2.56) 295.6 / 258.6, 3 x 8064 x 4 (2.95) 126.1 / 119.9,
//                                 12300 x 8 (3.03) 188.5 / 179.9, 6200 x 16 (3.06) 96.9 / 95.4
//   full   d128  FULL / HALF      2100 x 32 (2.12) 101.0 / 94.5, 2400 x 32 (2.38) 116.1 / 108.3, 2700 x 32 (2.75) 129.1 / 125.3, 3000 x 32 (3) 142.0 / 142.7, 4400 x
//                                 16 (2.19) 198.4 / 183.8, 5300 x 16 (2.62) 237.4 / 226.3, 17500 x 4 (2.14) 749.8 / 692.9; 2 x 1400 x 32 (2.75) DUO 70.3 / 72.3
bool above_a_round(const pith_attn_fwd_args* a, int64_t wgs, int64_t cus, Split* split) {
  const auto at_most = [&](int64_t n, int64_t d) { return d * wgs <= n * cus; };  // W <= n / d
  const int64_t keys = a->Skv;
  if (wgs <= cus) return false;
  if (!a->causal) {
    *split = Split::kHalf;
    return a->Dqk == 128 && wgs > 2 * cus && at_most(11, 4) && keys >= 2048;
  }
  if (keys != a->Sq) return false;  // several chunks
  if (a->Dqk == 64) {
    *split = wgs > 2 * cus ? Split::kSmall : Split::kQuarter;
    return wgs > 2 * cus ? at_most(25, 8) && keys > 6144 : (at_most(17, 16) && keys >= 4096) || (at_most(5, 4) && keys >= 8192);
  }
  const bool d192 = a->Dqk == 192;
  if (wgs > 2 * cus) {
    *split = Split::kHalf;
    return d192 ? (at_most(17, 8) && keys >= 4096) || (at_most(9, 4) && keys >= 8192) : at_most(5, 2) && keys >= 4096;
  }
  *split = d192 && keys < 2600 ? Split::kSmall : Split::kQuarter;
  if (*split == Split::kSmall) return at_most(5, 4) && keys >= 1024;
  return d192 ? (at_most(9, 8) && keys >= 4096) || (at_most(4, 3) && keys >= 8192) : at_most(23, 20) && keys >= 8192;
}

// More 64-row workgroups than units: where SMALL pays. By W = those workgroups per unit, us, SMALL / the best other:
//   64 features, rows unequal, two and more per unit
//     to 959 keys    SMALL is ahead while all of its workgroups run at once and 128 rows pad (192, 320 rows) or the tiles are many: W 3 512 x 96 heads
//                    10.6 / 11.9, 768 x 64 12.8 / 14.9; W 3.5-4 320 x 180 10.1 / 11.3, 600 x 90 13.1 / 14.1, 900 x 60 15.2 / 17.4, 768 x 84 14.3 / 16.1, 512 x 128
//                    12.2 / 12.6; but 256 rows W 3.3 x 210 10.7 / 9.4, 4 x 256 10.2 / 9.7, more than at once (4.2-4.5) 192 x 360 11.9 / 10.4, 370 x 192 15.4 /
//                    12.8, 768 x 96 17.6 / 16.7, and an odd number of heads, whose tiles wander over the XCDs, 448 x 135 14.2 / 13.4, 768 x 81 18.3 / 16.5
//     960 to 1535    W 4 1000 x 64 17.1 / 19.4, 1024 x 64 17.1 / 19.3, 4.25 1088 x 64 18.6 / 20.3, an odd number of heads 4.3 1024 x 69 22.9 / 21.2, 1200 x 58 21.9 / 22.6, 4.5 1400 x 52 23.4 / 25.7
//     1536 on        W 4.5 2 x 2048 x 18 31.9 / 35.9, 5 1 x 2048 x 40 35.2 / 36.2, but in several chunks with less unequal rows 2048 x 40/10 rank 2 118 / 111 (and 4.5 2 x 756 x 48/12, two
//                    ranks, rank 1 28.9 / 26.2; rank 0 2 x 582 x 64/16 56 / 71). With the backward behind it TEAMS is ahead from 2561 keys on while W is 3.25 at
//                    most: 4 x 2855 x 4 114.9 / 110.8, 2914 x 16 117.9 / 114.8, 2688 x 16 109.0 / 105.6, 5120 x 10 193.7 / 189.6, 6144 x 8 220.7 / 216.1, not 2560 x 20
//                    106.2 / 106.8, nor several chunks (1152 x 32/8, four ranks, rank 0 178 / 196), 4096 x 16 (W 4) equal, its forward alone 49.4 / 53.3
//   64 features without a mask, up to two per unit: to 384 keys from W 1.7 on (320 keys 1.35 9.1 / 8.6, 1.5 9.2 / 8.7, 1.75 9.6 / 10.2; 256 keys equal at best), 384 keys 44 to
//                    84 heads 8.7-9.6 / 9.0-9.9, but 75 heads 11.0 / 9.8; 1024 x 32 16.2 / 17.0; TEAMS above 2048 keys (2304 x 14 30.4 / 30.1, 6144 x 5 69.8 / 67.0)
//   128 and 192 features, rows unequal, up to two per unit: not for 128 rows, which one DUO workgroup holds (8.6 / 7.9, 9.2 / 8.9), nor up to 192 at W 1.05 (8.7 / 8.0
//                    and 9.9 / 9.2; 1.2: 8.1 / 8.4)
bool small_workgroups(const pith_attn_fwd_args* a, int64_t wgs64, int64_t cus, int mean) {
  const int64_t keys = a->Skv, heads = a->Hq * a->B;
  const bool unequal = mean <= 70, half = mean <= 52;  // half: one chunk, and rank 0 of a zigzag share
  const auto at_most = [&](int64_t n, int64_t d) { return d * wgs64 <= n * cus; };  // W <= n / d
  if (a->Dqk != 64) return unequal && at_most(2, 1) && keys >= 129 && keys < 1536 && (keys > 192 || !at_most(6, 5));
  if (!unequal) return at_most(2, 1) && keys >= 192 && keys <= 2048 && (keys >= 448 || (keys >= 384 ? heads % 4 == 0 : !at_most(17, 10)));
  if (at_most(2, 1)) return keys >= 128 && keys < 1536;
  if (keys < 128 || keys > 6144) return false;
  if (keys >= 1536) return (half ? at_most(5, 1) : at_most(9, 2)) && (keys <= 2560 || keys != a->Sq || !at_most(13, 4));
  if (keys >= 960) return half && (keys >= 1200 || heads % 2 == 0) ? at_most(9, 2) : at_most(4, 1);
  const bool pads = (a->Sq + 63) / 64 % 2 != 0;  // half of a 128-row workgroup
  return heads % 2 == 0 && (keys >= 384 || pads) ? at_most(4, 1) : at_most(3, 1);
}

// `mean` = mean length of the rows' key streams in percent of the longest (a masked chunk: 50).
Split pick_split(const pith_attn_fwd_args* a, int mean) {
  const int64_t cus = compute_units_or_default();
  const int64_t wgs = ((a->Sq + 127) / 128) * a->Hq * a->B, wgs64 = ((a->Sq + 63) / 64) * a->Hq * a->B;  // of 128 and 64 rows
  Split above;
  if (above_a_round(a, wgs, cus, &above) && wgs64 > 2 * cus) return above;
  const bool d64 = a->Dqk == 64, unequal = mean <= 70;  // HALF is 3 % slower than DUO at 0.75, 5-10 % above
  if (a->Skv > 64 && wgs64 <= cus) return a->Skv > (d64 ? 384 : 512) ? Split::kQuarter : Split::kSmall;
  if (unequal && wgs64 <= 2 * cus) {
    const bool quarter_more = 4 * wgs64 > 5 * cus, half_more = 2 * wgs64 > 3 * cus;  // workgroups than one round of QUARTER
    int64_t from = d64 ? 1536 : half_more ? (a->Dqk == 192 ? 2048 : 3072) : quarter_more ? (a->Dqk == 192 ? 1400 : 1536) : 1024;
    const bool one_chunk = a->Skv == a->Sq, both_long = mean > 64;  // (of several chunks: the half that sees less, too)
    if (both_long && d64 && 5 * wgs64 > 7 * cus) from = 2048;
    if (both_long && !d64 && 5 * wgs64 > 6 * cus) from = 10 * wgs64 > 13 * cus ? 6144 : 3072;
    // 64-row workgroups of the longer half of a zigzag share's rows; what a second round holds besides is short
    const int64_t longer = ((a->Sq + 63) / 64 - a->Sq / 2 / 64) * a->Hq * a->B;
    const bool second_round = (one_chunk || longer <= cus) && (a->Sq >= 1536 || !(one_chunk || (d64 && both_long)));
    if (a->Skv >= from && (!half_more || second_round)) return Split::kQuarter;
  }
  if (small_workgroups(a, wgs64, cus, mean)) return Split::kSmall;
  const Split key_split = d64 ? Split::kTeams : Split::kHalf;
  if (wgs <= cus && a->Skv > (d64 ? 1024 : a->Dqk == 192 ? 383 : 256)) return key_split;  // (128 features without a mask, 256 keys: 4 x 27 heads 11.7 / 12.4)
  // (mean 1/2: one chunk, and rank 0 of a zigzag share; short rows that are less unequal, DUO / HALF: rank 2 of four, 2 x 396 x 40/8 of 128 36.7 / 42.9)
  if (unequal && wgs <= 2 * cus && a->Skv > (d64 ? 2048 : 2 * wgs <= 3 * cus && mean <= 52 ? 1023 : 1535)) return key_split;
  // FULL under the mask also for shorter rows of many heads whose K and V outgrow the last-level cache (half the streams in
  // flight; 2048 x 256 heads 355 -> 314 us, 2048 x 224 293 -> 276, 1024 x 512 221 -> 207, 2048 x 192 (192 MiB) 231 -> 235; not
  // for rows of a few workgroups: 8 x 512 x 128 155 -> 167)
  const bool many_heads = a->Sq >= 1024 && a->Skv == a->Sq && a->B * a->Skv * a->Hkv * (a->Dqk + a->Dv) * 2 >= 224ll << 20;
  // Several chunks of unequal rows (zigzag) a little above two or four 128-row workgroups per unit, which are 1.15 (long rows against more than two chunks: 2.25)
  // of FULL at most, an odd number of them to a head: where the longer half of the rows begins within the middle one, and not at the end of one that then walks
  // as far. DUO / FULL, forward of four ranks unless others are named, by FULL workgroups per unit: 1.1 2100 x 32/4 161 / 153, rank 0 253 / 231, 2 x 2100 x 16/4 193 /
  // 173, rank 0 2176 x 32/4 264 / 239, 2200 x 32/8 173 / 164, 2200 x 32/4, eight ranks, 392 / 345, 1664 x 40/8 130 / 120, 1792 x 40/8 148 / 151; 2.25 2200 x 64/4 323
  // / 305, rank 0 2300 x 64/4 501 / 456, 4 x 2168 x 16/4 332 / 322. Even: 2944 x 24/3 221 / 212, but rank 0 2862 x 24/3 341 / 376, 1364 x 48/8 177 / 196,
  // 1920 x 40/8 155 / 178, 2 x 2944 x 24/3, two ranks, 262 / 284. Less than two chunks' keys: 1588 x 40/5, two ranks, 66.6 / 73.3. More workgroups: 2.25 with
  // short rows 2 x 1408 x 48/8 228 / 238, 2.5 2 x 1100 x 64/4 172 / 177. Nor where 256 rows waste a fifth (with the backward 2 x 1040 x 32/4 375 / 377, 1090
  // x 64/4, two ranks, 218 / 225) or every head has keys of its own (4 x 2100 x 16 1350 / 1374)
  const int64_t tiles256 = (a->Sq + 255) / 256, wgs256 = tiles256 * a->Hq * a->B;
  if (a->Dqk == 128 && a->causal && a->Skv >= 2 * a->Sq && unequal && a->Hq > a->Hkv && a->Sq >= 1024 && 25600 * tiles256 <= 117 * a->Sq && tiles256 % 2 == 1 &&
      ((wgs > 2 * cus && 20 * wgs256 <= 23 * cus) || (wgs > 4 * cus && 4 * wgs256 <= 9 * cus && a->Sq >= 2048 && a->Skv > 2 * a->Sq)))
    return Split::kFull;
  // (without a mask, FULL / DUO: 1100 x 32/4 30.0 / 28.4, 8 x 1100 x 16 104.3 / 97.4, 2 x 1400 x 32/4 73.2 / 70.3, 1500 x 32/4 39.7 / 40.0, 1999 x 32/4 60.9 /
  // 61.1, 3457 x 32/4 176 / 183)
  if (a->Dqk == 128 && (unequal ? (a->Sq >= 3072 || many_heads) && wgs > 2 * cus : a->Skv > (a->causal ? 1024 : 1408) && wgs > cus)) return Split::kFull;
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
  else launch_fwd_duo(p, dqk, split == Split::kDuo ? 1 : split == Split::kTeams ? 2 : split == Split::kSmall ? 3 : 4, causal, st);
  return check_launch(who);
}

// (query row, key) pairs of a chunk
int64_t pairs_seen(const pith_attn_fwd_args* a, const pith_key_chunk& c, bool diagonal) { return diagonal ? c.rows * a->Sq / 2 : c.rows * (a->Sq - c.q_row0); }

// Of several chunks: by the whole stream (a->Skv) and by how unequal the rows' streams are.
Split pick_chunks_split(const pith_attn_fwd_args* a, int64_t seen) { return pick_split(a, (int)(100 * seen / (a->Skv * a->Sq))); }

}  // namespace

extern "C" int pith_attn_fwd_split(const pith_attn_fwd_args* args, const pith_key_chunk* chunks, int64_t n, int32_t* split) {
  const char* who = "pith_attn_fwd_split";
  if (!args || !split) return fail(PITH_ERR_NULL_POINTER, "%s: %s is NULL", who, args ? "split" : "args");
  pith_attn_fwd_args a = *args;
  int64_t seen = 0;
  if (chunks) {
    if (n < 1 || n > kMaxChunks) return fail(PITH_ERR_BAD_SHAPE, "%s: %lld chunks, not 1..%d", who, (long long)n, kMaxChunks);
    a.Skv = 0;
    for (int64_t i = 0; i < n; ++i) {
      a.Skv += chunks[i].rows;
      seen += pairs_seen(&a, chunks[i], i == n - 1);
    }
    a.causal = 1;
  }
  if (a.B <= 0 || a.Sq <= 0 || a.Skv <= 0 || a.Hq <= 0 || a.Hkv <= 0) return fail(PITH_ERR_BAD_SHAPE, "%s: bad shape", who);
  *split = (int32_t)(chunks ? pick_chunks_split(&a, seen) : pick_split(&a, a.causal ? 50 : 100));
  return PITH_OK;
}

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
    seen += pairs_seen(args, c, diagonal);
  }
  p.n_chunks = (int)n;
  a.Skv = keys;
  const Split split = pick_chunks_split(&a, seen);
  if (n == 1) return launch<FwdParams>(p, &a, split, stream, who);
  return launch(p, &a, split, stream, who);
}
