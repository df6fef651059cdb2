// Query-gradient kernel for head dims (128, 128) and (192, 128) on gfx950 that reads dS instead of recomputing it:
// dQ = scale * dS K (pithtrain/operators/mla/triton.py:205-266, the last product of the loop body),
// with dS = P*(dP - delta) taken, already rounded to bf16 and with its sign flipped, from the images
// that the dK/dV kernels of attn_bwd_dkdv_d128.h, attn_bwd_dkdv_wide.h and attn_bwd_dkdv_d192.h leave in p.ds (layout documented in the former). The two score products that the
// other dQ kernels repeat are gone; the price is one trip of dS through memory, so this kernel is
// bound by the rate at which it can stream the images, not by the matrix pipe.
//
// Work split (128 features; 192 below): a workgroup of 8 wavefronts owns 512 query rows of one (batch, head), a wave one 64-row query tile of the
// writer (under the mask in a grid of one round two blocks of 256 rows, see dq_ds_pairs). Keys are visited in steps of 32 (one
// wave pair of the writer). Per step the K tile (shared, packed and swizzled like everywhere else, 8 KB) and, per
// wave, the 4 KB image of its tile for that pair (copied verbatim) go global -> LDS directly. What
// bounds the kernel is how many bytes of dS each compute unit keeps in flight (a compute unit's
// vector cache holds about 64 outstanding 128-byte requests, i.e. ~8 KB per ~650 cycles of latency, so
// every unit must stay busy and spend its requests on dS), so the LDS goes to dS: K tiles live in a
// ring of 3 stages (they come from L2), the images in a ring of 4 stages of 32 KB. A wave's vector
// loads complete in issue order, so one wave cannot wait for a K tile requested two steps ago without
// also waiting for every image it requested before that tile; therefore waves 0..3 request the K
// tiles and nothing else, and waves 4..7 request the images of all eight waves (each its own and that
// of wave w - 4). Every wave waits for its own requests and the step's barrier publishes them.
// dQ += dS K: K fragments (B operands: 32 features x 16 keys) come from transposing reads of the K tile
// and serve both 32-row blocks of the wave's tile, dS fragments (A operands: 32 query rows x 16 keys)
// from transposing reads of the image, in the same key slot order. The accumulators therefore hold
// dQ untransposed (a lane owns one feature column of 16 rows) and the epilogue reads and writes whole
// 128-byte lines (store_rows32).
// The images are read once, by one workgroup: loaded non-temporally they leave the caches to K and to what the dK/dV launch wrote last.
// The kernel alone over 4096 x 32/4 heads, plain / non-temporal: under the mask 118 / 99
// us, without 196 / 169 (6.4 TB/s); with the dK/dV launch before it (the same rows) 436 / 422, 8192 x 32/4 1584 / 1559, 3 x 1999 x 32/4
// 363 / 348, 4 x 1024 x 32/4 152.5 / 151.6. So where all images fit the 256 MB last-level cache: backward of 16 heads of 192/128, 8 x 512 (40 MiB)
// 68.5 / 67.2, 3 x 1021 (54) 77.9 / 73.2, 4 x 1024 (72) 95.5 / 93.3, 2 x 2048 (136) 151 / 146. Past the vector cache only (sc1), or past more than that (sc0 nt, sc1 nt, sc0 sc1 nt): 0-3 %
// slower than nt.
// (192, 128): accumulators for 512 rows do not fit, so a workgroup owns 256 rows (under the mask in one round two blocks of 128), and
// two neighbouring waves share a 64-row tile, each with 96 of the features (either block's four waves lie on four SIMDs: with a tile's
// waves four apart the late block, alone for most of the longest walk, had two; 4096 x 16 causal 83 -> 72 us): a wave reads 2 + 3 KB of fragments per 6 products, and neither its images
// nor K are requested twice. K is 43 % of what a unit requests, so the images get the deeper ring: 7 stages of 16 KB beside 3 of 12.
// dQ from dS / the recomputing kernels, us (dK/dV with / without the stores): 4096 x 16 causal 72 / 130 (166 / 160), 8192 x 16 251 / 438
// (660 / 578), 4096 x 2048 x 16 68 / 114 (150 / 145), 4096 x 128 causal 570 / 936 (1468 / 1280).
// With its reads between the products (walk) and a request of a few scalar instructions (both were serial, without loads 0.26 and with products alone
// 0.55 of the 0.63 us of a step), the kernel alone on images from memory: 4096 x 16 causal 80 -> 72 us, 3072 x 16 57 -> 50, 4096 x 16 without a
// mask 116 -> 108, 8192 x 16 257 -> 246; backward of a share of 4096 x 16, 4 ranks, zigzag, ranks 0, 1, 3 959 / 945 / 915 -> 935 / 917 / 892. Rings of
// 4 + 7, 5 + 6 and 6 + 5 stages are equal to 3 + 7.
#include <type_traits>

#include "attn_bwd_common.h"
#include "attn_bwd_dkdv_d192.h"

namespace pith {
namespace {

constexpr int kThreads = 512;
constexpr int kBN = 32;      // keys per step
constexpr int kRingK = 3;    // K tiles: step s in use, s+1 and s+2 requested

// s_waitcnt with vmcnt = N, the other counters left at their maxima (gfx9 encoding: vmcnt in bits
// 3:0 and 15:14).
template <int N>
__device__ __forceinline__ void wait_vector_loads_but() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
// the same for a wave-uniform run-time count LO <= n <= HI, as a binary decision tree (a switch over
// the counts compiles to a chain of one compare and branch per case, a few hundred cycles per call)
template <int LO, int HI>
__device__ __forceinline__ void wait_vector_loads_but(int n) {
  if constexpr (LO == HI) {
    wait_vector_loads_but<LO>();
  } else {
    constexpr int MID = (LO + HI) / 2;
    if (n <= MID) wait_vector_loads_but<LO, MID>(n);
    else wait_vector_loads_but<MID + 1, HI>(n);
  }
}

// An image, 4 KB in a row on both sides (the instructions' offset counts on both), like load_lds16_once.
__device__ __forceinline__ void load_image_once(const char* base, int offset, char* dst_wave) {
  const uint32_t lds_addr = (uint32_t)(uintptr_t)(lds_char*)dst_wave;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024 nt\n\t"
               "global_load_lds_dwordx4 %1, %2 offset:2048 nt\n\tglobal_load_lds_dwordx4 %1, %2 offset:3072 nt"
               :
               : "s"(lds_addr), "v"(offset), "s"(base)
               : "memory");
}

// MULTI: over several chunks, whose steps are one stream; dQ is written once.
template <int DQK, bool CAUSAL, typename OutT, bool MULTI = false>
__global__ __launch_bounds__(kThreads) void attn_bwd_dq_ds_kernel(BwdArgs<MULTI> p) {
  constexpr int FS = DQK == 192 ? 2 : 1;    // waves that share 64 query rows, a part of the features each
  constexpr int RG = 8 / FS;                // 64-row groups of a workgroup
  constexpr int DB = DQK / 32 / FS;         // feature blocks per wave
  constexpr int QW = 64;                    // query rows per wave
  constexpr int RBW = QW / 32;              // 32-row blocks per wave
  constexpr int kBM = RG * QW;              // query rows per workgroup
  constexpr int kKStage = kBN * DQK * 2;                             // 8 KB, 12 KB
  constexpr int kDsWave = RBW * 2048;                                // per row group and step
  constexpr int kDsStage = RG * kDsWave;                             // 32 KB, 16 KB
  constexpr int kRingD = DQK == 192 ? 7 : 4;                         // images: step s in use, the next ones requested
  constexpr int kOffDs = kRingK * kKStage;
  constexpr int kLoadsDs = 2 * RBW;                                  // per image
  constexpr int kImages = RG / 4;                                    // per image-moving wave and step
  constexpr int kLoadsK = DQK / 64;                                  // per K-moving wave and step
  static_assert(kOffDs + kRingD * kDsStage <= 160 * 1024, "the rings must fit the LDS");
  __shared__ __attribute__((aligned(1024))) char smem[kOffDs + kRingD * kDsStage];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, g = lane >> 5;
  int m_tile, h, b;
  decode_block(blockIdx.x, p.Hq, p.B, p.q_tiles, p.group, m_tile, h, b);
  const int hk = h / p.group;
  // Query tiles of the waves: eight consecutive ones, or, with ds_pairs, two 256-row blocks, waves 0..3 the m_tile-th from the
  // start and waves 4..7 the m_tile-th from the end, so that all workgroups read the same number of images (the middle one of
  // an odd number of blocks goes to waves 4..7 alone).
  const int rg = wave / FS, fh = wave % FS;
  const bool pairs = CAUSAL && p.ds_pairs;
  const int half_blocks = (p.Sq + kBM / 2 - 1) / (kBM / 2);
  auto rows_of = [&](int w) __attribute__((always_inline)) {
    if (!pairs) return m_tile * kBM + w * QW;
    const int late = half_blocks - 1 - m_tile;
    const int block = w >= RG / 2 ? late : m_tile < late ? m_tile : half_blocks;  // half_blocks: none
    return block * (kBM / 2) + (w & (RG / 2 - 1)) * QW;
  };
  const int m_end = pairs ? (half_blocks - m_tile) * (kBM / 2) : (m_tile + 1) * kBM;  // behind the workgroup's last row
  const int q_wave0 = rows_of(rg);

  const bool two_part = MULTI && p.k_pe != nullptr;  // keys in two parts
  const int k_head = two_part ? 128 : DQK;
  const int kv_row_bytes = p.HkvT * k_head * 2, extra_row_bytes = two_part ? (int)p.k_pe_rs * 2 : kv_row_bytes;

  // Key steps of chunk i: of the workgroup all that one of its rows sees, in the queries' own chunk up to the diagonal (every wave
  // walks these); of the 64-row group from q0 on what it sees, none if the tile does not exist (ragged Sq).
  const int last = MULTI ? chunk_count(p) - 1 : 0;
  auto chunk_steps = [&](int i) __attribute__((always_inline)) {
    const KeyChunk& ch = chunk_of(p, i);
    const int all = (ch.rows + kBN - 1) / kBN;
    return CAUSAL && i == last ? min(all, (m_end - 1) / kBN + 1) : ch.q_row0 < m_end ? all : 0;
  };
  auto group_steps = [&](int i, int q0) __attribute__((always_inline)) {
    const KeyChunk& ch = chunk_of(p, i);
    const int all = (ch.rows + kBN - 1) / kBN;
    if ((q0 >> 6) >= p.ds_qt) return 0;
    return CAUSAL && i == last ? min(all, (q0 + QW - 1) / kBN + 1) : q0 >= ch.q_row0 ? all : 0;
  };

  // ---- requests. Waves 0..3: K tiles. Waves 4..7: the images of row groups w-4 and, with 8 of them, w. What a request costs in scalar
  // instructions is on the way from one barrier to the next.
  const bool k_mover = wave < 4;
  DirectTile128<kBN, 256> mover;
  mover.init(kv_row_bytes, wave & 3, lane);
  dkdv_d192::DirectExtra<kBN / 2> extra;  // features 128..191
  if constexpr (DQK == 192) extra.init(extra_row_bytes, wave & 3, lane);
  int image_lane = lane << 4;
  // the mover's place in the stream, ahead of the products: what it moves next, tiles or images left of its chunk
  const char* src[kImages] = {};
  int left[kImages] = {};
  const int64_t src_step = k_mover ? (int64_t)kBN * kv_row_bytes : kDsWave;
  int at_chunk = -1, steps_left = 0, keys_left = 0;
  const char* extra_src = nullptr;
  unsigned issued = 0;  // kImages bits per step, those of the last one requested lowest: loads were issued for it
  auto next_chunk = [&]() __attribute__((always_inline)) {
    ++at_chunk;
    if constexpr (MULTI) {
      while (at_chunk <= last && chunk_steps(at_chunk) == 0) ++at_chunk;
      if (at_chunk > last) return;
    }
    steps_left = chunk_steps(at_chunk);
    const KeyChunk& ch = chunk_of(p, at_chunk);
    keys_left = ch.rows;
#pragma unroll
    for (int r = 0; r < kImages; ++r) {
      const int q0 = rows_of((wave & 3) + 4 * r);
      const int64_t bh = b * p.Hq + h;
      const char* image;  // key step s = pair s&3 of key block s>>2: 4 KB each, consecutive in s
      if constexpr (MULTI) {
        const BwdChunk& c = p.chunk[at_chunk];
        const int64_t tile = at_chunk == last ? ds_tile_start<true>(q0 >> 6, c.ds_kb) : ds_tile_start<false>((q0 - ch.q_row0) >> 6, c.ds_kb);
        image = p.ds + c.ds_off + bh * c.ds_hs + tile * kDsBlockBytes;
      } else {
        image = p.ds + bh * p.ds_hs + ds_tile_start<CAUSAL>(q0 >> 6, p.ds_kb) * kDsBlockBytes;
      }
      const char* k_src = reinterpret_cast<const char*>(ch.k + b * p.k_bs + (int64_t)hk * k_head);
      src[r] = k_mover ? k_src : image;  // (an image that does not exist is not loaded)
      left[r] = !k_mover ? group_steps(at_chunk, q0) : r == 0 ? steps_left : 0;
      extra_src = two_part ? reinterpret_cast<const char*>(ch.k_pe + b * p.k_pe_bs) - 256 : k_src;  // (the mover adds the first part's 256 bytes)
    }
  };
  next_chunk();
  int k_slot = 0, k_next = kRingK - 1, d_slot = 0, d_next = kRingD - 1;  // of the step and of the next one to request
  auto request_next = [&](int slot) __attribute__((always_inline)) {
    issued <<= kImages;
    if constexpr (MULTI) {
      if (steps_left == 0 && at_chunk <= last) next_chunk();
      --steps_left;
    }
#pragma unroll
    for (int r = 0; r < kImages; ++r) {
      if (left[r] <= 0) continue;
      if (r == 0 && k_mover) {
        char* const stage = smem + slot * kKStage;
        mover.issue(src[0], keys_left, stage, wave & 3, lane);
        if constexpr (DQK == 192) {
          extra.issue(two_part ? extra_src : src[0], keys_left, stage + kBN * kRowBytes128, wave & 3, lane);
          extra_src += (int64_t)kBN * extra_row_bytes;
        }
        keys_left -= kBN;
      } else {
        load_image_once(src[r], image_lane, smem + kOffDs + slot * kDsStage + ((wave & 3) + 4 * r) * kDsWave);
      }
      src[r] += src_step;
      --left[r];
      issued |= 1u << r;
    }
  };
  if (k_mover) {
#pragma unroll 1
    for (int d = 0; d < kRingK - 1; ++d) request_next(d);
  } else {
#pragma unroll 1
    for (int d = 0; d < kRingD - 1; ++d) request_next(d);
  }
  // The next step: every wave waits until its loads for it have landed (those issued for later ones may stay in flight) and the
  // barrier publishes them; everyone is done with the step before, whose slots are requested anew.
  auto begin = [&]() __attribute__((always_inline)) {
    if (k_mover) {
      static_assert(kRingK == 3, "one K step in flight");
      if (issued & 1) wait_vector_loads_but<kLoadsK>();
      else wait_vector_loads_but<0>();
    } else {
      constexpr int kLater = (kRingD - 2) * kImages;  // images requested after this step's
      constexpr unsigned kAll = (1u << kLater) - 1, kUpper = kAll / 3 * 2;
      static_assert(kLater * kLoadsDs < 32, "loads in flight fit the decision tree");
      const unsigned in_flight = issued & kAll;
      if (in_flight == kAll) wait_vector_loads_but<kLater * kLoadsDs>();
      else if (kImages == 2 && in_flight == kUpper) wait_vector_loads_but<kLater / 2 * kLoadsDs>();  // the later rows' alone
      else if (in_flight == 0) wait_vector_loads_but<0>();
      else wait_vector_loads_but<0, 31>(kLoadsDs * __builtin_popcount(in_flight));
    }
    __syncthreads();
    request_next(k_mover ? k_next : d_next);
  };
  auto advance = [&]() __attribute__((always_inline)) {
    k_slot = k_slot + 1 == kRingK ? 0 : k_slot + 1;
    k_next = k_next + 1 == kRingK ? 0 : k_next + 1;
    d_slot = d_slot + 1 == kRingD ? 0 : d_slot + 1;
    d_next = d_next + 1 == kRingD ? 0 : d_next + 1;
  };

  f32x16 acc[RBW][DB];  // [32-row block][feature block]
#pragma unroll
  for (int rb = 0; rb < RBW; ++rb)
#pragma unroll
    for (int o = 0; o < DB; ++o)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[rb][o][v] = 0.f;

  // per-lane read offsets. K tile: transposing reads of the lower / upper 8 keys of a 16-key step at
  // feature block 0; block o follows by XOR with o << 6 (the swizzle is an XOR of the piece index).
  // Image: this lane supplies, for its 16-lane block (g, chalf) and r = 4i + m, the 8 bytes that hold
  // key 4g + i (+ 8 for the upper read) at queries 16*chalf + 4m .. +3 of a 32-row block: 16-row step
  // chalf of the block, writer lane group m&1, fragment half m>>1.
  const int t_base[2] = {transposed_offset128(0, 0, 0, lane), transposed_offset128(0, 1, 0, lane)};
  // with 192 features per 16-key step and block of this wave, blocks 4 and 5 in the extra tile (its two 16-key steps side by side)
  int k_off[DQK == 192 ? 2 : 1][DB][2];
  if constexpr (DQK == 192) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int o = 0; o < DB; ++o) {
        const int fb = DB * fh + o;
        const int tile = fb < 4 ? ks * 16 * kRowBytes128 : kBN * kRowBytes128;
        const int piece_bits = fb < 4 ? fb << 6 : (8 * ks + 4 * (fb - 4)) << 4;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) k_off[ks][o][hh] = tile + (t_base[hh] ^ piece_bits);
      }
  }
  int ds_off[2];
  {
    const int r = lane & 15, chalf = (lane >> 4) & 1;
    const int i = r >> 2, m = r & 3, gl = m & 1;
    const int key = 4 * g + i;
    ds_off[0] = chalf * 1024 + gl * 512 + ((key ^ (gl << 3) ^ (chalf << 2)) << 4) + (m >> 1) * 8;
    ds_off[1] = ds_off[0] ^ 128;  // key + 8: bit 3 of the key index
  }

  // fragments of 16 of a step's keys, and their products
  struct Half {
    bf16x8 ds[RBW], k[DB];
  };
  auto read = [&](Half& f, int ks) __attribute__((always_inline)) {
    const char* const stage = smem + k_slot * kKStage;
    const char* const img = smem + kOffDs + d_slot * kDsStage + rg * kDsWave + ks * 256;
#pragma unroll
    for (int rb = 0; rb < RBW; ++rb) f.ds[rb] = lds_read_transposed_at(img + rb * 2048 + ds_off[0], img + rb * 2048 + ds_off[1]);
#pragma unroll
    for (int o = 0; o < DB; ++o) {
      if constexpr (DQK == 192) {
        f.k[o] = lds_read_transposed_at(stage + k_off[ks][o][0], stage + k_off[ks][o][1]);
      } else {
        const char* kt = stage + ks * 16 * kRowBytes128;
        f.k[o] = lds_read_transposed_at(kt + (t_base[0] ^ (o << 6)), kt + (t_base[1] ^ (o << 6)));
      }
    }
  };
  auto multiply = [&](const Half& f) __attribute__((always_inline)) {
#pragma unroll
    for (int o = 0; o < DB; ++o)
#pragma unroll
      for (int rb = 0; rb < RBW; ++rb) acc[rb][o] = mfma32(f.ds[rb], f.k[o], acc[rb][o]);
  };
  // multiplies `f` while the next half's fragments are read into `next`, two reads behind every product
  auto multiply_and_read = [&](const Half& f, Half& next, int ks) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    read(next, ks);
    multiply(f);
#pragma unroll
    for (int m = 0; m < DB * RBW; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // The steps of chunk i. At 192 features the late rows walk most of the longest streams alone, one wave to a SIMD, and with the reads in
  // front of its products a wave does one or the other: there the reads of either half go between the products of the half before
  // (a step begins between its predecessor's halves). 128 features wait for the images: the same woven, 0-0.5 % slower.
  auto walk = [&](int i) __attribute__((always_inline)) {
    const int n_wg = chunk_steps(i), n_own = group_steps(i, q_wave0);
    int s = 0;
    Half first, second;
    if constexpr (DQK == 192) {
      if (n_own > 0) {
        begin();
        read(first, 0);
        for (; s + 1 < n_own; ++s) {
          multiply_and_read(first, second, 1);
          advance();
          begin();
          multiply_and_read(second, first, 0);
        }
        multiply_and_read(first, second, 1);
        multiply(second);
        advance();
        ++s;
      }
    } else {
      for (; s < n_own; ++s) {
        begin();
        read(first, 0);
        multiply(first);
        read(second, 1);
        multiply(second);
        advance();
      }
    }
    // other waves of the workgroup may still have steps to visit: keep moving tiles, keep in step
    for (; s < n_wg; ++s) {
      begin();
      advance();
    }
  };
  if constexpr (MULTI)
    for (int i = 0; i <= last; ++i) walk(i);
  else walk(0);

  OutT* dqh = reinterpret_cast<OutT*>(p.dq) + b * p.dq_bs + (int64_t)h * DQK + fh * (32 * DB);
  const float sc = -p.scale;  // the images hold -dS (the writer forms delta - dP)
  const int64_t row_stride = (int64_t)p.HqT * DQK;
#pragma unroll
  for (int rb = 0; rb < RBW; ++rb) {
    const int row0 = q_wave0 + 32 * rb;
    __bf16* fin = nullptr;  // rows whose gradient is complete with this call go out as bf16
    if (p.dq_final != nullptr && row0 >= p.final_r0 && row0 < p.final_r1)
      fin = p.dq_final + b * p.dq_final_bs + (int64_t)h * DQK + fh * (32 * DB) + row0 * row_stride;
    store_rows32<OutT, DB>(dqh + row0 * row_stride, row_stride, p.Sq - row0, acc[rb], sc, p.accumulate_dq != 0, c, g, fin);
  }
}

}  // namespace

// Under the mask a workgroup of 512 consecutive rows carries up to twice the average work. In a grid of one round the heaviest
// one is the kernel's time, so there the rows go out as pairs of blocks of equal work. In more rounds consecutive rows, the
// heaviest first, fill the units by themselves, while pairs, all alike, leave the last round as empty as it is. The kernel
// alone, consecutive rows / pairs, us:
//   one round         4096 x 32/4 heads 143 / 118, 8192 x 16 273 / 219, 4 x 1024 x 32/4 38 / 35, 8 x 512 x 32/4 24 / 24
//   1.125 rounds      9216 x 16 328 / 382, 4608 x 32/4 168 / 204, 3 x 1536 x 32/4 55 / 89
//   1.25, 1.5, 1.75   5120 x 32/4 196 / 225, 6144 x 32/4 256 / 271, 3 x 1999 x 32/4 102 / 114, 7168 x 32/4 322 / 337
//   2, 2.25           8192 x 32/4 405 / 409, 2 x 4096 x 32/4 224 / 233, 9216 x 32/4 517 / 599
//   2.75, 3, 4        11264 x 32/4 785 / 799, 12288 x 32/4 921 / 904, 3 x 4096 x 32/4 341 / 353, 16384 x 32/4 1524 / 1565
// 256 rows of 192 features, 16 heads unless others are named, the same:
//   up to one round   3072 71 / 54, 4096 100 / 80, 2 x 2048 55 / 45, 4 x 1024 33 / 29, 8 x 512 22 / 20, 16384 x 4 368 / 283
//   1.12-2            4608 114 / 142, 5120 129 / 159, 3 x 1999 62 / 79, 6144 160 / 194, 8192 248 / 279, 1024 x 128 51 / 56
//   2.25-8            9216 328 / 412, 12288 568 / 608, 4096 x 64 266 / 300, 4096 x 128 564 / 609
// and shares of four ranks, rank 1, whose rows walk the other chunks at equal length (backward without delta, zigzag and contiguous):
//   up to one round   3072 620 / 571 and 431 / 418, 4096 1004 / 948 and 697 / 680, in two parts 1015 / 958, 4 x 1024 329 / 314 and 224 / 220
//   1.12-2            4608 1234 / 1363 and 902 / 974, 5120 1481 / 1620 and 1088 / 1152, 6144 2042 / 2190 and 1538 / 1587, 8192 3520 / 3646 and 2644 / 2660
bool dq_ds_pairs(int64_t workgroups) { return workgroups <= compute_units_or_default(); }

void launch_dq_from_ds(BwdParams p, int dqk, bool causal, bool f32_out, hipStream_t st) {
  p.ds_pairs = dq_ds_pairs((int64_t)p.q_tiles * p.Hq * p.B);
  const dim3 grid((unsigned)(p.q_tiles * p.Hq * p.B)), block(kThreads);
  auto launch = [&](auto dqk) {
    constexpr int D = decltype(dqk)::value;
    if (causal) {
      if (f32_out) hipLaunchKernelGGL((attn_bwd_dq_ds_kernel<D, true, float>), grid, block, 0, st, p);
      else hipLaunchKernelGGL((attn_bwd_dq_ds_kernel<D, true, __bf16>), grid, block, 0, st, p);
    } else {
      if (f32_out) hipLaunchKernelGGL((attn_bwd_dq_ds_kernel<D, false, float>), grid, block, 0, st, p);
      else hipLaunchKernelGGL((attn_bwd_dq_ds_kernel<D, false, __bf16>), grid, block, 0, st, p);
    }
  };
  if (dqk == 192) launch(std::integral_constant<int, 192>{});
  else launch(std::integral_constant<int, 128>{});
}

void launch_dq_from_ds_chunks(BwdChunkParams p, hipStream_t st) {
  const unsigned workgroups = (unsigned)(p.q_tiles * p.Hq * p.B);
  p.ds_pairs = dq_ds_pairs(workgroups);
  hipLaunchKernelGGL((attn_bwd_dq_ds_kernel<192, true, __bf16, true>), dim3(workgroups), dim3(kThreads), 0, st, p);
}

}  // namespace pith
