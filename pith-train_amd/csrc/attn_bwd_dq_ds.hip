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
  const char* kh = reinterpret_cast<const char*>(p.k + b * p.k_bs + (int64_t)hk * DQK);

  // key steps: all of them, or up to the diagonal; a wave whose query tile does not exist (ragged
  // Sq) has no images and visits nothing. Rows q0 .. q0+QW-1 lie in the writer's 64-row tile q0 >> 6.
  const int n_steps_all = (p.Skv + kBN - 1) / kBN;
  const int n_steps_wg = CAUSAL ? min(n_steps_all, (m_end - 1) / kBN + 1) : n_steps_all;
  auto steps_of = [&](int q0) __attribute__((always_inline)) {
    if ((q0 >> 6) >= p.ds_qt) return 0;
    return CAUSAL ? min(n_steps_all, (q0 + QW - 1) / kBN + 1) : n_steps_all;
  };
  const int n_steps_wave = steps_of(q_wave0);
  // images of the query tile of rows q0..: key step s = pair s&3 of key block s>>2, 4 KB each,
  // consecutive in s; the rows' part starts 1 KB per 16 rows into each image
  auto images_of = [&](int q0) __attribute__((always_inline)) {
    const int mt = min(q0 >> 6, p.ds_qt - 1);
    return p.ds + (int64_t)(b * p.Hq + h) * p.ds_hs + ds_tile_start<CAUSAL>(mt, p.ds_kb) * kDsBlockBytes + (q0 & 63) * 64;
  };

  // ---- requests. Waves 0..3: K tiles. Waves 4..7: the images of row groups w-4 and, with 8 of them, w.
  const bool k_mover = wave < 4;
  DirectTile128<kBN, 256> mover;
  mover.init(kv_row_bytes, wave & 3, lane);
  dkdv_d192::DirectExtra<kBN / 2> extra;  // features 128..191
  if constexpr (DQK == 192) extra.init(extra_row_bytes, wave & 3, lane);
  const char* ds_src[kImages];  // only used by waves 4..7
  int ds_steps[kImages];
#pragma unroll
  for (int r = 0; r < kImages; ++r) {
    const int q0 = rows_of((wave & 3) + 4 * r);
    ds_src[r] = images_of(q0);
    ds_steps[r] = k_mover ? 0 : steps_of(q0);
  }
  auto request_k = [&](int s, int slot) __attribute__((always_inline)) {
    char* stage = smem + slot * kKStage;
    const char* k_src = kh + (int64_t)s * kBN * kv_row_bytes;
    mover.issue(k_src, p.Skv - s * kBN, stage, wave & 3, lane);
    if constexpr (DQK == 192) extra.issue(k_src, p.Skv - s * kBN, stage + kBN * kRowBytes128, wave & 3, lane);
  };
  auto request_ds = [&](int s, int slot) __attribute__((always_inline)) {
    int off = lane << 4;
    asm volatile("" : "+v"(off));
#pragma unroll
    for (int r = 0; r < kImages; ++r)
      if (s < ds_steps[r]) {
        const char* src = ds_src[r] + (int64_t)s * 4096;
        char* dst = smem + kOffDs + slot * kDsStage + (wave - 4 + 4 * r) * kDsWave;
#pragma unroll
        for (int j = 0; j < kLoadsDs; ++j) load_lds16_once(src + j * 1024, off, dst + j * 1024);
      }
  };
  // loads this wave issued for step t
  auto loads_of = [&](int t) __attribute__((always_inline)) {
    if (t >= n_steps_wg) return 0;
    if (k_mover) return kLoadsK;
    int n = 0;
#pragma unroll
    for (int r = 0; r < kImages; ++r) n += t < ds_steps[r] ? kLoadsDs : 0;
    return n;
  };
  // ring slots of step s (K tiles, dS parts) and of the steps to request next; advanced by one per step
  int k_slot = 0, k_next = kRingK - 1, d_slot = 0, d_next = kRingD - 1;
  auto advance = [&]() __attribute__((always_inline)) {
    k_slot = k_slot + 1 == kRingK ? 0 : k_slot + 1;
    k_next = k_next + 1 == kRingK ? 0 : k_next + 1;
    d_slot = d_slot + 1 == kRingD ? 0 : d_slot + 1;
    d_next = d_next + 1 == kRingD ? 0 : d_next + 1;
  };
  // waits until this wave's loads for step s have landed: the steps requested after it (all but the
  // last of the ring, which follows after the barrier) may stay in flight. Away from the end of the key
  // range that is a constant number of loads.
  constexpr int kSteadyDs = (kRingD - 2) * kImages * kLoadsDs;
  static_assert(kRingK == 3 && kSteadyDs < 32, "one K step in flight; dS loads in flight fit the decision tree");
  const int ds_steady_end = min(min(ds_steps[0], ds_steps[kImages - 1]), n_steps_wg) - (kRingD - 2);  // steps below: steady state
  const int ds_single_end = min(ds_steps[kImages - 1], n_steps_wg) - (kRingD - 2);
  auto wait_step = [&](int s) __attribute__((always_inline)) {
    if (k_mover) {
      if (s + 1 < n_steps_wg) wait_vector_loads_but<kLoadsK>();
      else wait_vector_loads_but<0>();
    } else if (s < ds_steady_end) {
      wait_vector_loads_but<kSteadyDs>();
    } else if (CAUSAL && kImages == 2 && s >= ds_steps[0] && s < ds_single_end) {  // only the later block's images are left
      wait_vector_loads_but<kSteadyDs / 2>();
    } else {
      int n = 0;
#pragma unroll
      for (int d = 1; d < kRingD - 1; ++d) n += loads_of(s + d);
      wait_vector_loads_but<0, 31>(n);
    }
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

  auto compute = [&](const char* stage, const char* img) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {  // 16 keys each
      bf16x8 dsf[RBW];
#pragma unroll
      for (int rb = 0; rb < RBW; ++rb) {
        const char* d = img + rb * 2048 + ks * 256;
        dsf[rb] = lds_read_transposed_at(d + ds_off[0], d + ds_off[1]);
      }
#pragma unroll
      for (int o = 0; o < DB; ++o) {
        bf16x8 a;
        if constexpr (DQK == 192) {
          a = lds_read_transposed_at(stage + k_off[ks][o][0], stage + k_off[ks][o][1]);
        } else {
          const char* kt = stage + ks * 16 * kRowBytes128;
          a = lds_read_transposed_at(kt + (t_base[0] ^ (o << 6)), kt + (t_base[1] ^ (o << 6)));
        }
#pragma unroll
        for (int rb = 0; rb < RBW; ++rb) acc[rb][o] = mfma32(dsf[rb], a, acc[rb][o]);
      }
    }
  };

  if constexpr (MULTI) {
    static_assert(!MULTI || (CAUSAL && kImages == 1 && DQK == 192), "one image per mover and step");
    // Every wave walks the same steps: chunk by chunk those that any row of the workgroup sees, in the last chunk up to the diagonal.
    const int last = chunk_count(p) - 1;
    auto chunk_steps = [&](int i) __attribute__((always_inline)) {
      const KeyChunk& ch = chunk_of(p, i);
      const int all = (ch.rows + kBN - 1) / kBN;
      return i == last ? min(all, (m_end - 1) / kBN + 1) : ch.q_row0 < m_end ? all : 0;
    };
    auto group_steps = [&](int i, int q0) __attribute__((always_inline)) {
      const KeyChunk& ch = chunk_of(p, i);
      const int all = (ch.rows + kBN - 1) / kBN;
      if ((q0 >> 6) >= p.ds_qt) return 0;
      return i == last ? min(all, (q0 + QW - 1) / kBN + 1) : q0 >= ch.q_row0 ? all : 0;
    };
    // The mover's place in the stream, ahead of the products, and what it needs of that chunk.
    int req_i = -1, req_s = 0, req_n = 0, keys_left = 0, image_steps = 0;
    const char *k_src = nullptr, *extra_src = nullptr, *image = nullptr;
    const int q_image0 = rows_of(wave & 3);
    auto next_chunk = [&]() __attribute__((always_inline)) {
      do ++req_i;
      while (req_i <= last && chunk_steps(req_i) == 0);
      if (req_i > last) return;
      req_s = 0;
      req_n = chunk_steps(req_i);
      const KeyChunk& ch = chunk_of(p, req_i);
      keys_left = ch.rows;
      k_src = reinterpret_cast<const char*>(ch.k + b * p.k_bs + (int64_t)hk * k_head);
      extra_src = two_part ? reinterpret_cast<const char*>(ch.k_pe + b * p.k_pe_bs) - 256 : k_src;  // (the mover adds the first part's 256 bytes)
      image_steps = k_mover ? 0 : group_steps(req_i, q_image0);
      if (image_steps > 0) {
        const BwdChunk& c = p.chunk[req_i];
        const int64_t tile = req_i == last ? ds_tile_start<true>(q_image0 >> 6, c.ds_kb) : ds_tile_start<false>((q_image0 - ch.q_row0) >> 6, c.ds_kb);
        image = p.ds + c.ds_off + (int64_t)(b * p.Hq + h) * c.ds_hs + tile * kDsBlockBytes;
      }
    };
    unsigned issued = 0;  // bit j: loads were issued for the step j before the last one requested
    auto request_next = [&](int slot) __attribute__((always_inline)) {
      issued <<= 1;
      if (req_i > last) return;
      if (k_mover) {
        char* const stage = smem + slot * kKStage;
        mover.issue(k_src, keys_left, stage, wave & 3, lane);
        extra.issue(extra_src, keys_left, stage + kBN * kRowBytes128, wave & 3, lane);
        k_src += (int64_t)kBN * kv_row_bytes;
        extra_src += (int64_t)kBN * extra_row_bytes;
        keys_left -= kBN;
        issued |= 1;
      } else if (req_s < image_steps) {
        int off = lane << 4;
        asm volatile("" : "+v"(off));
        char* const dst = smem + kOffDs + slot * kDsStage + (wave - 4) * kDsWave;
#pragma unroll
        for (int j = 0; j < kLoadsDs; ++j) load_lds16_once(image + j * 1024, off, dst + j * 1024);
        image += 4096;
        issued |= 1;
      }
      if (++req_s == req_n) next_chunk();
    };
    next_chunk();
    if (k_mover) {
      for (int d = 0; d < kRingK - 1; ++d) request_next(d);
    } else {
      for (int d = 0; d < kRingD - 1; ++d) request_next(d);
    }
    auto step = [&](auto compute_tag) __attribute__((always_inline)) {
      if (k_mover) {
        if (issued & 1) wait_vector_loads_but<kLoadsK>();
        else wait_vector_loads_but<0>();
      } else {
        constexpr unsigned kLater = (1u << (kRingD - 2)) - 1;  // the steps requested after this one
        if ((issued & kLater) == kLater) wait_vector_loads_but<kSteadyDs>();
        else wait_vector_loads_but<0, 31>(kLoadsDs * __builtin_popcount(issued & kLater));
      }
      __syncthreads();  // every wave's requests for this step have landed; everyone is done with the one before
      request_next(k_mover ? k_next : d_next);
      if constexpr (decltype(compute_tag)::value)
        compute(smem + k_slot * kKStage, smem + kOffDs + d_slot * kDsStage + rg * kDsWave);
      advance();
    };
    for (int i = 0; i <= last; ++i) {
      const int n_wg = chunk_steps(i), n_own = group_steps(i, q_wave0);
      int s = 0;
      for (; s < n_own; ++s) step(std::true_type{});
      for (; s < n_wg; ++s) step(std::false_type{});
    }
  } else {
    if (k_mover) {
#pragma unroll
      for (int d = 0; d < kRingK - 1; ++d)
        if (d < n_steps_wg) request_k(d, d);
    } else {
#pragma unroll
      for (int d = 0; d < kRingD - 1; ++d)
        if (d < n_steps_wg) request_ds(d, d);
    }
    auto step = [&](int s, auto compute_tag) __attribute__((always_inline)) {
      wait_step(s);
      __syncthreads();  // every wave's requests for step s have landed; everyone is done with step s-1
      if (k_mover) {
        if (s + kRingK - 1 < n_steps_wg) request_k(s + kRingK - 1, k_next);
      } else {
        if (s + kRingD - 1 < n_steps_wg) request_ds(s + kRingD - 1, d_next);
      }
      if constexpr (decltype(compute_tag)::value)
        compute(smem + k_slot * kKStage, smem + kOffDs + d_slot * kDsStage + rg * kDsWave);
      advance();
    };
    int s = 0;
    for (; s < n_steps_wave; ++s) step(s, std::true_type{});
    // other waves of the workgroup may still have steps to visit: keep moving tiles, keep in step
    for (; s < n_steps_wg; ++s) step(s, std::false_type{});
  }

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
