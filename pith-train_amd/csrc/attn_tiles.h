// Device building blocks shared by the attention kernels (forward, dQ, dK/dV) on gfx950.
//
// Matrix-core conventions used everywhere (v_mfma_f32_32x32x16_bf16, one wavefront of 64 lanes,
// lane = 32*g + c with c = lane % 32, g = lane / 32):
//   A operand (32 x 16): lane holds row c, contraction slots k = 8*g + e, e = 0..7
//   B operand (16 x 32): lane holds column c, the same contraction slots
//   C/D      (32 x 32): lane holds column c, rows 8*(v/4) + 4*g + v%4, v = 0..15
// A result tile can therefore be fed back as the B operand of a product that contracts over
// its ROW index without leaving registers: slot (g, e) of contraction step j then stands for
// row 16*j + 8*(e/4) + 4*g + e%4 of the tile ("slot order"). The other operand of that product
// is fetched from LDS in the same slot order.
//
// Tiles streamed through LDS are packed, swizzled rows (see below). They are read
//   - "straight": lane takes 8 consecutive columns of row c            (one ds_read_b128), or
//   - "transposed": lane takes column c at 8 rows in slot order         (two ds_read_b64_tr_b16).
#pragma once

#include "pith_common.h"

namespace pith {

typedef __attribute__((address_space(3))) char lds_char;

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Transposed fragments in slot order: for a wavefront the A (or B) operand whose non-contracted index is the tile COLUMN
// col_base + c and whose contraction slots (g, e) are the tile ROWS row_base + 8*(e/4) + 4*g + e%4 (lds_read_transposed_at
// below). ds_read_b64_tr_b16 works on blocks of 16 lanes: lane r of a block supplies the address of 4
// consecutive columns; lanes 4i..4i+3 of the block must cover 16 consecutive columns of row i;
// lane r then receives column r of rows 0..3 of the block.

// Row index (0..31) inside a 32x32 result tile of accumulator element v for lane group g.
__device__ __forceinline__ int acc_row(int v, int g) { return 8 * (v >> 2) + 4 * g + (v & 3); }

// max / sum across the two lanes (c, c+32) that share a result column.
__device__ __forceinline__ float pair_max(float x) {
  const int xi = __float_as_int(x);
  const auto r = __builtin_amdgcn_permlane32_swap(xi, xi, false, false);
  return fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const int xi = __float_as_int(x);
  const auto r = __builtin_amdgcn_permlane32_swap(xi, xi, false, false);
  return __int_as_float(r[0]) + __int_as_float(r[1]);
}

// Eight fp32 accumulator values -> bf16 fragment (round-to-nearest-even).
__device__ __forceinline__ bf16x8 to_bf16x8(float a0, float a1, float a2, float a3, float a4, float a5, float a6,
                                            float a7) {
  bf16x8 r;
  r[0] = (__bf16)a0; r[1] = (__bf16)a1; r[2] = (__bf16)a2; r[3] = (__bf16)a3;
  r[4] = (__bf16)a4; r[5] = (__bf16)a5; r[6] = (__bf16)a6; r[7] = (__bf16)a7;
  return r;
}

// Maps a linear workgroup id to (tile, head, batch) so that
//   - tiles are visited from `tiles-1` down to 0 (under a causal mask the late tiles carry the most work, and
//     the lightest workgroups should be the last ones dispatched);
//   - workgroups are dealt round-robin to the 8 XCDs of the device, each with its own L2: the
//     heads of one level are permuted so that an XCD keeps a contiguous range of heads, i.e. the
//     query heads that share a kv head read their K/V through the same L2;
//   - with more than 8 kv heads per level (`group` = query heads per kv head) and at least `chunked` tiles
//     the heads are taken in chunks of 8 kv heads, all tiles of a chunk before the next chunk: the workgroups an
//     XCD holds at one time then belong to ONE kv head and stream the same K/V tiles at about the same time,
//     instead of one stream per head. Each chunk ends with its light tiles, so the order is no longer
//     heaviest-first over the whole grid: measured 9-14 % faster at 128 heads x 32768 rows, 2-6 % slower at 4096
//     rows (16-32 tiles), hence the threshold; the forward with 128-row workgroups goes by the size of K and V instead
//     (attn_fwd_duo.hip).
constexpr int kChunkedTiles = 64;
__device__ __forceinline__ void decode_block(int linear, int heads, int batch, int tiles, int group, int& tile, int& h, int& b, int chunked = kChunkedTiles) {
  const int per_level = heads * batch;
  const int chunk = 8 * group;
  int level, pos;
  if (tiles >= chunked && per_level > chunk && per_level % chunk == 0) {
    const int per_chunk = chunk * tiles;
    const int c = linear / per_chunk;
    const int rem = linear - c * per_chunk;
    level = rem / chunk;
    const int u = rem - level * chunk;
    pos = c * chunk + (u & 7) * group + (u >> 3);
  } else {
    level = linear / per_level;
    pos = linear - level * per_level;
    if ((per_level & 7) == 0) pos = (pos & 7) * (per_level >> 3) + (pos >> 3);
  }
  tile = tiles - 1 - level;
  b = pos / heads;
  h = pos - b * heads;
}

// ---------------------------------------------------------------------------------------------
// Several K/V chunks in one launch. A ring share attends its queries to one chunk per ring step; where all of them are at
// hand, a query-stationary workgroup simply walks the key tiles of every chunk its rows can see as one stream: no partial
// results, no merges, one set of first tiles and one epilogue. The chunks come sorted: those without a causal mask by the
// first query row that sees them, then (CAUSAL kernels) the chunk that holds the queries' own keys, under the mask.
constexpr int kMaxChunks = PITH_MAX_CHUNKS;
struct KeyChunk {
  const __bf16* k;
  const __bf16* v;
  const __bf16* k_pe;  // keys in two parts (the same for all chunks: all or none)
  int rows;            // keys of the chunk
  int q_row0;          // query rows below do not see it
};

// How a workgroup walks its stream. MULTI = false: one chunk, addressed by the tile number, which costs nothing beyond what
// a kernel without chunks costs; MULTI = true: several, tiles taken strictly in order (the scalar state of three walks
// measured 1 us per launch and 1-4 % in the loops: worth it only where it saves launches and merges). The kernels'
// parameters P come with chunk_of(p, id) and chunk_count(p).
//
// The chunks that query rows below row_end see: ids 0 .. n_full-1 and, CAUSAL, the last one.
template <bool MULTI, bool CAUSAL, int BN>
struct ChunkRange {
  int n_full, last, tiles_full;
  template <typename P>
  __device__ __forceinline__ ChunkRange(const P& p, int row_end) {
    if constexpr (MULTI) {
      last = chunk_count(p) - 1;
      n_full = tiles_full = 0;
      const int most = CAUSAL ? last : last + 1;
      while (n_full < most && chunk_of(p, n_full).q_row0 < row_end) {
        tiles_full += (chunk_of(p, n_full).rows + BN - 1) / BN;
        ++n_full;
      }
    } else {
      last = 0;
      n_full = CAUSAL ? 0 : 1;
      tiles_full = CAUSAL ? 0 : (chunk_of(p, 0).rows + BN - 1) / BN;
    }
  }
  // the chunk behind chunk i of the stream
  __device__ __forceinline__ int next(int i) const { return i + 1 < n_full ? i + 1 : last; }
  __device__ __forceinline__ int first() const { return MULTI && n_full == 0 ? last : 0; }
};

// Where the requests for one operand stand: address of a tile's first row (`base(chunk id)` gives the chunk's) and rows left
// from it on. Wave-uniform.
template <bool MULTI, bool CAUSAL, int BN>
struct TileSource {
  int id, rows_left, row_bytes;
  const char* at;
  template <typename P, typename Base>
  __device__ __forceinline__ TileSource(const P& p, const ChunkRange<MULTI, CAUSAL, BN>& r, int row_bytes_, Base base) {
    id = r.first();
    rows_left = chunk_of(p, id).rows;
    row_bytes = row_bytes_;
    at = base(id);
  }
  __device__ __forceinline__ const char* src(int t) const { return MULTI ? at : at + (int64_t)t * BN * row_bytes; }
  __device__ __forceinline__ int left(int t) const { return MULTI ? rows_left : rows_left - t * BN; }
  template <typename P, typename Base>
  __device__ __forceinline__ void advance(const P& p, const ChunkRange<MULTI, CAUSAL, BN>& r, Base base) {
    if constexpr (MULTI) {
      rows_left -= BN;
      at += BN * row_bytes;
      if (rows_left <= 0) {
        id = r.next(id);
        rows_left = chunk_of(p, id).rows;
        at = base(id);
      }
    }
  }
};

// Where the softmax stands: which keys of its tile a query row may see.
template <bool MULTI, bool CAUSAL, int BN>
struct TileMask {
  int id, first_key, rows, q_row0;
  template <typename P>
  __device__ __forceinline__ void enter(const P& p, int i) {
    id = i;
    first_key = 0;
    rows = chunk_of(p, i).rows;
    q_row0 = MULTI ? chunk_of(p, i).q_row0 : 0;
  }
  template <typename P>
  __device__ __forceinline__ TileMask(const P& p, const ChunkRange<MULTI, CAUSAL, BN>& r) { enter(p, r.first()); }
  template <typename P>
  __device__ __forceinline__ void advance(const P& p, const ChunkRange<MULTI, CAUSAL, BN>& r) {
    if constexpr (MULTI) {
      first_key += BN;
      if (first_key >= rows) enter(p, r.next(id));
    }
  }
  __device__ __forceinline__ int key0(int t) const { return MULTI ? first_key : t * BN; }
  __device__ __forceinline__ bool diagonal(const ChunkRange<MULTI, CAUSAL, BN>& r) const { return CAUSAL && (!MULTI || id == r.last); }
  // whether some of the wave's query rows from q0 on do not see the whole tile: it crosses the diagonal, is a chunk's ragged
  // last one, or belongs to a chunk that only later rows see
  __device__ __forceinline__ bool partial(const ChunkRange<MULTI, CAUSAL, BN>& r, int t, int q0) const {
    return (diagonal(r) && key0(t) + BN - 1 > q0) || key0(t) + BN > rows || (MULTI && q0 < q_row0);
  }
  // last key of the chunk that row `qrow` sees (-1: none)
  __device__ __forceinline__ int limit(const ChunkRange<MULTI, CAUSAL, BN>& r, int qrow) const {
    const int l = diagonal(r) ? min(qrow, rows - 1) : rows - 1;
    return MULTI && qrow < q_row0 ? -1 : l;
  }
};

// Key tiles of a wave of a query-stationary workgroup: a wave whose 32 rows all lie beyond the last one (ragged Sq) is done with the first
// tile and only moves tiles for the others. It used to multiply to the end for nothing, under the mask in the longest workgroup. us, before /
// after: forward 8 x 643 x 64/4 heads of 128 causal 95.1 / 90.6 (27 % of the work was padding), 8200 x 16 246 / 237, 4100 x 32/4 136.7 / 131.0, 3 x
// 1999 x 32/4 100.7 / 99.4, 4 x 1030 x 16 of 192 32.5 / 31.0, 8 x 1290 x 16/4 of 64 39.7 / 38.0; forward + backward 2 x 414 x 128 of 192 171.1 / 166.1, 5
// x 400 x 32/4 of 128 110.3 / 105.8; shares 4120 x 16 of 192 1609 / 1535, 4100 x 32/4 2605 / 2551. Without a mask only in the forward of small
// workgroups (8 x 643 x 64/4 147 / 140, 6 x 530 x 32/4 42.0 / 39.8, 8 x 1290 x 32/8 of 64 129 / 126): the others know there that all waves walk as far
// as their workgroup, and lose more in the loops without it (256-row forward 8200 x 16 570 / 638, 4 x 1564 x 16 85 / 89; dQ 4100 x 8/2 362 / 371,
// 3 x 3457 x 4 of 64 206 / 211). Nor in the forward of several chunks by wave pairs, which loses with and without such waves: without / with it 4200 x 8/2,
// eight ranks, 397 / 421, 5000 x 8/2 537 / 566, 1262 x 32/4 149 / 155, 4096 x 16 of 192, four ranks, rank 0 322 / 330; 4100 x 8/2 contiguous 262 / 259; nor in
// that of two teams (64 features: 7790 x 8 90.1 / 92.0, 3072 x 16 36.5 / 37.3).
__device__ __forceinline__ int tiles_of_wave(int tiles, int q_wave0, int sq) { return q_wave0 < sq ? tiles : min(tiles, 1); }

// ---------------------------------------------------------------------------------------------
// 128-feature tiles moved global memory -> LDS directly (global_load_lds_dwordx4), without
// passing through registers. One wavefront instruction moves 64 pieces of 16 bytes to 1 KB of
// consecutive LDS (lane L -> byte 16*L of the region), so tile rows are packed at 256 bytes
// (16 pieces) with no padding; bank conflicts are avoided by keeping piece q of row r at
// position q ^ tile_swizzle(r). The swizzle is a bijection of r % 16 (16 consecutive rows read
// "straight" at one feature offset hit 16 different positions) and moves rows r..r+3 to four
// different 64-byte groups (what the transposing read touches at once).
constexpr int kRowBytes128 = 256;

__device__ __forceinline__ int tile_swizzle(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }

// Byte offset inside a packed tile of the 16-byte piece `piece` (0..15) of row `row`.
__device__ __forceinline__ int swizzled_offset(int row, int piece) {
  return row * kRowBytes128 + ((piece ^ tile_swizzle(row)) << 4);
}

// 16 bytes per lane from global address `base` + `offset` (base the same for all lanes, offset
// per lane, unsigned) to LDS at `dst_wave` + 16 * lane; `dst_wave` must be the same for all lanes
// of the wavefront. Completion is tracked by vmcnt, in issue order with the other vector loads.
// Written as inline assembly on purpose: the compiler does not see an LDS write, so it places no
// wait between this load and later LDS reads of OTHER tiles; the caller waits (s_waitcnt vmcnt)
// and synchronises the workgroup before anyone reads the destination.
// The statement overwrites M0 behind the compiler's back: M0 is a reserved register that cannot
// be declared as clobbered (clang warns that such a declaration is not honoured). That is sound
// only while the compiler itself emits no M0 use in a kernel that includes this header (dynamic
// register indexing, s_sendmsg, LDS-DMA or GWS builtins would); tests/test_cabi.py compiles every
// source to assembly and fails if M0 appears anywhere outside these inline statements.
__device__ __forceinline__ void load_lds16(const char* base, int offset, char* dst_wave) {
  const uint32_t lds_addr = (uint32_t)(uintptr_t)(lds_char*)dst_wave;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_addr), "v"(offset), "s"(base)
               : "memory");
}

// The same for bytes that nobody reads again: they pass through the caches without displacing what is read later.
__device__ __forceinline__ void load_lds16_once(const char* base, int offset, char* dst_wave) {
  const uint32_t lds_addr = (uint32_t)(uintptr_t)(lds_char*)dst_wave;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
               :
               : "s"(lds_addr), "v"(offset), "s"(base)
               : "memory");
}

// 16 bytes per lane to `base` (wave-uniform) + `offset`, written through the second-level cache (sc1) and kept by none (nt): for what
// another launch reads, while this one shares tiles through that cache. dS images, plain / nt / sc1 nt / sc0 sc1 nt, forward + backward of
// 4096 x 32/4 heads of 128 569 / 533 / 525 / 527 us, share of 8192 x 32/4 7820 / 7440 / 7353 / 7352 us. The wait states are those
// that a VALU write of the data registers needs behind a store of more than 8 bytes; the compiler does not see the store.
__device__ __forceinline__ void store16_through(char* base, int offset, bf16x8 value) {
  asm volatile("global_store_dwordx4 %0, %1, %2 sc1 nt\n\ts_nop 1" : : "v"(offset), "v"(__builtin_bit_cast(u32x4, value)), "s"(base) : "memory");
}

// 4 bytes per lane from the per-lane global address `src` to LDS at `dst_wave` + 4 * lane (same
// conventions as load_lds16).
__device__ __forceinline__ void load_lds4(const void* src, char* dst_wave) {
  const uint32_t lds_addr = (uint32_t)(uintptr_t)(lds_char*)dst_wave;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
               :
               : "s"(lds_addr), "v"(src)
               : "memory");
}

// Moves a [ROWS x 128] bf16 tile with THREADS threads (THREADS / 64 wavefronts): wavefront w
// moves the 4 tile rows of every 1 KB region n * WAVES + w. With 4 * WAVES a multiple of 16 the
// swizzle of a lane's row is the same in every region, so one per-lane source offset serves all
// regions and the region only moves the (uniform) source address on.
template <int ROWS, int THREADS>
struct DirectTile128 {
  static constexpr int kWaves = THREADS / 64;
  static constexpr int kPerThread = ROWS * 16 / THREADS;
  static_assert(ROWS * 16 % THREADS == 0, "tile must split evenly over the threads");
  static_assert((4 * kWaves) % 16 == 0, "rows of successive regions must share their swizzle");
  static constexpr int kTileBytes = ROWS * kRowBytes128;
  int src_off;  // byte offset of this lane's source piece in region 0 from the tile's first row
  int row_bytes;

  // row_bytes: distance between consecutive rows in global memory, in bytes
  __device__ __forceinline__ void init(int row_bytes_, int wave, int lane) {
    row_bytes = row_bytes_;
    const int row = 4 * wave + (lane >> 4);
    src_off = row * row_bytes + (((lane & 15) ^ tile_swizzle(row)) << 4);
  }
  // tile_src: address of [first row of the tile][feature 0] of the head slice (uniform);
  // rows_left: valid rows from there on (>= 1), rows beyond are read from the last valid row.
  // `slot` is the LDS tile (uniform).
  __device__ __forceinline__ void issue(const char* tile_src, int rows_left, char* slot, int wave, int lane) const {
    if (rows_left >= ROWS) {
      // The offset is pinned in a register BEFORE the first load is issued: were it spilled, the
      // compiler would reload it between two loads and wait for the reload with a counter wait that
      // also waits for every tile load issued before it.
      int off = src_off;
      asm volatile("" : "+v"(off));
#pragma unroll
      for (int n = 0; n < kPerThread; ++n)
        load_lds16(tile_src + (int64_t)n * 4 * kWaves * row_bytes, off, slot + (n * kWaves + wave) * 1024);
    } else {
      issue_clamped(tile_src, rows_left, slot, wave, lane);
    }
  }
  // The same for any rows_left, source offsets formed on the spot: a few more vector instructions, but no per-lane
  // register lives from one tile to the next (for kernels that would spill it).
  __device__ __forceinline__ void issue_clamped(const char* tile_src, int rows_left, char* slot, int wave, int lane) const {
#pragma unroll
    for (int n = 0; n < kPerThread; ++n) {
      const int row = 4 * (n * kWaves + wave) + (lane >> 4);
      const int src_row = row < rows_left ? row : rows_left - 1;
      load_lds16(tile_src, src_row * row_bytes + (((lane & 15) ^ tile_swizzle(row)) << 4),
                 slot + (n * kWaves + wave) * 1024);
    }
  }
};

// ---------------------------------------------------------------------------------------------
// Features 128..191 of a 64-row tile of a 192-feature operand (the MLA key / query): a second
// packed tile that holds TWO tile rows per 256-byte LDS row, row r in pieces 0-7 and row r + 32
// in pieces 8-15 of LDS row r (r < 32), under the same swizzle. Read like a 32-row, 128-feature
// tile whose features 64..127 are the second 32-row block: a straight fragment of row block kb,
// row c, contraction step x (0..3) is piece 2x + g + 8*kb of LDS row c; a transposed fragment of
// row block kb, feature block f (0..1) uses col_base = 64*kb + 32*f.
constexpr int kExtraTileBytes = 32 * kRowBytes128;

// Moves that part of a tile global memory -> LDS: one global_load_lds per thread of a 512-thread
// workgroup (wave w fills LDS rows 4w .. 4w+3). Source rows are 384 bytes of features per head.
struct DirectExtra64 {
  int src_off, row_bytes, col_bytes;
  __device__ __forceinline__ static int source(int row_bytes, int col_bytes, int wave, int lane, int rows_left) {
    const int row = 4 * wave + (lane >> 4);
    const int piece = (lane & 15) ^ tile_swizzle(row);
    int key = row + 32 * (piece >> 3);
    key = key < rows_left ? key : rows_left - 1;
    return key * row_bytes + col_bytes + ((piece & 7) << 4);
  }
  // row_bytes: distance between consecutive source rows; col_bytes: where the 64 features start
  // within a source row (256 when they follow the first 128 features of the same row, 0 when they
  // are a tensor of their own)
  __device__ __forceinline__ void init(int row_bytes_, int col_bytes_, int wave, int lane) {
    row_bytes = row_bytes_;
    col_bytes = col_bytes_;
    src_off = source(row_bytes_, col_bytes_, wave, lane, 64);
  }
  __device__ __forceinline__ void issue(const char* tile_src, int rows_left, char* slot, int wave, int lane) const {
    if (rows_left >= 64) load_lds16(tile_src, src_off, slot + wave * 1024);
    else issue_clamped(tile_src, rows_left, slot, wave, lane);
  }
  // source offset formed on the spot, see DirectTile128::issue_clamped
  __device__ __forceinline__ void issue_clamped(const char* tile_src, int rows_left, char* slot, int wave, int lane) const {
    load_lds16(tile_src, source(row_bytes, col_bytes, wave, lane, rows_left), slot + wave * 1024);
  }
};

// The same for tiles of KEYS rows and workgroups of THREADS threads, and for whole 64-feature operands: LDS row r holds
// tile rows r and r + KEYS/2. Wave w fills LDS rows 4w + 4*WAVES*n .. +3, and with 4 * WAVES a multiple of 16 the swizzle
// (hence the source offset) of a lane does not depend on n.
template <int KEYS, int THREADS>
struct DirectPaired64 {
  static constexpr int kWaves = THREADS / 64;
  static constexpr int kPerThread = KEYS / 2 / (4 * kWaves);
  static_assert(KEYS / 2 % (4 * kWaves) == 0 && (4 * kWaves) % 16 == 0, "rows of successive pieces must share their swizzle");
  static constexpr int kTileBytes = KEYS / 2 * kRowBytes128;
  int src_off, row_bytes, col_bytes;
  __device__ __forceinline__ static int source(int row_bytes, int col_bytes, int row, int lane, int rows_left) {
    const int piece = (lane & 15) ^ tile_swizzle(row);
    int key = row + KEYS / 2 * (piece >> 3);
    key = key < rows_left ? key : rows_left - 1;
    return key * row_bytes + col_bytes + ((piece & 7) << 4);
  }
  __device__ __forceinline__ void init(int row_bytes_, int col_bytes_, int wave, int lane) {
    row_bytes = row_bytes_;
    col_bytes = col_bytes_;
    src_off = source(row_bytes_, col_bytes_, 4 * wave + (lane >> 4), lane, KEYS);
  }
  __device__ __forceinline__ void issue(const char* tile_src, int rows_left, char* slot, int wave, int lane) const {
    if (rows_left >= KEYS) {
      int off = src_off;
      asm volatile("" : "+v"(off));  // pinned before the first load, see DirectTile128::issue
#pragma unroll
      for (int n = 0; n < kPerThread; ++n)
        load_lds16(tile_src + (int64_t)n * 4 * kWaves * row_bytes, off, slot + (n * kWaves + wave) * 1024);
    } else {
      issue_clamped(tile_src, rows_left, slot, wave, lane);
    }
  }
  __device__ __forceinline__ void issue_clamped(const char* tile_src, int rows_left, char* slot, int wave, int lane) const {
#pragma unroll
    for (int n = 0; n < kPerThread; ++n)
      load_lds16(tile_src, source(row_bytes, col_bytes, 4 * (n * kWaves + wave) + (lane >> 4), lane, rows_left),
                 slot + (n * kWaves + wave) * 1024);
  }
};

// ---------------------------------------------------------------------------------------------
// A wavefront's 32 stationary rows (Q, dO, K or V) on their way into registers as MFMA B fragments: staged in a wave-private
// LDS area (tile slots that hold nothing yet) with whole-row direct loads, then read like a tile. Fetched straight into
// registers, a fragment load touches 32 rows with 32 bytes each: every lane of a quad on a line of its own, which the address
// unit serves at one lane per cycle (64 cycles per instruction against 16 for contiguous rows). A workgroup of 8 waves then
// spent 2-5 us only on issuing them, in front of or behind its first tiles. From the start of a workgroup of the second round
// to its first interval (stamps inside the kernels), before -> now: forward 4096 x 16 heads of 192 5.3 -> 3.6 us, its dQ 5.7 ->
// 4.0, its dK/dV 4.1 -> 2.6, dK/dV of 4096 x 32/4 of 128 3.8 -> 2.5; fwd + bwd of a layer of 4096 x 16 of 192 (with the spills
// in dQ and the epilogues of this change) 397 -> 382 us, of 4096 x 32/4 of 128 575 -> 571: there the chip is at its power limit
// and gives most of the time back as a lower clock.
//
// Features [col, col + 128) (WIDE: 8 KB, eight loads) or [col, col + 64) (4 KB, four loads, rows r and r + 16 in one 256-byte
// LDS row) of rows row0 .. row0 + 31; rows from `rows` on are read from the last one (row0 may lie beyond it). `src` points to
// row 0, feature `col` of the head. Completion as for tiles (vmcnt); the wave needs no barrier before it reads its own area.
// Waves that own the same rows share an area and the loads: this one issues the loads n0 .. n0 + N - 1 (wave-uniform).
template <bool WIDE, int N = WIDE ? 8 : 4>
__device__ __forceinline__ void stage_rows32(const char* src, int row0, int rows, int row_bytes, char* area, int lane, int n0 = 0) {
  const int first = min(row0, rows - 1), left = rows - first;
  const char* const base = src + (int64_t)first * row_bytes;
  const int sub = lane >> 4, piece = lane & 15;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int n = n0 + i;
    const int p = piece ^ tile_swizzle(4 * n + sub);
    int row = 4 * n + sub + (WIDE ? 0 : 16 * (p >> 3));
    row = row < left ? row : left - 1;
    load_lds16(base, row * row_bytes + ((WIDE ? p : p & 7) << 4), area + n * 1024);
  }
}
// The fragment of contraction step ks (features 16 ks ..) of the row this lane owns, c = lane % 32.
template <bool WIDE>
__device__ __forceinline__ bf16x8 staged_fragment(const char* area, int ks, int c, int g) {
  const int off = WIDE ? swizzled_offset(c, 2 * ks + g) : swizzled_offset(c & 15, (2 * ks + g) | ((c >> 4) << 3));
  return *reinterpret_cast<const bf16x8*>(area + off);
}
// Waits for the wave's own loads; `later` of them, the last ones issued, may stay in flight.
template <int LATER = 0>
__device__ __forceinline__ void wait_staged() {
  static_assert(LATER < 16, "the immediate has four low bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | LATER);
  asm volatile("" ::: "memory");
}

// Per-lane offsets for reading a packed swizzled tile.
// straight_offset(c, piece): fragment of row c (+ a multiple of 16 rows added by the caller as
// rows * 256 bytes), features 8*piece .. 8*piece+7.
__device__ __forceinline__ int straight_offset128(int row, int piece) { return swizzled_offset(row, piece); }

// Offset for one ds_read_b64_tr_b16 of a transposed fragment: tile
// rows row_base + 8*half + 4*(blk>>1) + (r>>2), features col_base + 16*(blk&1) + 4*(r&3) .. +3.
// row_base must be a multiple of 16, col_base a multiple of 32.
__device__ __forceinline__ int transposed_offset128(int row_base, int half, int col_base, int lane) {
  const int r = lane & 15, blk = lane >> 4;
  const int row = row_base + 8 * half + 4 * (blk >> 1) + (r >> 2);
  const int col = col_base + 16 * (blk & 1) + 4 * (r & 3);  // features
  return swizzled_offset(row, col >> 3) + ((col & 7) << 1);
}

__device__ __forceinline__ bf16x8 lds_read_transposed_at(const char* lo_addr, const char* hi_addr) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(lo_addr));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(hi_addr));
  typedef __attribute__((ext_vector_type(8))) short s16x8;
  s16x8 v;
  v[0] = lo[0]; v[1] = lo[1]; v[2] = lo[2]; v[3] = lo[3];
  v[4] = hi[0]; v[5] = hi[1]; v[6] = hi[2]; v[7] = hi[3];
  return __builtin_bit_cast(bf16x8, v);
}

// ---------------------------------------------------------------------------------------------
// Epilogue of the kernels whose accumulators hold their result TRANSPOSED (a lane owns one result
// row, its registers 4-feature pieces of it: accT[o][v] = R[row c][feature 32*o + acc_row(v, g)] for lane
// (c, g)). Written straight from that layout a store instruction touches 32 rows with 16 or 32 bytes
// each, i.e. 32 memory lines, and a compute unit's vector cache keeps only about 64 requests in flight;
// turned through LDS first, every instruction reads or writes whole rows (2 rows x 512 bytes of fp32 per
// instruction at 128 features). `lds` is a wave-private area of kRowsViaLdsBytes<NB> bytes (the tile
// rings are free by then: the caller has passed the barrier behind their last reader); `factor` is this
// lane's (= this row's) scale; rows at or beyond rows_valid are neither read nor written (rows_valid may be <= 0).
// With `accumulate` all old values are read before the first store. With `final_block` (wave-uniform; the same rows of
// a bf16 tensor laid out like `block`) the result, old values included, is rounded to bf16 and written there, and
// `block` keeps what it held.
// bf16 rows leave in one of two ways (through_results): workgroups that are still in their loops share K and V (Q and dO) through the
// second-level cache, which plain stores fill with rows that wait there to be written. fp32 rows are read again soon, by the sums over head parts
// (written through or plain, see there) or the next ring step (plain, nt 0.3 % slower).
template <int NB>
constexpr int kRowsViaLdsBytes = 32 * (NB * 128 + 16);

// Whether results of that many bytes (O, dQ, or dK and dV of a launch together) are written through the second-level caches (sc1) rather than
// non-temporally: as long as the 8 x 4 MB of them could hold it. Either keeps the tiles of the other workgroups cached, but what went out non-temporally its next reader fetches from
// memory. Plain / sc1 / nt, us, the forward alone and with the projection that reads O:
//   2-4 MiB   1024 x 16/4 heads of 64 10.8 / 10.7 / 10.7 and 20.3 / 20.4 / 21.8, 512 x 32/4 of 128 11.1 / 10.7 / 10.8 and 31.8 / 29.9 / 32.5
//   8 MiB     2 x 512 x 32/4 of 128 14.7 / 13.8 / 13.8 and 39.9 / 38.5 / 40.1, 2048 x 16 of 192/128 40.3 / 39.7 / 40.0 and 59.6 / 59.3 / 61.9, 2 x 2048 x 16/4 of 64
//             31.2 / 30.7 / 30.5 and 47.7 / 44.8 / 45.1
//   16 MiB    4 x 512 x 32/4 of 128 18.1 / 17.8 / 16.9 and 53.1 / 51.9 / 52.5, 4096 x 16 of 192/128 91.3 / 90.7 / 89.9 and 123.7 / 123.1 / 125.0
//   32 MiB    8 x 512 x 32/4 of 128 33.4 / 30.3 / 30.2 and 91.2 / 88.5 / 89.7, 4096 x 32/4 126.0 / 124.3 / 124.8 and 183.9 / 181.4 / 183.9
//   47 MiB    3 x 1999 x 32/4 of 128 106.3 / 105.2 / 102.8 and 183.8 / 183.6 / 183.2
// and the backward with the products that read dQ, dK and dV: 512 x 32/4 of 128 71.2 / 71.0 / 72.3, 2048 x 16 of 192/128 181.0 / 181.1 / 182.7, the others within
// 0.5 %. sc1 nt as nt, sc0 sc1 as sc1.
// The fp32 partial sums of a launch (head parts, k_pe per head) follow the same line by the bytes of all of them, with plain stores instead of nt beyond it: their reader is the
// next launch, and what they leave in the second-level caches is written back at the end of the launch. Forward + backward, plain / sc1 / nt, us: 32 MiB 1024 x 32/4 of
// 128 without a mask 94.7 / 92.0 / 93.6, 2 x 2048 x 16/4 of 64 105.0 / 104.3 / 105.7; 56 to 78 MiB 8 x 512 x 32/4 142.3 / 140.8 / 142.5, 3 x 768 x 32/4
// 123.1 / 121.5 / 123.2, but 4 x 947 x 64/4 330 / 332 / 334, 4096 x 32/4 523 / 528 / 532, 4992 x 32/8 of 64 472.5 / 472.9 / 475.3. Per-head k_pe, plain / sc1, equal: 12 MiB
// 1021 x 16, four ranks, 157.5 / 157.5, 32 MiB 4096 x 16, two ranks, 912 / 913, 128 MiB 2 x 4096 x 16 4034 / 4048, 8192 x 16 5073 / 5074.
inline bool through_results(int64_t bytes) { return bytes <= (int64_t)32 << 20; }

template <typename OutT, int NB>
__device__ __forceinline__ void store_rows32_via_lds(char* lds, OutT* block, int64_t row_stride, int rows_valid,
                                                     const f32x16 (&accT)[NB], float factor, bool accumulate, int lane,
                                                     bool through, __bf16* final_block = nullptr) {
#pragma clang fp contract(off)  // product rounded, then added: what accumulating into a separate tensor gives
  constexpr int kPitch = NB * 128 + 16;  // bytes; the 16 spread the 32 rows of a column over the banks
  constexpr int kPieces = NB * 8;        // 16-byte pieces (4 features) per row
  constexpr int kIters = 32 * kPieces / 64;
  // a block that lies wholly beyond the last row (the same for the whole wave): nothing to store, and the
  // clamped old-value loads below would start from `block`, which is itself out of range then
  if (rows_valid <= 0) return;
  const int c = lane & 31, g = lane >> 5;
#pragma unroll
  for (int o = 0; o < NB; ++o)
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) {
      const f32x4 x = {accT[o][4 * b4] * factor, accT[o][4 * b4 + 1] * factor, accT[o][4 * b4 + 2] * factor,
                       accT[o][4 * b4 + 3] * factor};
      *reinterpret_cast<f32x4*>(lds + c * kPitch + (32 * o + 8 * b4 + 4 * g) * 4) = x;
    }
  // the reads below see the writes above: one wave's LDS operations execute in order
  f32x4 val[kIters];
  int row[kIters], piece[kIters];
#pragma unroll
  for (int it = 0; it < kIters; ++it) {
    const int idx = it * 64 + lane;
    row[it] = idx / kPieces;
    piece[it] = idx - row[it] * kPieces;
    val[it] = *reinterpret_cast<const f32x4*>(lds + row[it] * kPitch + piece[it] * 16);
  }
  if (accumulate) {
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
      const OutT* src = block + (row[it] < rows_valid ? row[it] : 0) * row_stride + 4 * piece[it];
      if constexpr (sizeof(OutT) == 4) {
        val[it] += *reinterpret_cast<const f32x4*>(src);
      } else {
        const u32x2 old = *reinterpret_cast<const u32x2*>(src);
        val[it][0] += bf16lo_to_f32(old[0]);
        val[it][1] += bf16hi_to_f32(old[0]);
        val[it][2] += bf16lo_to_f32(old[1]);
        val[it][3] += bf16hi_to_f32(old[1]);
      }
    }
  }
  if (final_block != nullptr) {
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
      if (row[it] < rows_valid) {
        u32x2 w;
        w[0] = pack_bf16x2(val[it][0], val[it][1]);
        w[1] = pack_bf16x2(val[it][2], val[it][3]);
        *reinterpret_cast<u32x2*>(final_block + row[it] * row_stride + 4 * piece[it]) = w;
      }
    }
    return;
  }
  auto store = [&](auto through_tag) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
      if (row[it] < rows_valid) {
        OutT* dst = block + row[it] * row_stride + 4 * piece[it];
        if constexpr (sizeof(OutT) == 4) {
          const u32x4 bits = __builtin_bit_cast(u32x4, val[it]);
          if constexpr (decltype(through_tag)::value) asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(dst), "v"(bits) : "memory");
          else *reinterpret_cast<u32x4*>(dst) = bits;
        } else {
          u32x2 w;
          w[0] = pack_bf16x2(val[it][0], val[it][1]);
          w[1] = pack_bf16x2(val[it][2], val[it][3]);
          if constexpr (decltype(through_tag)::value)  // (a store of device scope is what writes through)
            __hip_atomic_store(reinterpret_cast<uint64_t*>(dst), __builtin_bit_cast(uint64_t, w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          else __builtin_nontemporal_store(w, reinterpret_cast<u32x2*>(dst));
        }
      }
    }
  };
  if (!through) store(std::false_type{});
  else store(std::true_type{});
}

// The same turn through LDS for the forward kernel's merging epilogue: row r of the block becomes
//     f_new[r] * accT[r] + f_old[r] * prev[r]
// (the online-softmax combine of the chunk result in the accumulators with the running result `prev`, bf16 or fp32,
// whose per-row weights the caller has formed from the two LSEs) and is written as bf16 to `out_bf16` and / or as fp32
// to `out_f32` (either may be null, either may alias `prev`: a lane reads the old values of a piece before it writes
// that piece, and no other lane touches it). f_new / f_old are this lane's (= this row's) weights; the old weight
// travels to the lanes that handle the row's pieces through the 16 bytes of padding behind the row in LDS.
// All three tensors are addressed from row 0 of the block, feature 0 of the head.
template <int NB>
__device__ __forceinline__ void merge_rows32_via_lds(char* lds, const void* prev, bool prev_f32, int64_t prev_row_stride,
                                                     __bf16* out_bf16, int64_t out_row_stride, float* out_f32,
                                                     int64_t acc_row_stride, int rows_valid, const f32x16 (&accT)[NB],
                                                     float f_new, float f_old, int lane) {
  constexpr int kPitch = NB * 128 + 16;
  constexpr int kPieces = NB * 8;
  constexpr int kIters = 32 * kPieces / 64;
  if (rows_valid <= 0) return;  // wave-uniform
  const int c = lane & 31, g = lane >> 5;
  // the running values first: their memory latency then overlaps the turn through LDS (the accumulators are still
  // live, which the epilogue can afford)
  f32x4 old[kIters];
  int row[kIters], piece[kIters];
#pragma unroll
  for (int it = 0; it < kIters; ++it) {
    const int idx = it * 64 + lane;
    row[it] = idx / kPieces;
    piece[it] = idx - row[it] * kPieces;
    const int src_row = row[it] < rows_valid ? row[it] : 0;
    if (prev_f32) {
      old[it] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(prev) + src_row * prev_row_stride + 4 * piece[it]);
    } else {
      const u32x2 w = *reinterpret_cast<const u32x2*>(reinterpret_cast<const __bf16*>(prev) + src_row * prev_row_stride + 4 * piece[it]);
      old[it] = f32x4{bf16lo_to_f32(w[0]), bf16hi_to_f32(w[0]), bf16lo_to_f32(w[1]), bf16hi_to_f32(w[1])};
    }
  }
#pragma unroll
  for (int o = 0; o < NB; ++o)
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) {
      const f32x4 x = {accT[o][4 * b4] * f_new, accT[o][4 * b4 + 1] * f_new, accT[o][4 * b4 + 2] * f_new,
                       accT[o][4 * b4 + 3] * f_new};
      *reinterpret_cast<f32x4*>(lds + c * kPitch + (32 * o + 8 * b4 + 4 * g) * 4) = x;
    }
  if (g == 0) *reinterpret_cast<float*>(lds + c * kPitch + NB * 128) = f_old;
  // the reads below see the writes above: one wave's LDS operations execute in order
#pragma unroll
  for (int it = 0; it < kIters; ++it) {
    const f32x4 val = *reinterpret_cast<const f32x4*>(lds + row[it] * kPitch + piece[it] * 16);
    const float fo = *reinterpret_cast<const float*>(lds + row[it] * kPitch + NB * 128);
    if (row[it] >= rows_valid) continue;
    const f32x4 r = val + old[it] * fo;
    if (out_f32) *reinterpret_cast<f32x4*>(out_f32 + row[it] * acc_row_stride + 4 * piece[it]) = r;
    if (out_bf16) {
      u32x2 w;
      w[0] = pack_bf16x2(r[0], r[1]);
      w[1] = pack_bf16x2(r[2], r[3]);
      *reinterpret_cast<u32x2*>(out_bf16 + row[it] * out_row_stride + 4 * piece[it]) = w;
    }
  }
}

}  // namespace pith
