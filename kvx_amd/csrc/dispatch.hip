// Host-side launch planning: picks a kernel family, its chunk width, tile
// shape and grid for a validated write or gather plan, and enqueues it on
// the caller's stream through the run_* entry points of kernels.h.
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "kvx_internal.h"

namespace kvx {
namespace dev {
namespace {

GeomBytes to_bytes(const Geom &g, int esize) {
  GeomBytes r;
  r.s_block = g.s_block * esize;
  r.s_off = g.s_off * esize;
  r.s_head = g.s_head * esize;
  r.s_piece = g.s_piece * esize;
  r.s_inner = g.s_inner * esize;
  r.pack = g.pack;
  r.pad_ = 0;
  return r;
}

bool aligned(const void *p, int64_t b) {
  return ((uintptr_t)p % (uintptr_t)b) == 0;
}

// True when chunks of g elements (g*esize bytes each) stay inside one
// contiguous cache piece and every cache address they use is aligned.  A
// block of one token never steps by the offset stride, nor a cache of one
// head by the head stride (size-1 axes, whose strides can be anything, e.g.
// 1 for vLLM's [num_blocks, H, D, 1] value cache).
bool cache_chunk_ok(const Geom &g, const void *base, int esize, int head_dim,
                    int ge, int64_t block_size, int64_t heads) {
  const int64_t bytes = (int64_t)ge * esize;
  if (ge > 1 && g.s_inner != 1) return false;
  if (g.pack % ge != 0 || head_dim % ge != 0) return false;
  if (!aligned(base, bytes)) return false;
  const int64_t strides[4] = {g.s_block, block_size == 1 ? 0 : g.s_off, heads == 1 ? 0 : g.s_head,
                              g.s_piece};
  for (int64_t st : strides) {
    if ((st * esize) % bytes != 0) return false;
  }
  return true;
}

// Widest chunk (elements) that works for K, V and the io buffers.  The io
// side is contiguous with rows of H*D elements of io_size bytes.
int pick_chunk(const Geom &gk, const Geom &gv, const void *ck, const void *cv,
               int cache_size, const void *ik, const void *iv, int io_size,
               int head_dim, int max_chunk_bytes_cache, int64_t block_size, int64_t heads) {
  for (int ge = max_chunk_bytes_cache / cache_size; ge >= 1; ge /= 2) {
    if (!cache_chunk_ok(gk, ck, cache_size, head_dim, ge, block_size, heads)) continue;
    if (!cache_chunk_ok(gv, cv, cache_size, head_dim, ge, block_size, heads)) continue;
    const int64_t io_bytes = (int64_t)ge * io_size;
    if (!aligned(ik, io_bytes) || !aligned(iv, io_bytes)) continue;
    return ge;
  }
  return 1;
}

int lpt_log2_for(int nchunks) {
  int lg = 0;
  while ((1 << lg) < nchunks && lg < 6) ++lg;
  return lg;
}

hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

// HIP's limits on one grid dimension: at most 2^31 - 1 workgroups and
// 2^32 - 1 work-items (gridDim.x * blockDim.x).
bool grid_fits(int64_t workgroups, int threads) {
  return workgroups <= 0x7FFFFFFF && workgroups * threads <= 0xFFFFFFFFll;
}

int log2_exact(int64_t v) {
  if (v <= 0 || (v & (v - 1)) != 0) return -1;
  int lg = 0;
  while ((int64_t(1) << lg) < v) ++lg;
  return lg;
}

// Row (head, dim) elements at consecutive addresses: row-major layouts, and
// any dense layout whose block holds one row (HND, x-packed or token axis
// innermost with block_size 1 store a row as H * D consecutive elements).
// With one head the head stride is never used (HND with H = 1 is row-major
// whenever rows are D elements apart).  On MI355X (c2's lengths in
// one-token blocks) such gathers took 1592-1615 us per layer in the flat
// kernel against 3517-3551 us in the tile kernels.
bool row_elems_contiguous(const Geom &g, int64_t D, int64_t H) {
  return g.s_inner == 1 && (g.s_head == D || H == 1) && (g.pack == D || g.s_piece == g.pack);
}

// Elements of one per-token contiguous run when `g` is a dense block in
// (run, offset, within-run) order, element e of row o at
// (e / W) * bs * W + o * W + e % W, else -1: W = H * D (row-major), D (HND),
// x (x-packed) or 1 (token axis innermost).  Any block stride.
int64_t dense_run_elems(const Geom &g, int64_t bs, int64_t H, int64_t D) {
  // one row, or rows of one head D elements apart: row-major
  if (row_elems_contiguous(g, D, H) && (bs == 1 || g.s_off == H * D)) return H * D;
  const int64_t p = g.pack;
  const bool split = p < D;  // d = (d / p) * p + d % p with its own strides
  if (g.s_inner == 1 && (!split || g.s_piece == p)) {
    if (g.s_off == H * D && g.s_head == D) return H * D;
    if (g.s_off == D && g.s_head == bs * D) return D;
  }
  if (split && g.s_inner == 1 && g.s_off == p && g.s_piece == bs * p && g.s_head == bs * D)
    return p;
  if (g.s_off == 1 && g.s_inner == bs && (!split || g.s_piece == bs * p) && g.s_head == bs * D)
    return 1;
  return -1;
}

// Transposing-gather plan (gather_tiles_kernel) for a PACKED-table gather of
// dense blocks of which at least one is not row-major, or false.  On MI355X
// (c2 shapes, bf16) it beats the row kernel for every run length measured:
// token-innermost 2.45 -> 5.90 TB/s, x-packed 4.66 -> 5.88, HND (256-byte
// runs) 5.14 -> 5.87.  kTileBytes is the cache bytes per tensor of one
// tile (8 KiB measured best against 4 and 16 KiB); workgroups have about
// one thread per kTileBytesPerThread bytes of tile.
constexpr int64_t kTileBytes = 8192;
constexpr int64_t kTileBytesPerThread = 32;
// Narrowest tile width (cache bytes per row) the halving below goes to.
constexpr int64_t kTileMinWidth = 128;
// Tiles whose width is not a power of two: at most kOddTileBytes of cache
// bytes per tensor, at least kOddTileMin.
constexpr int64_t kOddTileBytes = 12288;
constexpr int64_t kOddTileMin = 4096;

int64_t gcd64(int64_t a, int64_t b) {
  while (b != 0) {
    const int64_t t = a % b;
    a = b;
    b = t;
  }
  return a;
}

// div_magic's multiplier for divisor d >= 2: ceil(2^32 / d).
uint32_t magic_for(int64_t d) { return (uint32_t)(((uint64_t(1) << 32) + (uint64_t)d - 1) / (uint64_t)d); }

// Tile width of whole runs (a multiple of `unit`) that divides the row, for
// rows or runs that are not a power of two, phase 2 dividing by chunks per
// row with a multiply-high (HND heads of 96 or 80 bf16 elements, three
// 256-byte heads): widths of whole 128-byte lines first, then the tile
// nearest `target` bytes, the wider on a tie, within kOddTileMin and
// max(target, kOddTileBytes); -1 if none.  On MI355X (c2's table, 4
// layers) such gathers took 5-8% less time than in gather_rows_kernel;
// widths that split output lines between two workgroups (320 or 192
// bytes) measured 7-12% slower than line-multiple ones (640 or 384 bytes),
// three 256-byte heads 20% slower in 4 KiB tiles than in 12 KiB ones, and
// HND 8 x 96 bf16 3% faster in 6 KiB tiles than in 12 KiB ones.
int64_t odd_tile_width(int64_t row, int64_t unit, int64_t bs, int64_t target) {
  if (row % unit != 0) return -1;
  const int64_t cap = target > kOddTileBytes ? target : kOddTileBytes;
  int64_t tw = -1, best = 0;
  for (int64_t k = row / unit; k >= 1; --k) {
    if ((row / unit) % k != 0) continue;
    const int64_t w = unit * k, bytes = w * bs;
    if (bytes < kOddTileMin || bytes > cap) continue;
    const int64_t dist = bytes > target ? bytes - target : target - bytes;
    const int64_t score = (w % 128 == 0 ? 0 : (int64_t)1 << 40) + dist;
    if (tw < 0 || score < best) {
      tw = w;
      best = score;
    }
  }
  return tw;
}

// gather_rows_kernel: cache row bytes per tensor of one workgroup's share
// of a block, at least (blocks of up to kRowsTileBytes stay whole).
constexpr int64_t kRowsTileBytes = 32768;

bool plan_tiles(const GatherPlan &p, int cs, int is, int src_chunk, TileArgs *t,
                int64_t *grid, uint32_t *lds_bytes) {
  const bool offsets = p.format == KVX_BLOCK_TABLE_KV_OFFSETS;
  const bool ragged = p.format == KVX_BLOCK_TABLE_RAGGED;
  // a block's rows, or those of one of its parts.  Of 1-byte runs (a
  // token-innermost FP8 tensor) 64 rows are half a line of every run, so parts
  // hold 128 there, but for rows of a whole number of KiB (8, 16 and 24 heads of
  // 128), which 64 suit better.  vLLM's pair, 128-token blocks, PACKED, E4M3
  // to bf16, 180000 tokens, 64 -> 128 rows, us: 2 x 128 59.7 -> 54.8, 8 x 96 171
  // -> 160, 12 x 128 348 -> 318, 576 (64-byte tiles) 127 -> 110; 8 x 128 202 ->
  // 212, 24 x 128 617 -> 631.  RAGGED loads a part's block ids with one wave.
  const int64_t full_bs = p.block_size;
  const int full_log2 = log2_exact(full_bs);
  const int64_t row_codes = (int64_t)p.heads * p.head_dim;
  int part_rows_log2 = kTileMaxRowsLog2;
  if (!ragged && cs == 1 && row_codes % 1024 != 0)
    for (const Geom *t : {&p.gk, &p.gv})
      if (dense_run_elems(*t, full_bs, p.heads, p.head_dim) == 1)
        part_rows_log2 = kTileMaxRowsLog2 + 1;
  const int parts_log2 = full_log2 > part_rows_log2 ? full_log2 - part_rows_log2 : 0;
  const int64_t bs = full_bs >> parts_log2;
  const int64_t H = p.heads;
  const int64_t D = p.head_dim;
  const int64_t row_cache = H * D * cs;
  const int bs_log2 = log2_exact(bs);
  if (full_log2 < 0 || row_cache < 16) return false;
  if (row_cache * full_bs > 0x7FFFFFFF) return false;  // 32-bit offsets in a block
  const Geom *g[2] = {&p.gk, &p.gv};
  const void *src[2] = {p.src_k, p.src_v};
  void *dst[2] = {p.dst_k, p.dst_v};
  int run_log2[2];
  int64_t run_bytes[2] = {0, 0};
  bool transposed = false, odd_run = false;
  int64_t min_tw = 16;
  int64_t unit = 16;  // a tile width holds whole runs and 16-byte chunks
  for (int i = 0; i < 2; ++i) {
    const int64_t w = dense_run_elems(*g[i], full_bs, H, D);
    if (w < 0) return false;
    run_log2[i] = w == H * D ? -1 : log2_exact(w * cs);
    if (w != H * D) {
      run_bytes[i] = w * cs;
      if (run_log2[i] < 0) {
        // runs that are not a power of two: 16-byte pieces, one run each
        if (run_bytes[i] % 16 != 0) return false;
        run_log2[i] = kRunOdd;
        odd_run = true;
      }
      transposed = true;
      if (w * cs > min_tw) min_tw = w * cs;
      unit = unit / gcd64(unit, run_bytes[i]) * run_bytes[i];
    }
    // block addresses: base + index * pitch, all 16-byte aligned
    const uintptr_t base =
        offsets ? reinterpret_cast<uintptr_t>(p.pool[0]) | reinterpret_cast<uintptr_t>(p.pool[1]) |
                      (uintptr_t)p.bytes_per_block
                : reinterpret_cast<uintptr_t>(src[i]) | (uintptr_t)(g[i]->s_block * cs);
    if (base % 16 != 0) return false;
    const int dst_align = src_chunk / cs * is;  // output bytes per chunk
    if (reinterpret_cast<uintptr_t>(dst[i]) % dst_align != 0) return false;
  }
  if (!transposed) return false;  // row-major pairs: the flat kernels
  // Copies of whole-line runs (HND) through RAGGED and KV_OFFSETS tables keep
  // gather_indexed_kernel where a whole block makes no tile (RAGGED: in any
  // block of parts), its waves are full (a power of two of 16-byte chunks a
  // row, or 64 and more) and its lanes hold a row's chunks (4 KiB; 3 KiB of
  // runs of more than 256 bytes).  Parts -> rows, us, 36000 tokens back to
  // back / cold / 180000 tokens, 256-token blocks: 8 x 128 bf16 RAGGED 53 / 59 /
  // 252 -> 42 / 46 / 250, KV_OFFSETS 51 / 59 / 251 -> 41 / 43 / 232; 2 x 128 f32
  // RAGGED 30 / 35 / 129 -> 22 / 28 / 130; 8 x 96 bf16 KV_OFFSETS 41 / 46 / 202
  // -> 27 / 38 / 192.  Left in parts: 3 x 128 bf16 RAGGED 22 / 26 / 92 (rows 19 /
  // 30 / 116), 8 x 128 f32 99 / 102 / 468 (117 / 97 / 546), 16 x 128 f32 190 /
  // 192 / 930 (234 / 211 / 1120).
  if (parts_log2 > 0 && p.conv == kConvCopy && (ragged || offsets)) {
    int64_t narrowest = row_cache;
    for (int i = 0; i < 2; ++i)
      if (run_bytes[i] > 0 && run_bytes[i] < narrowest) narrowest = run_bytes[i];
    const int64_t chunks = row_cache / 16;
    const bool full_waves = log2_exact(chunks) >= 0 || chunks >= kWave;
    const bool block_tile = !ragged && !odd_run && full_bs * (min_tw + kTilePad) <= 64 * 1024;
    if (narrowest >= 128 && row_cache <= (narrowest > 256 ? 3072 : 4096) && full_waves &&
        !block_tile)
      return false;
  }
  if ((D * cs) % src_chunk != 0) return false;  // chunks never straddle heads
  // Tile width: a power of two that divides the row and holds whole runs.
  // A row that is not a power of two (6 or 12 heads, say) makes several
  // tiles of its largest power-of-two divisor, when that still fills a tile:
  // on MI355X (c2's table) HND gathers of 6 x 128 and 12 x 64 bf16 heads
  // measured 0.676 of peak in 8 KiB tiles against 0.63 in gather_rows_kernel,
  // 3 x 128 heads 0.587 in 4 KiB tiles against 0.623.
  // (The whole block counts there: parts of 64 rows keep the width, in smaller
  // tiles, rather than take one that splits lines.  576-byte FP8 rows, x-packed,
  // 128 / 256-token blocks, 180000 tokens: 64-byte tiles 111 us, 144-byte 186.)
  int64_t tw = row_cache & -row_cache;
  if (odd_run || tw < min_tw ||
      ((row_cache & (row_cache - 1)) != 0 && tw * full_bs < kTileBytes)) {
    tw = odd_tile_width(row_cache, unit, bs, kTileBytes);
    if (tw < 0) return false;
  } else {
    // halve toward kTileBytes, but not below one 128-byte output line per
    // row: narrower rows split output lines between workgroups (x-packed
    // blocks of 128 tokens in 64-byte tile rows 2315 -> 1789 us per layer)
    while (tw * bs > kTileBytes && tw / 2 >= min_tw && tw / 2 >= kTileMinWidth) tw /= 2;
  }
  const int64_t pitch = tw + kTilePad;
  if (bs * pitch > 64 * 1024) return false;
  t->table = p.block_table;
  t->seq_lens = p.seq_lens;
  t->indptr = p.indptr;
  t->table_count = p.table_count;
  t->pool[0] = p.pool[0];
  t->pool[1] = p.pool[1];
  t->bytes_per_block = p.bytes_per_block;
  t->pool_blocks[0] = p.pool_blocks[0];
  t->pool_blocks[1] = p.pool_blocks[1];
  t->out_row_bytes = H * D * is;
  t->max_blocks_per_seq = p.max_blocks_per_seq;
  const int64_t by_len = ((int64_t)p.max_seq_len + bs - 1) / bs;
  // RAGGED rows do not use max_blocks_per_seq
  const int64_t by_table = (int64_t)p.max_blocks_per_seq << parts_log2;
  t->blocks_per_seq = (int32_t)(ragged || by_len < by_table ? by_len : by_table);
  t->tiles = (int32_t)(row_cache / tw);
  t->tw = (int32_t)tw;
  t->tw_log2 = log2_exact(tw);
  // phase 2 chunks per row; div_magic is exact for u * cpr <= 2^32, and
  // u * cpr < bs * tw * tw <= 2^16 * tw (bs * pitch <= 64 KiB below)
  t->cpr = (int32_t)(tw / src_chunk);
  t->cpr_magic = t->tw_log2 < 0 ? magic_for(t->cpr) : 0;
  t->pitch = (int32_t)pitch;
  // Workgroups of about one thread per kTileBytesPerThread bytes of
  // tile (64 to 256 threads): smaller tiles run in smaller workgroups, more
  // of them resident per CU, so that as many bytes are in flight as for the
  // 8 KiB tiles of wider rows.  On MI355X (c2's table, one KV head) 4 KiB
  // x-packed tiles took 198.8 us in 128-thread workgroups against 259.9 us
  // in 256-thread and 209.7 us in 64-thread ones; HND two-token blocks 1585
  // against 2058 us per layer.
  t->threads = kBlockThreads;
  while (t->threads > 64 && tw * bs < (int64_t)t->threads * kTileBytesPerThread)
    t->threads /= 2;
  t->max_seq_len = p.max_seq_len;
  t->num_blocks = p.num_blocks;
  t->head_dim = p.head_dim;
  t->row_elems = (int32_t)(H * D);
  t->bs_log2 = bs_log2;
  t->parts_log2 = parts_log2;
  t->cache_es_log2 = log2_exact(cs);
  t->io_es_log2 = log2_exact(is);
  const ScaleRef sc[2] = {p.k_scale, p.v_scale};
  for (int i = 0; i < 2; ++i) {
    t->t[i].src = static_cast<const char *>(src[i]);
    t->t[i].dst = static_cast<char *>(dst[i]);
    t->t[i].s_block = g[i]->s_block * cs;
    t->t[i].sc = sc[i];
    t->t[i].run_log2 = run_log2[i];
    // stage_tile_odd divides region offsets (< 64 KiB) by the run: exact
    // for runs below 2^16 bytes
    t->t[i].run_bytes = (int32_t)run_bytes[i];
    t->t[i].run_magic = run_log2[i] == kRunOdd ? magic_for(run_bytes[i]) : 0;
    const int64_t run = run_log2[i] < 0 ? row_cache : run_bytes[i];
    t->t[i].gap = run_log2[i] < 0 ? 0 : (int32_t)((full_bs - bs) * run);
    if (t->t[i].gap >= 1 << 24 || row_cache / run >= 1 << 24) return false;
    t->t[i].s_tile = tw * (run_log2[i] < 0 ? bs : full_bs);
    t->t[i].s_part = bs * run;
  }
  *grid = (int64_t)p.seq_count * t->blocks_per_seq * t->tiles;
  *lds_bytes = (uint32_t)(bs * pitch);
  return grid_fits(*grid, t->threads);
}

// Tiled write plan (write_tiles_kernel): dense blocks of which at least one
// is not row-major, 16-byte aligned block addresses, cache rows of whole
// 16-byte chunks, io rows aligned to the tile op's source chunk, and
// (quantizing) heads a whole number of 8-element chunks, so that every chunk
// has one scale.  The constants by measurement on MI355X (same process,
// medians, us per launch):
//
// kWriteTileBytes: cache bytes per tensor of one workgroup, and
// kWriteLdsCopyBytes those of a copy through LDS (76800 tokens of 8 x 128
// bf16 in 16-token blocks, 8 -> 16 KiB: x-packed 120.3 -> 118.7, vLLM's pair
// 121.6 -> 118.3; HND, direct, 118.2 -> 119.6).  A quantizing workgroup of 16
// KiB would take more than kTileLoads chunks per lane.  Batches that make
// fewer than kWriteTileWorkgroups of them per tensor (decode) halve them down
// to kWriteTileMin, so that the rows spread over the CUs (64 decode tokens,
// 8 -> 2 -> 1 KiB: x-packed 4.33 -> 3.63 -> 3.45, vLLM's pair 8.35 -> 6.07 ->
// 5.30; 4000 tokens unchanged).
constexpr int64_t kWriteTileBytes = 8192;
constexpr int64_t kWriteLdsCopyBytes = 16384;
constexpr int64_t kWriteTileMin = 1024;
constexpr int64_t kWriteTileWorkgroups = 512;
// Tokens per workgroup of staged and narrow tensors, at most: 16 store half
// lines of narrow runs (vLLM's pair, 64-token blocks, 19200 tokens: 74
// against 33) and x-packed chunks that start inside blocks took 38 against
// 27; 64 leave a wave no lanes for the rows that follow (narrow: 174).
constexpr int64_t kWriteTileRows = 32;
// Cache bytes per row of a workgroup through LDS, at least, where small batches
// make small tiles: kWriteStagedWidth, or kWriteNarrowRuns narrow runs where
// those are fewer bytes, so that a tile's rows hold whole units (16 rows of FP8
// codes).  Narrow tensors also have a thread for every kTileLoads runs, since
// decode batches store one run at a time.  vLLM's pair, us, 128-byte rows and
// threads by bytes -> now: E4M3, 4000 tokens of 1 x 128 in 64 / 128-token blocks
// 27.4 / 42 -> 6.0 / 6.3, 1000 of 3 x 128 23 / 28 -> 6.5 / 6.7, 64 decode tokens
// of 8 x 128 in 16-token blocks 6.6 -> 5.6, 8 tokens 6.1 -> 5.3; bf16, 1000
// tokens, 7% over heads and blocks; f32 the same.
constexpr int64_t kWriteStagedWidth = 128;
constexpr int64_t kWriteNarrowRuns = 32;
// Bytes of a narrow run that one workgroup stores whole, at most.
constexpr int64_t kWriteAlignBytes = 64;
// Bytes per row of a direct tensor's workgroup, at most: whole rows of 2 KiB
// measured 112 and 108 for HND 32-token blocks (76800 tokens, chunks starting
// inside blocks and on them), 512 bytes 117 and 117.
constexpr int64_t kWriteDirectWidth = 2048;

// Row-major pairs take this kernel (both tensors direct: four chunks of one
// tensor per lane where write_flat_kernel has one of each) when the bytes
// they read and write lie within these bounds, about what the 256 MB
// Infinity Cache holds of them.  NHD, flat -> tiles: 8 x 128 bf16, 1000 /
// 4000 / 10000 / 30000 tokens 3.19 / 8.28 / 16.97 / 47.25 -> 3.56 / 7.09 /
// 13.93 / 46.43; into E4M3 4000 / 10000 / 30000 tokens 7.50 / 14.52 / 34.65
// -> 7.64 / 12.46 / 34.69; 1 x 576 bf16, 30000 tokens 26.6 -> 24.3; 8 x 256
// f32, 4000 / 10000 tokens 24.4 / 58.4 -> 21.2 / 60.9.
// Those are back-to-back writes of the same rows.  Other states of the cache,
// one write at a time, 19200 tokens of 8 x 128 bf16 and 25600 into E4M3, flat
// -> tiles: rows just written by another kernel, the rest clean 26.6 -> 28.0
// and 32.3 -> 28.7, the rest dirty 33.4 -> 27.2 and 34.8 -> 30.8; everything
// evicted by reads 33.9 -> 34.4 and 36.4 -> 34.2; rows evicted and the cache
// full of dirty lines, which the rows' allocations then write back, 34.0 ->
// 46.1 and 36.5 -> 52.0.  A KV write's rows come from the kernel before it, so
// the last is not tuned for: non-temporal loads take it to 28 and 39, and the
// back-to-back E4M3 write from 25.4 to 28.3.  Rows of 576 bf16, whose tiles
// leave a second pass nearly empty, are 5% slower where the rest is clean.
constexpr int64_t kWriteRowsMin = 12 << 20;
constexpr int64_t kWriteRowsMax = 256 << 20;
constexpr int64_t kWriteRowsMinQuant = 32 << 20;
constexpr int64_t kWriteRowsMaxQuant = 192 << 20;

// The divisor of `row` that is a multiple of `unit` and at most `target`,
// the widest of whole 128-byte lines first; the narrowest one when all are
// wider than target.
int64_t tile_width(int64_t row, int64_t unit, int64_t target) {
  const int64_t n = row / unit;
  if ((n & (n - 1)) == 0) {
    int64_t w = unit;
    while (w < row && w * 2 <= target) w *= 2;
    return w;
  }
  int64_t best = -1, line = -1;
  for (int64_t k = 1; k <= n && (best < 0 || unit * k <= target); ++k) {
    if (n % k != 0) continue;
    best = unit * k;
    if (best % 128 == 0) line = best;
  }
  return line > 0 ? line : best;
}

bool plan_write_tiles(const WritePlan &p, int cs, int is, WriteTileArgs *wt, int64_t *grid,
                      int32_t *threads, uint32_t *lds_bytes) {
  const int64_t bs = p.block_size;
  const int64_t H = p.heads;
  const int64_t D = p.head_dim;
  const int64_t row = H * D * cs;  // cache bytes
  const bool quant = p.conv == kConvQuant;
  const int chunk = quant ? 8 : 16;  // cache bytes of the op's chunk
  const int src_chunk = chunk / cs * is;
  if (row % 16 != 0 || (quant && D % 8 != 0)) return false;
  const Geom *g[2] = {&p.gk, &p.gv};
  const void *src[2] = {p.src_k, p.src_v};
  void *dst[2] = {p.dst_k, p.dst_v};
  const ScaleRef sc[2] = {p.k_scale, p.v_scale};
  int64_t run_elems[2];
  for (int i = 0; i < 2; ++i) {
    run_elems[i] = dense_run_elems(*g[i], bs, H, D);
    if (run_elems[i] < 0) return false;
  }
  if (run_elems[0] == H * D && run_elems[1] == H * D) {
    const int64_t bytes = 2 * p.num_tokens * (row + H * D * is);
    if (bytes < (quant ? kWriteRowsMinQuant : kWriteRowsMin) ||
        bytes > (quant ? kWriteRowsMaxQuant : kWriteRowsMax))
      return false;  // the flat kernel
  }
  int64_t base_tile = kWriteTileBytes;
  while (base_tile > kWriteTileMin && p.num_tokens * row / base_tile < kWriteTileWorkgroups)
    base_tile /= 2;
  int64_t wgs = 0, need = 0, runs = 0, lds = 0;
  for (int i = 0; i < 2; ++i) {
    const int64_t w = run_elems[i];
    const int64_t run = w * cs;
    if (run % 16 != 0 && (run > 8 || (run & (run - 1)) != 0)) return false;
    if ((reinterpret_cast<uintptr_t>(dst[i]) | (uintptr_t)(g[i]->s_block * cs)) % 16 != 0)
      return false;
    if ((reinterpret_cast<uintptr_t>(src[i]) | (uintptr_t)(H * D * is)) % src_chunk != 0)
      return false;
    WriteTileTensor &t = wt->t[i];
    t.kind = w == H * D || run % 128 == 0 ? kTileDirect : run >= 16 ? kTileStaged : kTileNarrow;
    int64_t tile = base_tile;
    if (t.kind != kTileDirect && !quant && tile == kWriteTileBytes &&
        p.num_tokens * row / kWriteLdsCopyBytes >= kWriteTileWorkgroups)
      tile = kWriteLdsCopyBytes;
    // a tile holds whole 16-byte pieces and whole runs
    const int64_t unit = w == H * D || run < 16 ? 16 : run;
    const int64_t least = t.kind == kTileNarrow && kWriteNarrowRuns * run < kWriteStagedWidth
                              ? kWriteNarrowRuns * run
                              : kWriteStagedWidth;
    const int64_t target = t.kind == kTileDirect
                               ? (tile < kWriteDirectWidth ? tile : kWriteDirectWidth)
                               : (tile / kWriteTileRows < least ? least : tile / kWriteTileRows);
    const int64_t tw = tile_width(row, unit, target);
    int rows_log2 = 0;
    const int64_t cap = t.kind == kTileDirect ? kWave : kWriteTileRows;
    while ((2 << rows_log2) <= cap && (tw << (rows_log2 + 1)) <= tile) ++rows_log2;
    const int64_t cpr = tw / chunk;
    if ((cpr << rows_log2) > need) need = cpr << rows_log2;
    if (t.kind == kTileNarrow && ((tw / run) << rows_log2) > runs) runs = (tw / run) << rows_log2;
    t.src = static_cast<const char *>(src[i]);
    t.dst = static_cast<char *>(dst[i]);
    t.s_block = g[i]->s_block * cs;
    t.s_run = bs * run;
    t.sc = sc[i];
    t.run = (int32_t)run;
    t.run_log2 = log2_exact(run);
    t.rows = 1 << rows_log2;
    t.rows_log2 = rows_log2;
    t.tw = (int32_t)tw;
    t.tiles = (int32_t)(row / tw);
    t.cpr = (int32_t)cpr;
    // exact: u * cpr <= 2^32 for u < 4 * kBlockThreads and cpr of that order
    t.cpr_magic = cpr > 1 ? magic_for(cpr) : 0;
    t.pitch = (int32_t)(tw + kTilePad);
    // narrow runs: units of 16 bytes (8 bytes of 1-byte runs in 8-token
    // blocks) that blocks hold a whole number of
    t.seg = 1;
    if (t.kind == kTileNarrow) {
      const int64_t seg = 16 / run;
      if (bs % seg == 0) t.seg = (int32_t)seg;
      else if (run == 1 && bs % 8 == 0) t.seg = 8;
    }
    // aligned slots of one line (narrow: sector) of a run, as far as one
    // wave's lanes hold the slots of the rows and of those that follow them
    t.align = 1;
    if (t.kind == kTileStaged || t.seg > 1) {
      const int64_t whole = t.kind == kTileStaged ? 128 : kWriteAlignBytes;
      while (t.align * run < whole && bs % (t.align * 2) == 0 && t.align * 2 <= t.rows &&
             t.rows + t.align * 2 <= kWave)
        t.align *= 2;
      if (t.align < t.seg) t.align = 1;
    }
    const int64_t n = (p.num_tokens + t.rows - 1) / t.rows * t.tiles;
    if (n > 0x7FFFFFFF) return false;
    t.workgroups = (uint32_t)n;
    if (n > wgs) wgs = n;
    const int64_t lrows = t.rows + (t.align > 1 ? t.align : 0);
    const int64_t l = t.kind == kTileDirect ? 0 : lrows * (t.pitch + 12);
    if (l > lds) lds = l;
  }
  // about one thread per kTileBytesPerThread bytes of tile, and at most
  // kTileLoads chunks (and runs of a narrow tensor) each
  int64_t nt = kBlockThreads;
  while (nt > kWave && (nt / 2) * kTileLoads >= runs && (nt / 2) * kTileLoads >= need &&
         (nt / 2) * kTileBytesPerThread >= need * chunk)
    nt /= 2;
  if (need > nt * kTileLoads || lds > 64 * 1024) return false;
  wt->slots = p.slots;
  wt->num_tokens = p.num_tokens;
  wt->row_bytes = H * D * is;
  wt->slot_is64 = p.slot_is64;
  wt->block_size = p.block_size;
  wt->bs_log2 = log2_exact(bs);
  wt->num_blocks = p.num_blocks;
  wt->head_dim = p.head_dim;
  wt->cache_es_log2 = log2_exact(cs);
  *grid = wgs;
  *threads = (int32_t)nt;
  *lds_bytes = (uint32_t)lds;
  return grid_fits(*grid, (int)nt);
}

}  // namespace
}  // namespace dev

using namespace dev;

int dtype_size(kvx_dtype_t dt) {
  switch (dt) {
    case KVX_DTYPE_F32: return 4;
    case KVX_DTYPE_F16:
    case KVX_DTYPE_BF16: return 2;
    case KVX_DTYPE_F8_E4M3:
    case KVX_DTYPE_F8_E5M2: return 1;
    default: return 0;
  }
}

kvx_status_t enqueue_write(const WritePlan &p, void *stream) {
  const int cs = dtype_size((kvx_dtype_t)p.cache_dtype);
  const int is = dtype_size((kvx_dtype_t)p.io_dtype);
  const int max_bytes = (p.conv == kConvQuant) ? 8 : 16;
  const int ge = pick_chunk(p.gk, p.gv, p.dst_k, p.dst_v, cs, p.src_k,
                            p.src_v, is, p.head_dim, max_bytes, p.block_size, p.heads);
  const int64_t row_elems = (int64_t)p.heads * p.head_dim;

  WriteArgs a;
  a.src_k = static_cast<const char *>(p.src_k);
  a.src_v = static_cast<const char *>(p.src_v);
  a.dst_k = static_cast<char *>(p.dst_k);
  a.dst_v = static_cast<char *>(p.dst_v);
  a.slots = p.slots;
  a.ksc = p.k_scale;
  a.vsc = p.v_scale;
  a.gk = to_bytes(p.gk, cs);
  a.gv = to_bytes(p.gv, cs);
  a.num_tokens = p.num_tokens;
  a.slot_is64 = p.slot_is64;
  a.block_size = p.block_size;
  a.num_blocks = p.num_blocks;
  a.head_dim = p.head_dim;
  a.nchunks = (int32_t)(row_elems / ge);
  a.chunk_elems = ge;
  a.row_bytes = (int32_t)(row_elems * is);
  a.lpt_log2 = lpt_log2_for(a.nchunks);
  const int tpw = kWave >> a.lpt_log2;
  a.num_groups = (p.num_tokens + tpw - 1) / tpw;
  const int64_t want = (a.num_groups + kWavesPerBlock - 1) / kWavesPerBlock;
  WriteLaunch wl;
  // One wave per token group up to 65536 workgroups, then a grid-stride
  // loop: on MI355X a 2048-workgroup cap made c3-sized NHD prefill writes
  // 2-4% slower (8% with blocks in ascending order).
  wl.grid = (int)(want < 65536 ? want : 65536);
  wl.tiles = plan_write_tiles(p, cs, is, &wl.wt, &wl.tile_grid, &wl.tile_threads, &wl.tile_lds);
  // write_flat_kernel: K and V rows hold H * D consecutive elements.  A
  // chunk count that is not a power of two (576-element MLA rows: 72) finds
  // a chunk's token by multiply-high, exact while the largest flat index
  // times nchunks stays within 2^32.
  auto row_dense = [&](const Geom &g) { return row_elems_contiguous(g, p.head_dim, p.heads); };
  a.nchunks_log2 = log2_exact(a.nchunks);
  a.nchunks_magic = a.nchunks_log2 < 0 ? magic_for(a.nchunks) : 0;
  wl.flat_grid = 0;
  const int64_t flat_total = (int64_t)p.num_tokens * a.nchunks;
  const bool flat_div_ok =
      a.nchunks_log2 >= 0 || (flat_total + kFlatThreads) * a.nchunks <= (int64_t(1) << 32);
  if (row_dense(p.gk) && row_dense(p.gv) && flat_div_ok) {
    const int64_t fg = (flat_total + kFlatThreads - 1) / kFlatThreads;
    if (grid_fits(fg, kFlatThreads)) wl.flat_grid = fg;  // else write_kernel's grid-stride loop
  }
  hipStream_t s = as_stream(stream);

  if (p.conv == kConvCopy) {
    run_write_copy(ge * cs, a, wl, s);
  } else {
    const bool e5 = p.cache_dtype == KVX_DTYPE_F8_E5M2;
    switch (p.io_dtype) {
      case KVX_DTYPE_F32:
        (e5 ? run_write_quant_e5m2_f32 : run_write_quant_e4m3_f32)(ge, a, wl, s);
        break;
      case KVX_DTYPE_F16:
        (e5 ? run_write_quant_e5m2_f16 : run_write_quant_e4m3_f16)(ge, a, wl, s);
        break;
      default:
        (e5 ? run_write_quant_e5m2_bf16 : run_write_quant_e4m3_bf16)(ge, a, wl, s);
        break;
    }
  }
  return hipGetLastError() == hipSuccess ? KVX_STATUS_OK
                                         : KVX_STATUS_INTERNAL_ERROR;
}

kvx_status_t enqueue_gather(const GatherPlan &p, void *stream) {
  const int cs = dtype_size((kvx_dtype_t)p.cache_dtype);
  const int is = dtype_size((kvx_dtype_t)p.io_dtype);
  // RAGGED gathers of caches whose block rows are contiguous take
  // gather_ragged_tile_kernel.
  const int64_t row_elems_all = (int64_t)p.heads * p.head_dim;
  auto rows_contig = [&](const Geom &g) {
    return row_elems_contiguous(g, p.head_dim, p.heads) &&
           (g.s_off == row_elems_all || p.block_size == 1);
  };
  const bool ragged_tile =
      p.format == KVX_BLOCK_TABLE_RAGGED && rows_contig(p.gk) && rows_contig(p.gv);
  const bool rows_dense = row_elems_contiguous(p.gk, p.head_dim, p.heads) &&
                          row_elems_contiguous(p.gv, p.head_dim, p.heads);
  const bool indexed_f32 = p.conv == kConvDequant && is == 4 && !rows_dense &&
                           p.format != KVX_BLOCK_TABLE_PACKED &&
                           row_elems_all < kIndexedDequantF32Row;
  // bytes of cache per chunk at most (FP8: kDequantChunk and its comment)
  const int max_bytes = p.conv != kConvDequant                               ? 16
                        : indexed_f32                                        ? kDequantChunk
                        : p.format == KVX_BLOCK_TABLE_RAGGED && !ragged_tile && is != 4
                            ? kRaggedDequantChunk
                            : dequant_chunk(is);
  const void *base_k = p.src_k;
  const void *base_v = p.src_v;
  if (p.format == KVX_BLOCK_TABLE_KV_OFFSETS) {
    // Blocks start at pool + index * bytes_per_block: every such address is
    // as aligned as the OR of both pool pointers and the block pitch.
    base_k = base_v = reinterpret_cast<const void *>(
        reinterpret_cast<uintptr_t>(p.pool[0]) | reinterpret_cast<uintptr_t>(p.pool[1]) |
        (uintptr_t)p.bytes_per_block);
  }
  hipStream_t s = as_stream(stream);
  // PACKED gathers whose heads are contiguous runs of a power-of-two number
  // of whole 128-byte lines (HND, or HND beside NHD; power-of-two head
  // counts) take the flat kernel with head-run addressing instead of the LDS
  // tiles: every 16-byte load and store is then part of a whole line.
  auto head_runs = [&](const Geom &g) {
    return g.s_inner == 1 && (g.pack == p.head_dim || g.s_piece == g.pack);
  };
  const int64_t head_run_bytes = (int64_t)p.head_dim * cs;
  const bool head_run_flat =
      p.format == KVX_BLOCK_TABLE_PACKED && head_runs(p.gk) &&
      head_runs(p.gv) && !(rows_contig(p.gk) && rows_contig(p.gv)) &&
      log2_exact(p.heads) >= 0 && log2_exact(head_run_bytes) >= 0 && head_run_bytes >= 128 &&
      p.block_size >= kFlatHeadRunsMinBs;
  if (!head_run_flat) {
    // Dense blocks that are not all row-major: the transposing gather.
    TileArgs t;
    int64_t tgrid = 0;
    uint32_t tlds = 0;
    const bool dq = p.conv == kConvDequant;
    if (p.seq_count > 0 && plan_tiles(p, cs, is, dq ? dequant_chunk(is) : 16, &t, &tgrid, &tlds)) {
      if (tgrid == 0) return KVX_STATUS_OK;
      const bool i64 = p.lens_is64 != 0;
      const bool p64 = p.indptr_is64 != 0;
      if (!dq) {
        run_tiles_copy(t, p.format, i64, p64, tgrid, tlds, s);
      } else if (p.cache_dtype == KVX_DTYPE_F8_E5M2) {
        run_tiles_dequant_e5m2(p.io_dtype, t, p.format, i64, p64, tgrid, tlds, s);
      } else {
        run_tiles_dequant_e4m3(p.io_dtype, t, p.format, i64, p64, tgrid, tlds, s);
      }
      return hipGetLastError() == hipSuccess ? KVX_STATUS_OK : KVX_STATUS_INTERNAL_ERROR;
    }
  }
  const int ge = pick_chunk(p.gk, p.gv, base_k, base_v, cs, p.dst_k,
                            p.dst_v, is, p.head_dim, max_bytes, p.block_size, p.heads);
  const int64_t row_elems = (int64_t)p.heads * p.head_dim;

  GatherArgs a;
  a.src_k = static_cast<const char *>(p.src_k);
  a.src_v = static_cast<const char *>(p.src_v);
  a.dst_k = static_cast<char *>(p.dst_k);
  a.dst_v = static_cast<char *>(p.dst_v);
  a.table = p.block_table;
  a.seq_lens = p.seq_lens;
  a.ksc = p.k_scale;
  a.vsc = p.v_scale;
  a.gk = to_bytes(p.gk, cs);
  a.gv = to_bytes(p.gv, cs);
  a.out_row_bytes = row_elems * is;
  a.index_is64 = p.index_is64;
  a.lens_is64 = p.lens_is64;
  a.indptr = p.indptr;
  a.indptr_is64 = p.indptr_is64;
  a.table_count = p.table_count;
  a.pool[0] = p.pool[0];
  a.pool[1] = p.pool[1];
  a.bytes_per_block = p.bytes_per_block;
  a.pool_blocks[0] = p.pool_blocks[0];
  a.pool_blocks[1] = p.pool_blocks[1];
  a.format = p.format;
  a.rows_per_wg = 0;
  a.ragged_tile = 0;
  a.max_blocks_per_seq = p.max_blocks_per_seq;
  const int64_t by_len =
      ((int64_t)p.max_seq_len + p.block_size - 1) / p.block_size;
  a.blocks_per_seq =
      (int32_t)(by_len < p.max_blocks_per_seq ? by_len : p.max_blocks_per_seq);
  a.max_seq_len = p.max_seq_len;
  a.block_size = p.block_size;
  a.num_blocks = p.num_blocks;
  a.head_dim = p.head_dim;
  a.nchunks = (int32_t)(row_elems / ge);
  a.chunk_elems = ge;
  a.lpt_log2 = lpt_log2_for(a.nchunks);
  // Rows of a block form one contiguous run when each row is H*D
  // consecutive elements and consecutive offsets are one row apart.
  auto rows_contiguous = [&](const Geom &g) {
    return row_elems_contiguous(g, p.head_dim, p.heads) &&
           (g.s_off == row_elems || p.block_size == 1);
  };
  a.flat = rows_contiguous(p.gk) && rows_contiguous(p.gv);
  a.cph_log2 = -1;
  if (head_run_flat) {
    a.flat = 1;
    a.cph_log2 = log2_exact(p.head_dim / ge);  // ge divides the power-of-two run
  }
  a.split_log2 = 0;
  a.fold_log2 = 0;
  a.units_per_seq = 0;
  a.nchunks_log2 = log2_exact(a.nchunks);
  a.nchunks_magic = a.nchunks_log2 < 0 ? magic_for(a.nchunks) : 0;
  a.bs_log2 = log2_exact(p.block_size);
  if (p.format != KVX_BLOCK_TABLE_PACKED) {
    // indexed formats: tiles of rows, about TILE_BYTES of each tensor's cache
    // rows.  Rows that are H*D contiguous elements (any row stride) take the
    // flat kernels, which find a chunk's row by a shift or, for chunk counts
    // that are not a power of two (DeepSeek's 576-element MLA rows: 72), by
    // a multiply-high, exact while tile chunks * nchunks <= 2^32, for rows of
    // at most kFlatRowChunks chunks; otherwise the row kernel, with at least
    // one full pass of its row groups.
    const int max_chunks =
        p.conv == kConvDequant && is == 4 ? kFlatRowChunksDequantF32 : kFlatRowChunks;
    const bool chunks_ok = a.nchunks_log2 >= 0 || a.nchunks <= max_chunks;
    a.flat = rows_dense && chunks_ok;
    if (ragged_tile && chunks_ok) {
      // R rows of about kFlatTileBytes of cache per tensor: a power of
      // two <= 64 (one block id per lane) that divides block_size
      int64_t want = kFlatTileBytes / (row_elems * cs);
      int64_t r = 1;
      while (r * 2 <= want && r * 2 <= kWave && p.block_size % (r * 2) == 0) r *= 2;
      // a large batch whose table holds few of the rows the grid covers (one
      // entry per token: skewed lengths): tiles of twice the rows
      const int64_t entries = p.table_count;
      if (entries * kRaggedSparse < (int64_t)p.seq_count * p.max_seq_len &&
          entries >= r * kRaggedSparseTiles && r * 2 <= kWave && p.block_size % (r * 2) == 0)
        r *= 2;
      a.ragged_tile = 1;
      a.rows_per_wg = (int32_t)r;
      a.blocks_per_seq = (int32_t)(((int64_t)p.max_seq_len + r - 1) / r);
      // copies of sequences of kRaggedFoldMinUnits to kRaggedFoldMaxUnits
      // tiles: two tiles per workgroup, tile w and w + J (J workgroups per
      // sequence)
      a.units_per_seq = a.blocks_per_seq;
      if (p.conv == kConvCopy && a.blocks_per_seq >= kRaggedFoldMinUnits &&
          a.blocks_per_seq <= kRaggedFoldMaxUnits) {
        a.fold_log2 = 1;  // the kernel is built for one or two tiles
        a.blocks_per_seq = (a.blocks_per_seq + 1) >> 1;
      }
    }
    const bool ragged_copy = a.flat && p.format == KVX_BLOCK_TABLE_RAGGED && p.conv == kConvCopy;
    int64_t rows = (ragged_copy ? kRaggedCopyTileBytes : kGatherTileBytes) /
                   (row_elems * cs);
    const int64_t per_pass = a.flat ? 1 : (int64_t)kWavesPerBlock * (kWave >> a.lpt_log2);
    rows = rows < per_pass ? per_pass : rows;
    if (a.flat && p.format == KVX_BLOCK_TABLE_KV_OFFSETS) {
      // a power of two no larger than the (power-of-two) block: tiles never
      // straddle blocks
      int64_t r2 = 1;
      while (r2 * 2 <= rows && r2 * 2 <= p.block_size) r2 *= 2;
      rows = r2;
    }
    if (!a.ragged_tile) {
      a.rows_per_wg = (int32_t)rows;
      a.blocks_per_seq = (int32_t)(((int64_t)p.max_seq_len + rows - 1) / rows);
    }
  } else if (a.flat) {
    // split a block's chunks into a power-of-two number of equal ranges of
    // about kFlatTileBytes of cache per tensor, while the grid stays
    // within HIP's limits (larger ranges loop inside a workgroup)
    const int64_t chunks = (int64_t)p.block_size * a.nchunks;
    const int64_t chunk_bytes = (int64_t)ge * cs;
    const int64_t blocks = (int64_t)p.seq_count * a.blocks_per_seq;
    while ((chunks >> a.split_log2) * chunk_bytes > kFlatTileBytes &&
           ((chunks >> (a.split_log2 + 1)) << (a.split_log2 + 1)) == chunks &&
           a.split_log2 < 16 && grid_fits(blocks << (a.split_log2 + 1), kFlatThreads))
      ++a.split_log2;
    const int64_t per_seq = (int64_t)a.blocks_per_seq << a.split_log2;  // units
    if (per_seq > 0x7FFFFFFF) return KVX_STATUS_UNSUPPORTED;
    // up to 1 << fold_log2 units per workgroup, strided by the workgroups
    // per sequence (kFlatFoldLog2)
    a.units_per_seq = (int32_t)per_seq;
    if (per_seq >= kFlatFoldMinUnits && per_seq <= kFlatFoldMaxUnits) a.fold_log2 = kFlatFoldLog2;
    a.blocks_per_seq = (int32_t)((per_seq + (1 << a.fold_log2) - 1) >> a.fold_log2);
  } else if (a.bs_log2 >= 0) {
    // gather_rows_kernel: a power-of-two block's rows split into
    // 1 << split_log2 equal ranges of at least kRowsTileBytes of cache
    // rows per tensor (and one full pass of the row groups), so that big
    // blocks still give the grid enough workgroups: on MI355X (c2's lengths
    // in 256-token HND blocks, bf16) 2009 -> 1775 us per layer
    const int64_t per_pass = (int64_t)kWavesPerBlock * (kWave >> a.lpt_log2);
    int64_t want = kRowsTileBytes / (row_elems * cs);
    if (want < per_pass) want = per_pass;
    const int64_t blocks = (int64_t)p.seq_count * a.blocks_per_seq;
    while ((p.block_size >> (a.split_log2 + 1)) >= want && a.split_log2 < 16 &&
           grid_fits(blocks << (a.split_log2 + 1), kBlockThreads))
      ++a.split_log2;
    const int64_t per_seq = (int64_t)a.blocks_per_seq << a.split_log2;  // workgroups
    if (per_seq > 0x7FFFFFFF) return KVX_STATUS_UNSUPPORTED;
    a.blocks_per_seq = (int32_t)per_seq;
  }
  if (a.blocks_per_seq <= 0 || p.seq_count <= 0) return KVX_STATUS_OK;
  const int64_t grid = (int64_t)p.seq_count * a.blocks_per_seq;
  // threads per workgroup of the kernel launch_gather_typed picks
  int threads = kBlockThreads;
  if (p.format == KVX_BLOCK_TABLE_PACKED) {
    if (a.flat) threads = kFlatThreads;
  } else if (a.ragged_tile) {
    threads = kFlatThreads;
  } else if (a.flat && p.format == KVX_BLOCK_TABLE_RAGGED && p.conv == kConvCopy) {
    threads = kRaggedCopyThreads;
  }
  // one workgroup per (sequence, tile): a batch whose grid exceeds HIP's
  // limits (some 4 x 10^9 work-items) is not launched
  if (!grid_fits(grid, threads)) return KVX_STATUS_UNSUPPORTED;

  if (p.conv == kConvCopy) {
    run_gather_copy(ge * cs, a, grid, s);
  } else {
    const bool e5 = p.cache_dtype == KVX_DTYPE_F8_E5M2;
    switch (p.io_dtype) {
      case KVX_DTYPE_F32:
        (e5 ? run_gather_dequant_e5m2_f32 : run_gather_dequant_e4m3_f32)(ge, a, grid, s);
        break;
      case KVX_DTYPE_F16:
        (e5 ? run_gather_dequant_e5m2_f16 : run_gather_dequant_e4m3_f16)(ge, a, grid, s);
        break;
      default:
        (e5 ? run_gather_dequant_e5m2_bf16 : run_gather_dequant_e4m3_bf16)(ge, a, grid, s);
        break;
    }
  }
  return hipGetLastError() == hipSuccess ? KVX_STATUS_OK
                                         : KVX_STATUS_INTERNAL_ERROR;
}

}  // namespace kvx
