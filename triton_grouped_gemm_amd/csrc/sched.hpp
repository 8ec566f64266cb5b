// Per-workgroup tile scheduler for grouped GEMMs.
//
// Every workgroup rebuilds the same small table in LDS from the per-group sizes
// (an exclusive prefix sum of rows and of M-tiles) and then walks the tile space
// with a persistent, XCD-aware stride.  No host-side metadata, no workspace, no
// host/device synchronisation.
#pragma once
#include <type_traits>

#include "common.hpp"

namespace tgg {

constexpr int kMaxGroups = 1024;

template <int MAXG>
struct SchedTableT {
  int64_t row0[MAXG];      // first row of the group in A/C (M modes) or first k (K modes)
  int32_t rows[MAXG];      // valid rows (M modes) or k extent (K modes)
  int32_t tile0[MAXG + 1]; // M modes: exclusive prefix of ceil(rows / BM); K modes: the groups in the order of the tile space (sched_order_groups)
  int32_t pad_;            // how many tiles more a cut at half the tile height has (set by sched_init)
  int64_t scan_[16];       // per-wave totals of the workgroup-wide prefix sums that build the table
};
typedef SchedTableT<kMaxGroups> SchedTable;

struct Tile {
  int g;
  int64_t row0;   // first row of this tile in A and C (M modes); first m within the group (K modes)
  int rows;       // valid rows in this tile (<= BM)
  int n0;
  int64_t k0;     // reduction range [k0, k1)
  int64_t k1;
};

// The functions below that are marked TGG_HD contain no device-only construct: the library also runs them
// on the host to report the tile order (a test hook), so what the tests check is what the kernels execute.
#define TGG_HD __host__ __device__ __forceinline__

TGG_HD int64_t load_size(const void* p, int is64, int i) {
  int64_t v = is64 ? ((const int64_t*)p)[i] : (int64_t)((const int32_t*)p)[i];
  return v < 0 ? 0 : v;
}

// Entry g of the table before the prefix pass: the group's raw extent.
template <class Table>
TGG_HD void sched_load_group(const GemmParams& p, Table& t, int g) {
  if (p.mode == MODE_KG) {
    int64_t s = p.k_start[g], e = p.k_end[g];
    if (s < 0) s = 0;
    if (e > p.k_total) e = p.k_total;
    t.row0[g] = s;
    t.rows[g] = e > s ? (int32_t)(e - s) : 0;
  } else {
    t.rows[g] = (int32_t)load_size(p.sizes, p.sizes_i64, g);
  }
}

// Serial prefix pass over the loaded extents (every mode but MODE_KG, whose ranges are explicit).
template <int BM, class Table>
TGG_HD void sched_prefix(const GemmParams& p, Table& t) {
  const int G = p.G;
  int64_t row = 0;
  int32_t tile = 0;
  for (int g = 0; g < G; ++g) {
    int64_t sz = t.rows[g];
    int64_t start;
    if (p.mode == MODE_MASKED) {
      start = (int64_t)g * p.m_stride;
      if (sz > p.m_stride) sz = p.m_stride;
    } else {
      start = (p.mode == MODE_MG_PAD && p.row_start) ? (int64_t)p.row_start[g] : row;
      row += (p.mode == MODE_MG_PAD) ? ((sz + p.align - 1) / p.align) * p.align : sz;
    }
    const int64_t limit = (p.mode == MODE_KG_COUNT) ? p.k_total : p.m_total;
    if (start < 0 || start >= limit) sz = 0;  // never touch rows (or k) outside the operands (a negative start can only come from row_start)
    else if (start + sz > limit) sz = limit - start;
    t.row0[g] = start;
    t.rows[g] = (int32_t)sz;
    t.tile0[g] = tile;
    tile += (int32_t)((sz + BM - 1) / BM);
  }
  t.tile0[G] = tile;
}

// K-grouped tile space: a tile costs what its group has tokens, every group has the same number of tiles, and the
// persistent workgroups take tile ids with a fixed stride -- so with 192 tiles per group and 256 workgroups each
// workgroup misses every fourth group, and which fourth decides its load.  The tile space therefore runs over the
// groups in order of decreasing token count (ties by index): the sums over every fourth group of a sorted sequence
// differ by less than the largest group, and the launch ends on its cheapest tiles.  t.tile0[i] = the group whose
// tiles come i-th.  Position of group g = number of groups that precede it in that order.
template <class Table>
TGG_HD int sched_group_rank(const Table& t, int G, int g) {
  const int32_t mine = t.rows[g];
  int rank = 0;
  for (int h = 0; h < G; ++h) {
    const int32_t other = t.rows[h];
    rank += (other > mine) || (other == mine && h < g);
  }
  return rank;
}

// Serial form (host hook, and kernels whose workgroups have fewer threads than there are groups).
template <class Table>
TGG_HD void sched_order_groups_serial(const GemmParams& p, Table& t) {
  for (int g = 0; g < p.G; ++g) t.tile0[sched_group_rank(t, p.G, g)] = g;
}

// Inclusive prefix sum over the wave's lanes, by moves between lanes inside the vector unit: within a row of sixteen first, then
// the rows' totals.  (Exchanges through LDS take six dependent round trips of over a hundred cycles instead.)
TGG_DEV int64_t sched_wave_scan(int64_t v) {
#define TGG_SCAN_STEP(ctrl, rows) \
  { \
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, ctrl, rows, 0xf, false); \
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)((uint64_t)v >> 32), ctrl, rows, 0xf, false); \
    v += (int64_t)(((uint64_t)hi << 32) | lo); \
  }
  TGG_SCAN_STEP(0x111, 0xf)  // row_shr:1, 2, 4, 8: lanes whose source lies in front of the row add the zero
  TGG_SCAN_STEP(0x112, 0xf)
  TGG_SCAN_STEP(0x114, 0xf)
  TGG_SCAN_STEP(0x118, 0xf)
  TGG_SCAN_STEP(0x142, 0xa)  // row_bcast:15: a row's last lane to the next row, into rows 1 and 3
  TGG_SCAN_STEP(0x143, 0xc)  // row_bcast:31: lane 31 to rows 2 and 3
#undef TGG_SCAN_STEP
  return v;
}

// Exclusive prefix sum over the workgroup's threads (in thread order) and the total; all threads must call it.
// Wave-wide scans, the waves' totals through the table's scratch words.
template <class Table>
TGG_DEV int64_t sched_block_scan(int64_t v, Table& t, int64_t& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = ((int)blockDim.x + 63) >> 6;
  const int64_t inc = sched_wave_scan(v);
  if (lane == 63) t.scan_[wave] = inc;
  __syncthreads();
  int64_t base = 0, tot = 0;
  for (int w = 0; w < waves; ++w) {
    const int64_t s = t.scan_[w];
    if (w < wave) base += s;
    tot += s;
  }
  __syncthreads();  // the scratch words are free again
  total = tot;
  return base + inc - v;
}

// sched_prefix by the whole workgroup: every thread takes a run of neighbouring groups, the runs meet in two scans.  All
// threads must call this, with the loaded extents visible to them.  For the 1024-entry table of the shape-agnostic kernel,
// whose workgroups have fewer threads than there may be groups: one thread's serial pass is 0.15 us a group, half of a small
// launch again (K-grouped from sizes, outputs of 264 x 520 and 4 tokens a group: 1024 groups 502 -> 333 us, 600 groups 285 ->
// 186).  Same values.
template <int BM, class Table>
TGG_DEV void sched_prefix_runs(const GemmParams& p, Table& t) {
  const int per = (p.G + (int)blockDim.x - 1) / (int)blockDim.x;
  const int g0 = min(p.G, (int)threadIdx.x * per), g1 = min(p.G, g0 + per);
  auto step = [&](int64_t sz) { return p.mode == MODE_MG_PAD ? ((sz + p.align - 1) / p.align) * p.align : sz; };
  int64_t sum = 0, total;
  for (int g = g0; g < g1; ++g) sum += step(t.rows[g]);
  int64_t row = sched_block_scan(sum, t, total);
  const int64_t limit = (p.mode == MODE_KG_COUNT) ? p.k_total : p.m_total;
  sum = 0;
  for (int g = g0; g < g1; ++g) {
    int64_t sz = t.rows[g], start = row;
    row += step(sz);
    if (p.mode == MODE_MASKED) {
      start = (int64_t)g * p.m_stride;
      if (sz > p.m_stride) sz = p.m_stride;
    } else if (p.mode == MODE_MG_PAD && p.row_start) {
      start = (int64_t)p.row_start[g];
    }
    if (start < 0 || start >= limit) sz = 0;
    else if (start + sz > limit) sz = limit - start;
    t.row0[g] = start;
    t.rows[g] = (int32_t)sz;
    sum += (sz + BM - 1) / BM;
  }
  int64_t tile = sched_block_scan(sum, t, total);
  for (int g = g0; g < g1; ++g) {
    t.tile0[g] = (int32_t)tile;
    tile += (t.rows[g] + BM - 1) / BM;
  }
  if (threadIdx.x == 0) t.tile0[p.G] = (int32_t)total;
}

// K modes only (a no-op otherwise): fills t.tile0 with the groups in tile-space order once t.rows is final.  All
// threads of the workgroup must call this; ends with a barrier when it does anything.
template <class Table>
TGG_DEV void sched_order_groups(const GemmParams& p, Table& t) {
  if (p.mode != MODE_KG && p.mode != MODE_KG_COUNT) return;
  for (int g = threadIdx.x; g < p.G; g += blockDim.x) t.tile0[sched_group_rank(t, p.G, g)] = g;
  __syncthreads();
}

// Builds the table.  All threads of the workgroup must call this; ends with a barrier.
// With one thread per group (G <= workgroup size <= 1024) the two prefix sums of sched_prefix -- group starts, then
// tiles of the clipped sizes -- are workgroup-wide scans: about a microsecond, where the serial pass of one thread
// takes 0.2 us per group (15 us at 128 groups, a tenth of a decode-sized launch).  Same values as sched_prefix.
// The tile scan carries the prefix for tiles of half the height along in its upper word: the calling thread's group
// would start at the returned tile id under that cut, and t.pad_ receives how many tiles more that cut has in all
// (see sched_use_half_height).  With more groups than threads the serial pass (or sched_prefix_runs) takes the place of the
// scans, and t.pad_ is set so large that no caller prefers the half-height cut.
template <int BM, class Table>
TGG_DEV int32_t sched_init(const GemmParams& p, Table& t) {
  if (p.mode == MODE_KG || p.G > (int)blockDim.x || blockDim.x > 1024) {
    for (int g = threadIdx.x; g < p.G; g += blockDim.x) sched_load_group(p, t, g);
    __syncthreads();
    if (p.mode != MODE_KG) {
      if constexpr (std::is_same<Table, SchedTable>::value) sched_prefix_runs<BM>(p, t);
      else if (threadIdx.x == 0) sched_prefix<BM>(p, t);
      if (threadIdx.x == 0) t.pad_ = 1 << 30;
      __syncthreads();
    }
    sched_order_groups(p, t);
    return 0;
  }
  const int g = threadIdx.x;
  const bool live = g < p.G;
  int64_t sz = live ? load_size(p.sizes, p.sizes_i64, g) : 0;
  int64_t start;
  if (p.mode == MODE_MASKED) {
    start = (int64_t)g * p.m_stride;
    if (sz > p.m_stride) sz = p.m_stride;
  } else {
    const int64_t step = (p.mode == MODE_MG_PAD) ? ((sz + p.align - 1) / p.align) * p.align : sz;
    int64_t all;
    start = sched_block_scan(step, t, all);
    if (p.mode == MODE_MG_PAD && p.row_start && live) start = (int64_t)p.row_start[g];
  }
  const int64_t limit = (p.mode == MODE_KG_COUNT) ? p.k_total : p.m_total;
  if (start < 0 || start >= limit) sz = 0;  // never touch rows (or k) outside the operands (a negative start can only come from row_start)
  else if (start + sz > limit) sz = limit - start;
  constexpr int HALF = BM / 2;
  int64_t total;
  const int64_t both = sched_block_scan((sz + BM - 1) / BM + (((sz + HALF - 1) / HALF) << 32), t, total);
  if (live) {
    t.row0[g] = start;
    t.rows[g] = (int32_t)sz;
    t.tile0[g] = (int32_t)(both & 0xffffffff);
  }
  if (threadIdx.x == 0) {
    t.tile0[p.G] = (int32_t)(total & 0xffffffff);
    t.pad_ = (int32_t)(total >> 32) - (int32_t)(total & 0xffffffff);
  }
  __syncthreads();
  sched_order_groups(p, t);
  return (int32_t)(both >> 32);
}

// Switches a table built by sched_init<BM> to tiles of half that height: half_tile0 is what sched_init returned
// to this thread.  All threads of the workgroup must call this; starts and ends with a barrier (other threads may
// still be reading the totals that it overwrites).
template <class Table>
TGG_DEV void sched_use_half_height(const GemmParams& p, Table& t, int32_t half_tile0) {
  __syncthreads();
  if ((int)threadIdx.x < p.G) t.tile0[threadIdx.x] = half_tile0;
  if (threadIdx.x == 0) t.tile0[p.G] += t.pad_;
  __syncthreads();
}

// K-grouped by counts, known from them alone and in front of the table: whether the shape-agnostic launch has nothing to do (a count that
// is clipped stays a multiple of 16 where all of them are; what this leaves open sched_kg_gate_open decides).  The launch that
// returns costs 2 us less without the table: 4 groups of 512 x 1024, 128 tokens each 22.9 -> 21.0 us, 128 of 264 x 520 40.5 -> 35.8.
TGG_DEV bool sched_kg_gate_shut(const GemmParams& p) {
  if (p.kg_gate != 2) return false;
  int bad = 0;
  for (int g = threadIdx.x; g < p.G; g += blockDim.x) bad |= ((int)load_size(p.sizes, p.sizes_i64, g) & 15) != 0;
  return __syncthreads_count(bad) == 0;
}

// K-grouped by counts: does the launch pass its gate (GemmParams::kg_gate)?  All threads of the workgroup must call
// this after sched_init; the answer is the same in every workgroup of the launch.
template <class Table>
TGG_DEV bool sched_kg_gate_open(const GemmParams& p, const Table& t) {
  if (p.kg_gate == 0) return true;
  int bad = 0;
  for (int g = threadIdx.x; g < p.G; g += blockDim.x) bad |= (t.rows[g] & 15) != 0;
  const int n_bad = __syncthreads_count(bad);
  return p.kg_gate == 1 ? n_bad == 0 : n_bad != 0;
}

template <int BM, int BN, class Table>
TGG_HD int64_t sched_num_tiles(const GemmParams& p, const Table& t) {
  const int tiles_n = (p.N + BN - 1) / BN;
  if (p.mode == MODE_KG || p.mode == MODE_KG_COUNT) {
    const int tiles_m = (int)((p.m_total + BM - 1) / BM);
    return (int64_t)p.G * tiles_m * tiles_n;
  }
  return (int64_t)t.tile0[p.G] * tiles_n;
}

// Whether tiles of half the table's tile height pay for an M-grouped launch.  t.pad_ holds the tiles that the half
// height cut has over the table's cut (sched_init leaves it there).  The persistent workgroups work in rounds (one
// tile each per round), a half-height tile costs cost_half / cost_full of a full one (the eight-wave kernels: 0.7, measured over group counts 8-256 and
// 64-2048 rows per group, for both operand widths), and what decides is whole rounds: a launch whose full-height
// tiles just fit one round loses by going to two rounds of short tiles, whatever their number.
template <int BN, class Table>
__device__ __forceinline__ bool sched_short_tiles_pay(const GemmParams& p, const Table& t, int cost_full, int cost_half) {
  const int64_t tiles_n = (p.N + BN - 1) / BN, wgs = gridDim.x;
  const int64_t rounds_full = ((int64_t)t.tile0[p.G] * tiles_n + wgs - 1) / wgs;
  const int64_t rounds_half = ((int64_t)(t.tile0[p.G] + t.pad_) * tiles_n + wgs - 1) / wgs;
  return rounds_half * cost_half <= rounds_full * cost_full;
}

// Whether a launch that the four-wave kernel may take is its: 256-row tiles that are neither few enough for the narrow tiles (all
// of them fit one round of the persistent workgroups) nor of groups so small that the eight-wave kernels' 128-row tiles pay.  Such
// a tile costs three quarters of the four-wave kernel's.  Measured over 16-128 groups of 64-511 rows, seven
// pairs of N and K, 357 launches, time of the four-wave kernel over the eight-wave kernels' by rounds of short over rounds of
// full tiles: 1.0-1.1 1.08-1.19, 1.2-1.3 1.0-1.04, 1.4-1.5 0.93-0.99, 1.6 and more 0.91-0.97.  (With the 0.7 of
// sched_short_tiles_pay for the eight-wave kernels' own 256-row tiles, ratios of 1.33-1.43 went to the slower side: 128
// groups of 256 rows on average, N = 2048, K = 1536, B as [G, K, N]: 297 -> 270 us; N = 2048, K = 768: 165 -> 150 us.)
// t: a table built by sched_init<BM> with one thread per group.
template <int BM, int BN, class Table>
__device__ __forceinline__ bool sched_wide_tiles_chosen(const GemmParams& p, const Table& t) {
  return sched_num_tiles<BM, BN / 2>(p, t) > (int64_t)gridDim.x && !sched_short_tiles_pay<BN>(p, t, 4, 3);
}

// Tile order.  Consecutive tile ids are handed to workgroups that run at the same time on one XCD
// (see sched_walk), so a run of ids should cover a near-square block of tiles: a run of R tiles spanning
// w column tiles touches R / w row panels of A plus w column panels of B per K slab.  The N tiles are
// therefore cut into chunks of at most eight columns and ids run over (chunk, row tile, column within
// chunk), innermost last.  Eight rather than the square root of an XCD's 32 workgroups: B panels
// (weights) are reused by the following row tiles of the group, A panels are streamed once, so the
// wider side goes to B.
TGG_HD int sched_chunk_width(int tiles_n, int n_chunk) {
  if (n_chunk > 0) return n_chunk < tiles_n ? n_chunk : tiles_n;
  const int chunks = (tiles_n + 7) / 8;
  return (tiles_n + chunks - 1) / chunks;
}

// Splits the position `r` inside a block of `rows_m` row tiles x `tiles_n` column tiles into (row tile, column tile).
TGG_HD void sched_split(int r, int rows_m, int tiles_n, int nc, int& mt, int& nt) {
  const int chunk_tiles = rows_m * nc;
  int c = r / chunk_tiles;
  const int full = tiles_n / nc;
  int width = nc;
  if (c >= full) {  // the last, narrower chunk
    c = full;
    width = tiles_n - full * nc;
  }
  const int q = r - c * chunk_tiles;
  mt = q / width;
  nt = c * nc + (q - mt * width);
}

// Row-tile lookup shared by every consumer of the group table (every mode but the K-grouped ones): which group
// owns the global BM-row tile `mt_glob` (counted over the groups' tiles in order, independent of the tile-id
// order that sched_tile lays over the (row tile, column tile) space), where its rows start and how many are valid.
// g_hint: a group at or before the tile's group, if the caller knows one (a workgroup's walk visits tiles in
// increasing order, and within a column chunk their groups never decrease): the lookup then checks the hinted
// group and its successor before it falls back to the binary search, each probe being a dependent LDS read.
struct RowTile {
  int g;
  int64_t row0;
  int rows;
};

template <int BM, class Table>
TGG_HD RowTile sched_row_tile(const Table& t, int G, int mt_glob, int g_hint = -1) {
  int lo = 0, hi = G;  // last g with tile0[g] <= mt_glob
  if (g_hint >= 0 && g_hint < G && t.tile0[g_hint] <= mt_glob) {
    lo = g_hint;
    if (t.tile0[lo + 1] > mt_glob) hi = lo + 1;            // tile0 has G + 1 entries
    else if (lo + 2 <= G && t.tile0[lo + 2] > mt_glob) { lo = lo + 1; hi = lo + 1; }
    else lo = lo + 1;                                      // further on: search [lo, G)
  }
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (t.tile0[mid] <= mt_glob) lo = mid; else hi = mid;
  }
  RowTile r;
  r.g = lo;
  const int mt = mt_glob - t.tile0[lo];
  r.row0 = t.row0[lo] + (int64_t)mt * BM;
  const int left = t.rows[lo] - mt * BM;
  r.rows = left < BM ? left : BM;
  return r;
}

template <int BM, int BN, class Table>
TGG_HD Tile sched_tile(const GemmParams& p, const Table& t, int64_t tile_id, int g_hint = -1) {
  Tile r;
  const int tiles_n = (p.N + BN - 1) / BN;
  const int nc = sched_chunk_width(tiles_n, p.n_chunk);
  const int tid32 = (int)tile_id;  // the tile space is far below 2^31; 32-bit division is much cheaper
  if (p.mode == MODE_KG || p.mode == MODE_KG_COUNT) {
    const int tiles_m = (int)((p.m_total + BM - 1) / BM);
    const int per_group = tiles_m * tiles_n;
    const int slot = tid32 / per_group;
    r.g = t.tile0[slot];  // groups in order of decreasing size, see sched_group_rank
    int mt, nt;
    sched_split(tid32 - slot * per_group, tiles_m, tiles_n, nc, mt, nt);
    r.n0 = nt * BN;
    r.row0 = (int64_t)mt * BM;
    const int64_t left = p.m_total - r.row0;
    r.rows = left < BM ? (int)left : BM;
    r.k0 = t.row0[r.g];
    r.k1 = r.k0 + t.rows[r.g];
    return r;
  }
  int mt_glob, nt;
  sched_split(tid32, t.tile0[p.G], tiles_n, nc, mt_glob, nt);
  const RowTile rt = sched_row_tile<BM>(t, p.G, mt_glob, g_hint);
  r.n0 = nt * BN;
  r.g = rt.g;
  r.row0 = rt.row0;
  r.rows = rt.rows;
  r.k0 = 0;
  r.k1 = p.K;
  return r;
}

// Persistent walk of the tile space by workgroup b of P.  Consecutive workgroup ids land on
// different XCDs (round robin over 8), each with its own L2, so the walk is laid out per XCD:
//   split = true   XCD x owns the contiguous tile range [x*T/8, (x+1)*T/8) and its P/8 workgroups
//                  sweep it in runs of P/8 neighbouring tiles.  Neighbours share activation rows and
//                  expert weights, and an expert's weights are fetched by one or two XCDs only.
//                  Right when all tiles cost the same (M-grouped: K is fixed).
//   split = false  every sweep hands each XCD a run of P/8 neighbouring tiles, sweeps interleaved over
//                  the whole space.  Used when tile cost varies along the tile order (K-grouped:
//                  cost follows the group's token count), so that every XCD sees every group.
struct TileWalk {
  int64_t first, end, stride;
};

TGG_HD TileWalk sched_walk_of(int64_t num_tiles, bool split, int P, int b) {
  TileWalk w;
  if ((P & 7) != 0) {
    w.first = b; w.end = num_tiles; w.stride = P;
  } else if (split) {
    const int x = b & 7;
    w.first = (num_tiles * x) / 8 + (b >> 3);
    w.end = (num_tiles * (x + 1)) / 8;
    w.stride = P >> 3;
  } else {
    w.first = (int64_t)(b & 7) * (P >> 3) + (b >> 3);
    w.end = num_tiles;
    w.stride = P;
  }
  return w;
}

TGG_DEV TileWalk sched_walk(int64_t num_tiles, bool split) {
  return sched_walk_of(num_tiles, split, (int)gridDim.x, (int)blockIdx.x);
}

// The tile id behind the n-th draw from XCD xq's counter (R = workgroups per XCD): run n / R of that XCD, which is run
// xq of the deal's pass n / R when the pass runs forwards (even) and run 7 - xq when it runs backwards.
TGG_HD int sched_queue_id(int n, int xq, int R) {
  const int pass = n / R;
  return (pass * 8 + ((pass & 1) ? 7 - xq : xq)) * R + n % R;
}

// Lane x < 8 holds the value of XCD x's counter.  Bit x of the result: that counter's next draw stands for a tile (a counter
// only grows: one that has been seen exhausted stays so).  The whole wave calls it.
TGG_DEV int sched_queue_left(int seen, int total, int R) {
  const int x = lane_id();
  return (int)(uint32_t)__ballot(x < 8 && sched_queue_id(seen, x & 7, R) < total);
}

// The first counter behind `own` (in ring order) among those of the mask `left` (not empty).
TGG_HD int sched_queue_next(int left, int own) {
  const int turned = ((left >> own) | (left << (8 - own))) & 0xff;  // bit d: counter own + d
  return (own + __builtin_ctz(turned)) & 7;
}

// Work queue of the K-grouped tuned kernels: eight counters in global memory, one per XCD (zero at launch).  The
// tile space is cut into runs of R neighbouring tiles (R = workgroups per XCD; neighbours are tiles of one group,
// which share operand panels in an XCD's L2), and the runs are dealt to the XCDs in order of decreasing cost, back
// and forth (0..7, 7..0, ...) so that no XCD always gets the dearest of eight.  Within an XCD a tile goes to
// whichever workgroup asks next: like the static interleaved walk the XCD works through runs of neighbours, but a
// workgroup that drew expensive tiles draws fewer.  A workgroup whose own XCD has nothing left looks at all
// counters at once and goes on with the next one in ring order that has tiles, until none has: what the deal leaves uneven is
// evened out at the end.  (Finding them exhausted by a draw from one counter after the other takes seven more round
// trips at the end of every launch, half of a small one: bf16, 4 groups of 2048 x 1536, 64 / 256 / 1024 tokens a group 38 / 40 / 56
// -> 20 / 25 / 56 us; FP8, 4 groups of 768 x 2048, 128 / 1024 tokens 46 / 46 -> 27 / 37 us.)  For every counter the ids grow with the number of draws, so one id at or beyond `total` means that counter is exhausted.
//
// One wave of each workgroup draws for it.  A draw costs a round trip to the counter (about a microsecond), which on
// tiles of a slab or two is as long as the tile, so it is requested at the start of a slab and taken at the slab's
// own wait for its copies, in front of the barrier; only when the copy stream is about to run out of drawn tiles does
// the wave draw on the spot.  It draws when fewer than kAhead slabs are drawn and not yet requested by the copy
// stream, so a workgroup commits itself to its next expensive tile a few slabs before it needs it and not earlier:
// committing to several is what spoils the balance when a workgroup has only a dozen tiles in all.  Measured against a
// draw on the spot per tile, 128 groups of 2048 x 1536 outputs: bf16, 64 / 256 / 1024 tokens per group 203 / 303 / 853 ->
// 167 / 285 / 819 us (4096: the same), FP8, 128 / 256 / 1024 tokens 241 / 258 / 586 -> 199 / 224 / 582 us.  kAhead 2, 4, 8:
// FP8 at 128 tokens 222, 206, 199 us, no difference at 4096.  The branches are marked unlikely: laid out inside the
// slab loop they cost 1-1.5 % of a long FP8 launch.
template <int BM, int BN, class Table>
struct QueueDraw {
  static constexpr int kRing = 16;  // > tiles between the one in work and the last drawn: 3 + kAhead one-slab tiles
  static constexpr int kAhead = 8;
  const GemmParams& p;
  Table& t;
  const int total, slab_k;
  int ahead = 0;             // slabs drawn and not yet requested by the copy stream (kept by every wave's begin_slab, read by the drawing wave)
  int drawn = 0, xq;          // tiles drawn; the counter to draw from
  int exhausted = 0;          // counters that a draw has found without a tile, one bit each
  int looking = 0;            // 1: the next request does not draw but asks for the values of all eight counters
  int live;                   // 1 in the wave that draws, until it has put the end marker in the ring (integers, not
                              // truth values, so that they stay in scalar registers)
  int answer;                 // the counters' values once the wave's memory operations have been waited for

  TGG_DEV QueueDraw(const GemmParams& p_, Table& t_, int total_, int slab_k_, bool drawing)
      : p(p_), t(t_), total(total_), slab_k(slab_k_), xq((gridDim.x & 7) == 0 ? (int)(blockIdx.x & 7) : 0), live(drawing ? 1 : 0) {}

  TGG_DEV int32_t& ring(int pos) { return reinterpret_cast<int32_t*>(t.scan_)[pos & (kRing - 1)]; }
  TGG_DEV bool spread() const { return (gridDim.x & 7) == 0; }  // eight counters; else one
  TGG_DEV int wanted() { live = __builtin_amdgcn_readfirstlane(live); return ahead < kAhead ? live : 0; }
  // begin_slab has requested a slab of the tile (issued < slabs: there was one left)
  TGG_DEV void count(int issued, int slabs) { ahead -= (int)((uint32_t)(issued - slabs) >> 31); }

  // the answer to a request (a value per lane)
  TGG_DEV void accept(int value) {
    const int R = (int)gridDim.x >> 3;
    bool end = false;
    if (__builtin_expect(looking, 0)) {
      const int left = sched_queue_left(value, total, R) & ~exhausted;
      looking = 0;
      end = left == 0;
      if (!end) xq = sched_queue_next(left, xq);
    } else {
      const int n = __builtin_amdgcn_readfirstlane(value);
      const int id = spread() ? sched_queue_id(n, xq, R) : n;
      if (id < total) {
        const int per_group = (int)((p.m_total + BM - 1) / BM) * ((p.N + BN - 1) / BN);
        const int rows = __builtin_amdgcn_readfirstlane(t.rows[t.tile0[id / per_group]]);
        ring(drawn++) = id;
        ahead += rows > 0 ? (rows + slab_k - 1) / slab_k : 1;  // an empty group's tile has one slab of nothing
      } else {
        exhausted |= 1 << xq;
        looking = spread();
        end = !looking;
      }
    }
    if (end) {
      ring(drawn++) = total;
      live = 0;
    }
  }

  // lane 0 draws from the current counter, or (looking) lanes 0-7 read one counter each
  TGG_DEV int ask() {
    const int lane = lane_id();
    int value = 0;
    // The address is made a lane's own: for one that the wave shares the compiler merges the lanes' additions and reads
    // the result back on the spot, which is the wait that a request is to avoid.
    int at = looking ? (lane & 7) : xq;
    asm("" : "+v"(at));
    if (lane < (looking ? 8 : 1)) value = __hip_atomic_fetch_add(p.queue + at, looking ? 0 : 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return value;
  }

  TGG_DEV void draw_now() { accept(ask()); }

  TGG_DEV void first() { while (wanted()) draw_now(); }

  // `answer` is in flight until take().  A builtin, so that the compiler knows of the register in flight and waits wherever it
  // might touch it.
  TGG_DEV void request() { answer = ask(); }

  // The drawing wave, after it has waited for all of its memory operations and in front of a workgroup barrier.
  TGG_DEV void take(int requested) {
    asm volatile("" : "+v"(answer));  // arrived: not to be read any earlier than here
    if (__builtin_expect(requested, 0)) accept(answer);
    while (__builtin_expect(ahead <= 1 && live, 0)) draw_now();  // the next slab's request may ask for the next tile
  }
};

// End of a queued launch: every workgroup reports here once it has drawn its last id (the draw that found all eight
// counters exhausted has returned by then), and the workgroup that reports last puts the nine words back to zero, so
// that the next launch on the same stream finds the queue as this one found it.  Thread 0 of each workgroup calls it.
constexpr int kQueueDoneWord = 8;
TGG_DEV void sched_queue_finish(int32_t* queue) {
  if (atomicAdd(queue + kQueueDoneWord, 1) == (int)gridDim.x - 1) {
    for (int i = 0; i <= kQueueDoneWord; ++i) atomicExch(queue + i, 0);
  }
}

}  // namespace tgg
