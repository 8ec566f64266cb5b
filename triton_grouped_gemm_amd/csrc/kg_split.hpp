// K-grouped launches of few tiles and long segments (weight gradients of small outputs over many tokens), cut along K: a segment
// is computed in parts, each tile of a part by a workgroup of its own, the parts' fp32 sums go to a workspace and a second
// kernel adds them up in order and rounds once.  How long a part is depends on the sizes, so the device decides (split_plan);
// the same sizes on as many workgroups give the same parts, hence the same bits.
#pragma once
#include "launch.hpp"
#include "w4_common.hpp"

namespace tgg {

constexpr int kSplitHeadBytes = 4096;           // in front of the workspace's slots: {first slot, parts} of each group, parts <= 1: not split
constexpr int kSplitTileBytes = 256 * 256 * 4;  // a tile of a part: wave by wave, 16x16 block by block, 16 bytes a lane
static_assert(kFastMaxGroups * 8 <= kSplitHeadBytes, "a pair of integers per group");

// Costs in units of U tokens along K: what a tile costs beyond its steps, what a tile of a part costs to be written and read back
// with all CUs at it, and what the adding kernel costs besides.
template <int U, int TILE_COST, int PART_COST, int SUM_COST> struct SplitCost {
  static constexpr int U_TOKENS = U, TILE = TILE_COST, PART = PART_COST, SUM = SUM_COST;
};

// ceil(a / b) for 0 <= a < 2^26 and 1 <= b < 2^26, by a reciprocal and its corrections: an integer division is four times as many instructions, and
// a plan makes one for every group.  The estimate is off by less than 2^-21 of the quotient and one; its remainder over b makes that one at most.
TGG_DEV int split_div_up(int a, int b) {
  const float r = __builtin_amdgcn_rcpf((float)b);
  const int x = a + b - 1;
  int q = (int)((float)x * r);
  q += (int)((float)(x - q * b) * r);
  const int left = x - q * b;
  return q + (left >= b ? 1 : 0) - (left < 0 ? 1 : 0);
}

// The smallest of the workgroup's values (256 threads, all of which must call this).
template <class Table>
TGG_DEV int64_t split_block_min(int64_t v, Table& t) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int64_t o = __shfl_xor(v, d, 64);
    v = o < v ? o : v;
  }
  if ((threadIdx.x & 63) == 0) t.scan_[threadIdx.x >> 6] = v;
  __syncthreads();
  for (int w = 0; w < 4; ++w) v = t.scan_[w] < v ? t.scan_[w] : v;
  __syncthreads();
  return v;
}

// Turns the group table (sched_init) into one of segment parts and returns their number: t.rows / t.row0 / t.tile0 per part, and in
// meta the part's group and, plus one, its slot of the workspace (0: the group is in one part and is written directly).  Every workgroup comes to
// the same table; workgroup 0 leaves the slots in the workspace's head.  All threads (256, no fewer than groups) must call this.
//
// Tiles are drawn longest first, so a launch takes an even share of the work or, for some k, k + 1 of its tile number k P + 1 in that order:
// that is what an uncut launch is expected to take.  Part lengths: the best of 256 candidates, one per thread, from a
// quarter of an even share to four of them; expected are an even share or the rounds that the tiles of more than half that length make;
// a cut is made for a twelfth of the time at least.
// Every candidate is a look at all groups, and every workgroup makes the plan.  With a read from LDS and two integer divisions per group that took 0.16 us a group in front
// of the launch; with the groups in lanes' registers, runs of equal ones counted at once and the divisions by reciprocals (the same plan) 0.01-0.08.
// 53 groups of 376 x 1192, 2180 tokens each (nothing to cut) 189 -> 180 us, 173 by a launch that does not ask; 200 of 264 x 264, 512000 tokens, equal 284 -> 250,
// unequal 323 -> 270; 108 of 80 x 136, 3738 tokens 175 -> 102.
template <class Cost, class Table>
TGG_DEV int split_plan(const GemmParams& p, Table& t, int32_t* meta, int tiles_per_group) {
  const int tid = threadIdx.x, lane = lane_id(), G = p.G, P = (int)gridDim.x;
  constexpr int U = Cost::U_TOKENS, kNever = 0x3fffffff;
  const int my_rows = tid < G ? t.rows[tid] : 0;
  const int my_steps = (my_rows + U - 1) / U;
  const int64_t my_row0 = tid < G ? t.row0[tid] : 0;
  int64_t total;
  (void)sched_block_scan((int64_t)my_steps, t, total);
  const int share = (int)((total * tiles_per_group + P - 1) / P);
  const int ranked = tid * P / tiles_per_group;  // (at most 255 rounds count)
  const int uncut_k = ranked < G ? (tid + 1) * ((t.rows[t.tile0[ranked]] + U - 1) / U) : 0;
  int uncut = -(int)split_block_min((int64_t)-uncut_k, t);
  uncut = uncut > share ? uncut : share;
  int64_t best = (int64_t)kNever << 32;
  if (uncut > share + Cost::SUM + Cost::TILE) {  // (uniform)
    // factor 2^(e - 2) * (1 + f / 64)
    const int e = tid >> 6, f = tid & 63;
    int c = (int)(((int64_t)share * (64 + f)) >> (8 - e));
    if (c < 8) c = 8;
    const FixedDiv by_c(c);
    const int c_least = __builtin_amdgcn_readfirstlane(c);  // of the wave's candidates
    int parts = 0, slots = 0, longest = 0, n_long = 0, sum_long = 0, run = 0, seen = 0;
    auto count = [&]() __attribute__((always_inline)) {  // `run` groups of `seen` steps
      int n = 1, len = seen;
      if (seen > c_least && seen > c) {
        n = (int)by_c.div((uint32_t)(seen + c - 1));
        len = split_div_up(seen, n);
        slots += n * run;
      }
      parts += n * run;
      longest = len > longest ? len : longest;
      if (2 * len > c) { n_long += n * run; sum_long += seen * run; }
    };
    for (int g0 = 0; g0 < G; g0 += 64) {  // a lane's group each, then one after the other from the lanes' registers
      const int mine = g0 + lane < G ? (t.rows[g0 + lane] + U - 1) / U : 0, in = G - g0 < 64 ? G - g0 : 64;
      for (int i = 0; i < in; ++i) {
        const int steps = __builtin_amdgcn_readlane(mine, i);
        if (steps != seen) {  // (uniform)
          count();
          seen = steps;
          run = 0;
        }
        ++run;
      }
    }
    count();
    const int64_t tiles = (int64_t)parts * tiles_per_group, rounds_long = ((int64_t)n_long * tiles_per_group + P - 1) / P;
    int64_t expected = n_long > 0 ? rounds_long * sum_long / n_long : 0;
    if (expected < share) expected = share;
    if (expected < longest) expected = longest;
    expected += (tiles + P - 1) / P * Cost::TILE + ((int64_t)slots * tiles_per_group * Cost::PART + P - 1) / P + Cost::SUM;
    const bool pays = slots > 0 && slots <= p.split_slots && parts <= kFastMaxGroups &&
                      expected + expected / 12 < uncut + (int64_t)(G * tiles_per_group + P - 1) / P * Cost::TILE;
    best = split_block_min(((pays && expected < kNever ? expected : kNever) << 32) | (uint32_t)tid, t);  // the first of equals
  }
  const int who = (int)(best & 0xff), we = who >> 6, wf = who & 63;
  int c = (int)(((int64_t)share * (64 + wf)) >> (8 - we));
  if (c < 8) c = 8;
  const bool any = (best >> 32) < kNever;  // else there are no parts
  const int n = !any || my_steps <= c ? 1 : (my_steps + c - 1) / c;
  const int per = (my_steps + n - 1) / n * U;  // tokens of a part, the last one's may be fewer
  int64_t all;
  const int64_t at = sched_block_scan(tid < G ? (int64_t)n | ((int64_t)(n > 1 ? n : 0) << 32) : 0, t, all);
  const int first = (int)(at & 0xffffffff), slot0 = (int)(at >> 32);
  if (tid < G) {
    for (int q = 0; q < n; ++q) {
      const int left = my_rows - q * per;
      t.row0[first + q] = my_row0 + q * per;
      t.rows[first + q] = left < per ? left : per;
      meta[first + q] = tid | ((n > 1 ? slot0 + q + 1 : 0) << 16);
    }
    if (blockIdx.x == 0) {
      int32_t* const head = reinterpret_cast<int32_t*>(p.split_ws) + 2 * tid;
      head[0] = slot0;
      head[1] = n;
    }
  }
  const int V = (int)(all & 0xffffffff);
  if (V == G) {  // as before
    __syncthreads();
    return V;
  }
  __syncthreads();
  for (int v = tid; v < V; v += (int)blockDim.x) t.tile0[sched_group_rank(t, V, v)] = v;
  __syncthreads();
  return V;
}

// A wave's block of a finished tile of a part, from the accumulators to tile `at` of the workspace.  Behind the tile's last K step, whose last
// multiplies may have just been issued.
TGG_DEV void store_part(f32x4_t (&acc)[8][8], float* ws, int64_t at, int wave, int lane) {
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
  const i32x4_t r = make_rsrc32((uint64_t)ws + kSplitHeadBytes + (uint64_t)(at * kSplitTileBytes + wave * (kSplitTileBytes / 4)), kSplitTileBytes / 4);
  asm volatile("s_nop 4" : : "s"(r));
  int v = lane * 16;
  for_each<16>([&](auto Qc) __attribute__((always_inline)) {
    constexpr int q = decltype(Qc)::value, i = q / 2, j = q % 2 * 4;
    asm volatile("buffer_store_dwordx4 %0, %4, %5, 0 offen\n\tbuffer_store_dwordx4 %1, %4, %5, 0 offen offset:1024\n\t"
                 "buffer_store_dwordx4 %2, %4, %5, 0 offen offset:2048\n\tbuffer_store_dwordx4 %3, %4, %5, 0 offen offset:3072\n\ts_nop 1"
                 : : "a"(acc[i][j]), "a"(acc[i][j + 1]), "a"(acc[i][j + 2]), "a"(acc[i][j + 3]), "v"(v), "s"(r) : "memory");
    v += 4096;
  });
}

// Adds the parts up in order, one wave per 16 rows of a wave's block, rounds and writes the outputs.  FP8: the layout and the scales of fp8_w4.hip
// (a lane has four rows of eight neighbouring columns), else gemm_wgrad.hip's (one row, four columns of each block).
template <int OUT, bool FP8>
__global__ __launch_bounds__(256) void split_sum_kernel(const GemmParams p) {
  const int tiles_n = (p.N + 255) >> 8, per_group = (int)((p.m_total + 255) >> 8) * tiles_n;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, lg = lane >> 4;
  const int tile = blockIdx.x >> 3, i = blockIdx.x & 7, g = tile / per_group, at = tile - g * per_group;
  const int32_t* const head = reinterpret_cast<const int32_t*>(p.split_ws) + 2 * g;
  const int parts = __builtin_amdgcn_readfirstlane(head[1]), slot = __builtin_amdgcn_readfirstlane(head[0]);
  if (parts <= 1) return;
  const int m0 = (at / tiles_n) * 256 + (wave >> 1) * 128 + 16 * i, n0 = (at % tiles_n) * 256 + (wave & 1) * 128;
  if (m0 >= p.m_total || n0 >= p.N) return;
  const f32x4_t* src = reinterpret_cast<const f32x4_t*>(reinterpret_cast<const char*>(p.split_ws) + kSplitHeadBytes +
                                                        ((int64_t)slot * per_group + at) * kSplitTileBytes) + wave * 4096 + i * 512 + lane;
  f32x4_t sum[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) sum[j] = src[j * 64];
  for (int q = 1; q < parts; ++q) {
    src += (int64_t)per_group * (kSplitTileBytes / 16);
#pragma unroll
    for (int j = 0; j < 8; ++j) sum[j] += src[j * 64];
  }
  uint16_t* const out = reinterpret_cast<uint16_t*>(p.C) + (int64_t)g * p.m_total * p.N;
  if (FP8) {
    const int col = n0 + 8 * l16;
    if (col >= p.N) return;
    const float* const sn = p.scale_n + (int64_t)g * p.N + col;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + 4 * lg + r;
      if (row >= p.m_total) break;
      const float sm = p.scale_m[g * p.scale_m_sg + row];
      uint4 v;
      v.x = pack2<OUT>(sum[0][r] * sm * sn[0], sum[1][r] * sm * sn[1]);
      v.y = pack2<OUT>(sum[2][r] * sm * sn[2], sum[3][r] * sm * sn[3]);
      v.z = pack2<OUT>(sum[4][r] * sm * sn[4], sum[5][r] * sm * sn[5]);
      v.w = pack2<OUT>(sum[6][r] * sm * sn[6], sum[7][r] * sm * sn[7]);
      *reinterpret_cast<uint4*>(out + (int64_t)row * p.N + col) = v;
    }
  } else {
    const int row = m0 + l16;
    if (row >= p.m_total) return;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int col = n0 + 16 * j + 4 * lg;
      if (col < p.N) *reinterpret_cast<uint2*>(out + (int64_t)row * p.N + col) = pack4<OUT>(sum[j][0], sum[j][1], sum[j][2], sum[j][3]);
    }
  }
}

template <int OUT, bool FP8>
int launch_split_sum(const GemmParams& p, hipStream_t s) {
  const int64_t tiles = p.G * ((p.m_total + 255) / 256) * ((p.N + 255) / 256);
  hipLaunchKernelGGL((split_sum_kernel<OUT, FP8>), dim3((uint32_t)(tiles * 8)), dim3(256), 0, s, p);
  return check_launch("split_sum");
}

// Room for the parts: two rounds of tiles.
struct SplitRoom { int slots; int64_t bytes; };
inline SplitRoom split_room(const GemmParams& p) {
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  const int64_t per_group = ((p.m_total + 255) / 256) * ((p.N + 255) / 256);
  SplitRoom r;
  r.slots = (int)(2 * grid / per_group);
  r.bytes = kSplitHeadBytes + (int64_t)r.slots * per_group * kSplitTileBytes;
  return r;
}

// Bytes of workspace for a launch that may be cut along K, 0 where that does not pay.  The launch of the adding kernel costs 5 us where the sizes turn
// out to need no cut.  `gain`, in tokens: what a cut has to save for its parts to be written and added up.  With equal groups it saves what the
// last round of tiles lacks; with groups as a Dirichlet(1) draw deals them the largest has about ln G + 0.6 times the average, and
// the launch takes as long as that one.  The first alone decides where the launch is short, lest equal groups pay for nothing.
// The host does not know the sizes, so what unequal groups gain equal ones pay for.  Time with a cut offered over without, 800 random launches of 1-256
// groups: unequal ones 0.35 in the mean (16 bits, up to 1.04) and 0.32 (FP8, up to 1.02).  Equal ones 0.47 and 0.38 with up to 64 groups, 0.84 and 0.81 with 24-256; those in
// which the device finds nothing to cut pay 7 us, 1.01-1.06 in launches of 160 us and more.  Dearer is that what is not cut runs on the four-wave kernel also where the eight-wave
// one would be the faster: equal groups, 16 bits, few narrow tiles and a gain of 2000-3000 tokens up to 1.24 (108 groups of 80 x 136, 3738 tokens: 83 -> 102 us; unequal ones
// of that class 0.38-0.53), FP8, up to 256 columns, 1.02-1.17 (34 of 2080 x 96, 6524 tokens: 199 -> 234; unequal ones 0.48).
inline int64_t split_bytes(const GemmParams& p, int64_t gain, int64_t long_enough) {
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  const int64_t tiles = p.G * ((p.m_total + 255) / 256) * ((p.N + 255) / 256), tokens = p.k_total / p.G;
  const SplitRoom room = split_room(p);
  if (room.slots < 2 || tiles > 4 * grid) return 0;
  const int64_t rounds = (tiles + grid - 1) / grid, share = tokens * tiles / grid, equal = rounds * tokens - share;
  int log2_g = 0;
  while ((2 << log2_g) <= p.G) ++log2_g;
  const int64_t skewed = tokens * (69 * log2_g + 60) / 100 - share;
  return equal >= gain || (skewed >= gain && rounds * tokens >= long_enough) ? room.bytes : 0;
}

}  // namespace tgg
