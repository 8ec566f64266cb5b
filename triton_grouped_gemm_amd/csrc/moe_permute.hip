// MoE token permute / unpermute for gfx950: the steps either side of the grouped GEMMs that turn
// [tokens, hidden] activations plus a [tokens, topK] expert assignment into expert-contiguous rows and back.
//
// Sorting is a stable counting sort specialised to the key range (expert ids < 1024), not a general radix
// sort, and the per-expert row counts that the grouped GEMM takes as `size_per_group` fall out of it.  What bounds it
// is the number of dependent launches (4.6 us each behind one another, whatever they do), so it has as few as the
// size allows, and the row mover is the sort's own last step (with `in` / `out` null the map alone is made):
//   * up to kSmallAssignments assignments: one launch.  Every workgroup owns a run of tokens, counts all
//     assignments itself (in LDS, in total and in front of its run), ranks its own and moves its rows.  8192 indices
//     are 16 loads per thread; beyond that the repeated counting costs more than the launch it saves.
//   * more: count, then place and move.  count: each workgroup ranks a chunk of assignments (flat order
//     t * topK + k) and leaves the chunk's per-expert totals in table[chunk][e].  place: every workgroup owns a run
//     of tokens and sums the table's columns itself (in total for the experts' first rows, up to its chunk for its
//     own), which is cheaper than a launch while the table has at most kTableEntries entries; a larger table is
//     turned into prefixes by a launch in between.
// Ranks inside a wave come from one ballot per bit of the expert id (equal ids agree in every bit).
// destination = expert start + assignments of the expert in front; row_id_map[k * tokens + t] gets it (or -1 for
// dropped assignments: expert -1, or destination beyond the capacity).
//
//   * rows of more bytes than place_moves_rows says: the placing launch makes the map and a launch with a workgroup per token
//     moves the rows.  A thousand placing workgroups stream at 4.9 TB/s and the short ones at 5.6, which outweighs the launch
//     from 200 to 450 MiB read and written on; but the placing launch leaves more of its rows in the memory-side cache for the
//     call behind it, so the line is taken from whole passes (permute, unpermute and both gradients; moved by the placing
//     launch / by their own, rows of 4 KB, 128 experts, us):
//                   top-1        top-2        top-4        top-8
//       170 MiB    150 / 148    153 / 152    156 / 153    167 / 166
//       220        202 / 197    214 / 212    212 / 212    222 / 222
//       250        231 / 225    237 / 238    241 / 247    255 / 259
//       299        285 / 275    290 / 295    301 / 316    321 / 331
//     8 and 1024 experts and rows of 2 to 14 KB are alike.  Rows of 1 KB like the placing launch longer (top-1, 220 MiB 264 /
//     267, 299 351 / 348).  The permute alone, called over and over: 250 MiB 55.9 / 52.9, 54.3 / 54.0, 52.2 / 54.6, 59.9 / 55.0;
//     600 MiB 147 / 121, 138 / 126, 132 / 126, 140 / 126.
// Against four launches for the sort and one for the rows: 8192 tokens x top-8, 128 experts, 4 KB rows 70 -> 67 us, 81920
// tokens 589 -> 577, 4096 tokens 43 -> 29, 24 tokens 26 -> 4.4; top-1 to top-8 rows of 1 to 14 KB, 60 to 900 MiB: 0.54 to
// 0.96 of the time.
//
// The row movers are streaming kernels (16-byte accesses, fp32 arithmetic), bound by memory:
//   place           reads each token row once and writes it to its up to topK destinations
//   unpermute       out[t] = sum_k prob[t,k] * in[row_id_map[k,t]]
//   unpermute_bwd   act_grad[dest] = prob[t,k] * grad[t];  prob_grad[t,k] = <grad[t], fwd_in[dest]>
#include <mutex>

#include "common.hpp"
#include "launch.hpp"

namespace tgg {

namespace {

constexpr int kCountThreads = 1024;
constexpr int kMaxExperts = 1024;
constexpr int64_t kSmallAssignments = 8192;  // one-launch sort up to here
constexpr int64_t kTableEntries = 16384;     // the placing workgroups sum the count table themselves up to here
constexpr int kPlaceThreads = 512;
constexpr int kBatch = 1024;                 // assignments whose destinations a placing workgroup holds at a time

// Assignments per workgroup of the counting pass: as few as keep the table within kTableEntries, 1024 to 8192.
int64_t count_chunk(int64_t n, int num_experts) {
  int64_t chunk = kCountThreads;
  while (chunk < 8 * kCountThreads && ((n + chunk - 1) / chunk) * num_experts > kTableEntries) chunk *= 2;
  return chunk;
}

// Whether the placing workgroups move the rows too (see the top of the file): by the bytes read and written.
bool place_moves_rows(int64_t tokens, int topk, int64_t row_bytes) {
  const int64_t most = topk == 1 && row_bytes >= 2048 ? 200ll << 20 : 300ll << 20;
  return tokens * (topk + 1) * row_bytes <= most;
}

// The lanes of the wave whose (valid) key equals this lane's; keys below 2^bits.
TGG_DEV uint64_t match_lanes(int key, bool valid, int bits) {
  uint64_t same = __ballot(valid);
  for (int b = 0; b < bits; ++b) {
    const bool set = (key >> b) & 1;
    const uint64_t ones = __ballot(set);
    same &= set ? ones : ~ones;
  }
  return same;
}

TGG_DEV int lanes_before(uint64_t mask) { return __builtin_popcountll(mask & ((1ull << (threadIdx.x & 63)) - 1)); }

// table[chunk][e] = assignments of expert e in the chunk; rank[i] = rank of assignment i among the assignments of the
// same expert in its chunk, in flat order.  A wave takes chunk / 16 consecutive assignments, 64 at a time.
__global__ __launch_bounds__(kCountThreads) void moe_count_kernel(const int32_t* __restrict__ indices, int64_t n,
                                                                  int num_experts, int bits, int per_wave,
                                                                  int32_t* __restrict__ table, int32_t* __restrict__ rank) {
  constexpr int WAVES = kCountThreads / 64;
  extern __shared__ uint16_t wave_cnt[];  // [16 waves][num_experts]: at most per_wave each
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int x = tid; x < WAVES * num_experts; x += kCountThreads) wave_cnt[x] = 0;
  __syncthreads();
  uint16_t* const mine = wave_cnt + wave * num_experts;
  const int64_t i0 = ((int64_t)blockIdx.x * WAVES + wave) * per_wave;
  for (int j = lane; j < per_wave; j += 64) {
    const int64_t i = i0 + j;
    int e = i < n ? indices[i] : -1;
    const bool valid = e >= 0 && e < num_experts;  // anything else is a dropped assignment
    const uint64_t same = match_lanes(e, valid, bits);
    if (valid) {
      const int before = mine[e], ahead = lanes_before(same);
      rank[i] = before + ahead;
      if (ahead == 0) mine[e] = (uint16_t)(before + __builtin_popcountll(same));
    }
  }
  __syncthreads();
  // exclusive prefix over the waves, per expert; the chunk's total goes to the table
  for (int x = tid; x < num_experts; x += kCountThreads) {
    int run = 0;
    for (int w = 0; w < WAVES; ++w) {
      const int c = wave_cnt[w * num_experts + x];
      wave_cnt[w * num_experts + x] = (uint16_t)run;
      run += c;
    }
    table[(int64_t)blockIdx.x * num_experts + x] = run;
  }
  __syncthreads();
  for (int j = lane; j < per_wave; j += 64) {
    const int64_t i = i0 + j;
    const int e = i < n ? indices[i] : -1;
    if (e >= 0 && e < num_experts) rank[i] += mine[e];
  }
}

// Exclusive prefix sums, in place, of v[0 .. n); all threads of the workgroup, n <= 1024; lds: one int per wave.
template <int THREADS>
TGG_DEV void exclusive_scan_lds(int* v, int n, int* lds) {
  constexpr int PER = (kMaxExperts + THREADS - 1) / THREADS, WAVES = THREADS / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int x[PER], sum = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = tid * PER + j;
    x[j] = i < n ? v[i] : 0;
    sum += x[j];
  }
  int incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(incl, d, 64);
    if (lane >= d) incl += up;
  }
  if (lane == 63) lds[wave] = incl;
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < WAVES; ++w)
    if (w < wave) run += lds[w];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = tid * PER + j;
    if (i < n) v[i] = run;
    run += x[j];
  }
  __syncthreads();
}

// A table too large for the placing workgroups to sum: every column becomes exclusive prefixes over the chunks, its
// sum goes to totals[e].  64 experts per workgroup, the chunks in four runs.
__global__ __launch_bounds__(256) void moe_scan_table_kernel(int32_t* __restrict__ table, int chunks, int num_experts,
                                                             int32_t* __restrict__ totals) {
  __shared__ int run_sum[4][64];
  const int e = blockIdx.x * 64 + (threadIdx.x & 63), r = threadIdx.x >> 6;
  const int per = (chunks + 3) / 4, c0 = min(chunks, r * per), c1 = min(chunks, c0 + per);
  int sum = 0;
  if (e < num_experts)
    for (int c = c0; c < c1; ++c) sum += table[(int64_t)c * num_experts + e];
  run_sum[r][threadIdx.x & 63] = sum;
  __syncthreads();
  if (e >= num_experts) return;
  int run = 0;
  for (int q = 0; q < r; ++q) run += run_sum[q][threadIdx.x & 63];
  for (int c = c0; c < c1; ++c) {
    const int v = table[(int64_t)c * num_experts + e];
    table[(int64_t)c * num_experts + e] = run;
    run += v;
  }
  if (r == 3) totals[e] = run;
}

struct MoveArgs {
  const i32x4_t* in;   // [tokens, chunks16] 16-byte chunks; null: the map alone
  i32x4_t* out;
  const int32_t* indices;
  int32_t* row_id_map;
  void* counts;        // optional, int32 or int64
  int64_t tokens, capacity;
  int topk, num_experts, bits, chunks16, counts_i64, tokens_per_wg;
};

TGG_DEV void store_count(const MoveArgs& a, int e, int v) {
  if (a.counts_i64) ((int64_t*)a.counts)[e] = v; else ((int32_t*)a.counts)[e] = v;
}

// The rows of `count` tokens from token t0 on go to their destinations dest[token * topk + k] (LDS).  A thread takes
// a 16-byte chunk of a token: one load, topk stores.
template <int THREADS>
TGG_DEV void move_rows(const MoveArgs& a, const int* dest, int64_t t0, int count) {
  const uint32_t pieces = (uint32_t)count * (uint32_t)a.chunks16;
  for (uint32_t q = threadIdx.x; q < pieces; q += THREADS) {
    const uint32_t t = q / (uint32_t)a.chunks16, c = q - t * (uint32_t)a.chunks16;
    const i32x4_t v = a.in[(t0 + t) * a.chunks16 + c];
    const int* d = dest + t * a.topk;
    for (int k = 0; k < a.topk; ++k)
      if (d[k] >= 0) a.out[(int64_t)d[k] * a.chunks16 + c] = v;
  }
}

// One launch for the whole of a small problem.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void moe_small_kernel(const MoveArgs a) {
  __shared__ int total[kMaxExperts], front[kMaxExperts], scan[THREADS / 64], dest[kBatch];
  const int tid = threadIdx.x, n = (int)a.tokens * a.topk;
  for (int e = tid; e < a.num_experts; e += THREADS) total[e] = front[e] = 0;
  __syncthreads();
  const int t0 = (int)blockIdx.x * a.tokens_per_wg, t1 = min((int)a.tokens, t0 + a.tokens_per_wg);
  const int first = t0 * a.topk;
#pragma unroll 4
  for (int i = tid; i < n; i += THREADS) {
    const int e = a.indices[i];
    if (e >= 0 && e < a.num_experts) {
      atomicAdd(&total[e], 1);
      if (i < first) atomicAdd(&front[e], 1);
    }
  }
  __syncthreads();
  if (a.counts && blockIdx.x == 0)
    for (int e = tid; e < a.num_experts; e += THREADS) store_count(a, e, total[e]);
  __syncthreads();
  exclusive_scan_lds<THREADS>(total, a.num_experts, scan);
  const int per_batch = max(1, kBatch / a.topk);  // whole tokens; topk <= kBatch here
  for (int tb = t0; tb < t1; tb += per_batch) {
    const int count = min(per_batch, t1 - tb), items = count * a.topk;
    if (tid < 64) {  // the run's own assignments, 64 at a time in flat order
      for (int j = tid; j < ((items + 63) & ~63); j += 64) {
        const int i = tb * a.topk + j;
        const int e = j < items ? a.indices[i] : -1;
        const bool valid = e >= 0 && e < a.num_experts;
        const uint64_t same = match_lanes(e, valid, a.bits);
        int d = -1;
        if (valid) {
          const int before = front[e], ahead = lanes_before(same);
          if (total[e] + before + ahead < a.capacity) d = total[e] + before + ahead;
          if (ahead == 0) front[e] = before + __builtin_popcountll(same);
        }
        if (j < items) {
          dest[j] = d;
          const int t = i / a.topk;
          a.row_id_map[(int64_t)(i - t * a.topk) * a.tokens + t] = d;
        }
      }
    }
    __syncthreads();
    if (a.in) move_rows<THREADS>(a, dest, tb, count);
    __syncthreads();
  }
}

// Second launch of a larger problem (see the top of the file).  totals: null when the table still holds the chunks'
// own counts, else the experts' totals (the table then holds prefixes over the chunks).
template <int THREADS>
__global__ __launch_bounds__(THREADS) void moe_place_kernel(const MoveArgs a, const int32_t* __restrict__ table,
                                                            const int32_t* __restrict__ totals,
                                                            const int32_t* __restrict__ rank, int chunks, int64_t chunk) {
  __shared__ int start[kMaxExperts], front[kMaxExperts], scan[THREADS / 64], dest[kBatch];
  const int tid = threadIdx.x, E = a.num_experts;
  const int64_t t0 = (int64_t)blockIdx.x * a.tokens_per_wg;
  const int64_t t1 = min(a.tokens, t0 + a.tokens_per_wg);
  const int c0 = (int)(t0 * a.topk / chunk);
  for (int e = tid; e < E; e += THREADS) {
    start[e] = totals ? totals[e] : 0;
    front[e] = 0;
  }
  __syncthreads();
  if (!totals) {
    // columns of the table: `split` threads share one, each takes every split-th chunk
    const int split = max(1, THREADS / E), r = tid / E;
    for (int e = tid < split * E ? tid - r * E : E; e < E; e += THREADS) {
      int sum = 0, before = 0;
#pragma unroll 4
      for (int c = r; c < chunks; c += split) {
        const int v = table[(int64_t)c * E + e];
        sum += v;
        if (c < c0) before += v;
      }
      atomicAdd(&start[e], sum);
      atomicAdd(&front[e], before);
    }
    __syncthreads();
  }
  if (a.counts && blockIdx.x == 0)
    for (int e = tid; e < E; e += THREADS) store_count(a, e, start[e]);
  __syncthreads();
  exclusive_scan_lds<THREADS>(start, E, scan);
  const int per_batch = max(1, kBatch / a.topk);
  for (int64_t tb = t0; tb < t1; tb += per_batch) {
    const int count = (int)min((int64_t)per_batch, t1 - tb), items = count * a.topk;
    for (int j = tid; j < items; j += THREADS) {
      const int64_t i = tb * a.topk + j;
      const int e = a.indices[i];
      int64_t d = -1;
      if (e >= 0 && e < E) {
        d = (int64_t)start[e] + rank[i];
        const int c = (int)(i / chunk);
        if (totals) {
          d += table[(int64_t)c * E + e];
        } else {
          d += front[e];
          for (int q = c0; q < c; ++q) d += table[(int64_t)q * E + e];  // the run reaches into later chunks
        }
        if (d >= a.capacity) d = -1;
      }
      if (j < kBatch) dest[j] = (int)d;
      const int64_t t = i / a.topk;
      a.row_id_map[(i - t * a.topk) * a.tokens + t] = (int)d;
    }
    __syncthreads();
    if (a.in) {
      if (a.topk <= kBatch) {
        move_rows<THREADS>(a, dest, tb, count);
      } else {  // more destinations than the batch holds: straight from the map (this workgroup has just written it)
        __threadfence_block();
        for (int c = tid; c < a.chunks16; c += THREADS) {
          const i32x4_t v = a.in[tb * a.chunks16 + c];
          for (int k = 0; k < a.topk; ++k) {
            const int d = a.row_id_map[(int64_t)k * a.tokens + tb];
            if (d >= 0) a.out[(int64_t)d * a.chunks16 + c] = v;
          }
        }
      }
    }
    __syncthreads();
  }
}

// One workgroup per token, rows moved by a map that already exists: the row is read once and stored to every destination.
__global__ __launch_bounds__(256) void moe_permute_rows_kernel(const i32x4_t* __restrict__ in, i32x4_t* __restrict__ out,
                                                               const int32_t* __restrict__ row_id_map,
                                                               int64_t tokens, int topk, int chunks16) {
  const int64_t t = blockIdx.x;
  const i32x4_t* src = in + t * chunks16;
  for (int c = threadIdx.x; c < chunks16; c += 256) {
    const i32x4_t v = src[c];
    for (int k = 0; k < topk; ++k) {
      const int dest = row_id_map[(int64_t)k * tokens + t];  // wave-uniform
      if (dest >= 0) out[(int64_t)dest * chunks16 + c] = v;
    }
  }
}

template <int DT> struct Elem;  // 16 bytes <-> fp32 values
template <> struct Elem<DT_BF16> {
  static constexpr int N = 8;
  static TGG_DEV void unpack(i32x4_t v, float (&f)[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[2 * j] = __builtin_bit_cast(float, (uint32_t)v[j] << 16);
      f[2 * j + 1] = __builtin_bit_cast(float, (uint32_t)v[j] & 0xffff0000u);
    }
  }
  static TGG_DEV void store(void* p, const float (&f)[8]) {
    const uint2 a = pack4<DT_BF16>(f[0], f[1], f[2], f[3]), b = pack4<DT_BF16>(f[4], f[5], f[6], f[7]);
    i32x4_t v = {(int)a.x, (int)a.y, (int)b.x, (int)b.y};
    *(i32x4_t*)p = v;
  }
};
template <> struct Elem<DT_F16> {
  static constexpr int N = 8;
  static TGG_DEV void unpack(i32x4_t raw, float (&f)[8]) {
    const f16x8_t v = __builtin_bit_cast(f16x8_t, raw);
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = (float)v[j];
  }
  static TGG_DEV void store(void* p, const float (&f)[8]) {
    const uint2 a = pack4<DT_F16>(f[0], f[1], f[2], f[3]), b = pack4<DT_F16>(f[4], f[5], f[6], f[7]);
    i32x4_t v = {(int)a.x, (int)a.y, (int)b.x, (int)b.y};
    *(i32x4_t*)p = v;
  }
};
constexpr int DT_F32 = 4;  // only the permute kernels know fp32 activations
template <> struct Elem<DT_F32> {
  static constexpr int N = 4;
  static TGG_DEV void unpack(i32x4_t raw, float (&f)[4]) {
    const f32x4_t v = __builtin_bit_cast(f32x4_t, raw);
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = v[j];
  }
  static TGG_DEV void store(void* p, const float (&f)[4]) {
    f32x4_t v = {f[0], f[1], f[2], f[3]};
    *(f32x4_t*)p = v;
  }
};

// out[t, :] = sum_k prob[t, k] * in[row_id_map[k * tokens + t], :]   (prob == nullptr: plain sum)
// Bound by memory.  A wave takes 64 neighbouring 16-byte chunks of one token (so the map and the weights are scalar loads,
// and narrow rows leave no wave idle) and requests KU rows before it adds the first (one_row_at_a_time below says how
// many).  A workgroup per token, one row at a time, against this: 8192 x top-6 rows of 528 B 12.6 -> 6.3 us, 8192 x top-8 of
// 4 KB 47.0 -> 46.2 (6.3 TB/s; the card copies at 4.9 and reads at 6.2), of 14 KB 218 -> 206, 81920 x top-8 of 4 KB 574 ->
// 572, 65536 x top-1 of 4 KB 100.6 -> 101.4.  A wave of a top-1 launch has two short loads to wait for, so what it does
// before it requests its row shows: a 64-bit division for its token and a wait for the weight cost 2.5 % there.
template <int DT, int KU>
__global__ __launch_bounds__(256) void moe_unpermute_kernel(const char* __restrict__ in, char* __restrict__ out,
                                                            const int32_t* __restrict__ row_id_map,
                                                            const float* __restrict__ prob, int64_t tokens, int topk,
                                                            int chunks16, uint32_t waves_per_token, int shift,
                                                            uint32_t step_tokens, uint32_t step_pieces) {
  constexpr int N = Elem<DT>::N;
  // the launch's waves, four a workgroup and at most 2^24, walk the pieces of all tokens in order
  const uint32_t w = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t first = shift >= 0 ? w >> shift : w / waves_per_token;
  uint32_t piece = w - first * waves_per_token;
  for (int64_t t = first; t < tokens; t += step_tokens, piece += step_pieces) {
    if (piece >= waves_per_token) {
      piece -= waves_per_token;
      if (++t >= tokens) break;
    }
    const int c = (int)piece * 64 + lane_id();
    if (c >= chunks16) continue;
    float acc[N];
#pragma unroll
    for (int j = 0; j < N; ++j) acc[j] = 0.f;
    for (int k0 = 0; k0 < topk; k0 += KU) {
      i32x4_t row[KU];
      float weight[KU];
      bool kept[KU];
#pragma unroll
      for (int u = 0; u < KU; ++u) {
        const int k = k0 + u;
        const int src = k < topk ? row_id_map[(int64_t)k * tokens + t] : -1;
        kept[u] = src >= 0;
        if (kept[u]) {  // the weight behind the row's request, which would otherwise wait for it too
          row[u] = *(const i32x4_t*)(in + ((int64_t)src * chunks16 + c) * 16);
          weight[u] = prob ? prob[t * topk + k] : 1.f;
        }
      }
#pragma unroll
      for (int u = 0; u < KU; ++u)
        if (kept[u]) {
          float f[N];
          Elem<DT>::unpack(row[u], f);
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += weight[u] * f[j];
        }
    }
    Elem<DT>::store(out + (t * chunks16 + c) * 16, acc);
  }
}

// act_grad[dest, :] = prob[t, k] * grad[t, :];  prob_grad[t, k] = sum_h grad[t, h] * fwd_in[dest, h]
// One workgroup per token; KU forward rows are requested together and their dot products reduced together, with one
// barrier for all (two per row before): 8192 x top-8 rows of 4 KB 118 -> 113 us, 5.05 TB/s, half of it written.
template <int DT, int KU, bool SINGLE>
__global__ __launch_bounds__(256) void moe_unpermute_bwd_kernel(const char* __restrict__ grad, const char* __restrict__ fwd_in,
                                                                const int32_t* __restrict__ row_id_map,
                                                                const float* __restrict__ prob, char* __restrict__ act_grad,
                                                                float* __restrict__ prob_grad, int64_t tokens, int topk,
                                                                int chunks16) {
  constexpr int N = Elem<DT>::N;
  __shared__ float partial[4][KU];
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int k0 = 0; k0 < topk; k0 += KU) {
    int dest[KU];
    float weight[KU], dot[KU];
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int k = k0 + u;
      dest[u] = k < topk ? row_id_map[(int64_t)k * tokens + t] : -1;
      weight[u] = prob && k < topk && (!SINGLE || dest[u] >= 0) ? prob[t * topk + k] : 1.f;
      dot[u] = 0.f;
    }
    for (int c = threadIdx.x; c < chunks16; c += 256) {
      i32x4_t row[KU];
      float g[N];
      Elem<DT>::unpack(*(const i32x4_t*)(grad + (t * chunks16 + c) * 16), g);
      if (prob_grad && !SINGLE) {
#pragma unroll
        for (int u = 0; u < KU; ++u)
          if (dest[u] >= 0) row[u] = *(const i32x4_t*)(fwd_in + ((int64_t)dest[u] * chunks16 + c) * 16);
      }
#pragma unroll
      for (int u = 0; u < KU; ++u)
        if (dest[u] >= 0) {
          float s[N];
#pragma unroll
          for (int j = 0; j < N; ++j) s[j] = weight[u] * g[j];
          Elem<DT>::store(act_grad + ((int64_t)dest[u] * chunks16 + c) * 16, s);
          if (prob_grad) {
            if (SINGLE) {
              asm volatile("" ::: "memory");  // the store stays in front of the read
              row[u] = *(const i32x4_t*)(fwd_in + ((int64_t)dest[u] * chunks16 + c) * 16);
            }
            float x[N];
            Elem<DT>::unpack(row[u], x);
#pragma unroll
            for (int j = 0; j < N; ++j) dot[u] += g[j] * x[j];
          }
        }
    }
    if (prob_grad) {
#pragma unroll
      for (int u = 0; u < KU; ++u) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) dot[u] += __shfl_xor(dot[u], d, 64);
        if (lane == 0) partial[wave][u] = dot[u];
      }
      __syncthreads();
      if (threadIdx.x < KU && k0 + (int)threadIdx.x < topk)
        prob_grad[t * topk + k0 + threadIdx.x] = partial[0][threadIdx.x] + partial[1][threadIdx.x] +
                                                 partial[2][threadIdx.x] + partial[3][threadIdx.x];
      __syncthreads();
    }
  }
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct SortWorkspace {
  int32_t *table, *totals, *rank;
  int64_t chunk;
  int chunks;
  size_t bytes;
};

SortWorkspace carve(void* base, int64_t n, int num_experts) {
  SortWorkspace w;
  w.chunk = count_chunk(n, num_experts);
  w.chunks = (int)((n + w.chunk - 1) / w.chunk);
  size_t off = 0;
  char* b = (char*)base;
  w.table = (int32_t*)(b + off); off += align256((size_t)num_experts * (size_t)(w.chunks > 0 ? w.chunks : 1) * 4);
  w.totals = (int32_t*)(b + off); off += align256((size_t)num_experts * 4);
  w.rank = (int32_t*)(b + off); off += align256((size_t)(n > 0 ? n : 1) * 4);
  w.bytes = off;
  return w;
}

// Whether the one-launch sort takes the problem.  No assignments at all are always its own: the counting and placing
// launches would have empty grids.
bool small_sort(int64_t n, int topk) { return n == 0 || (n <= kSmallAssignments && topk <= kBatch); }

}  // namespace

int64_t moe_sort_workspace_bytes(int64_t tokens, int topk, int num_experts) {
  return small_sort(tokens * topk, topk) ? 0 : (int64_t)carve(nullptr, tokens * topk, num_experts).bytes;
}

// in / out null: the map (and counts) alone; otherwise the rows are moved as well.
int launch_moe_permute(const void* in, void* out, int64_t row_bytes, const int32_t* indices, int64_t tokens, int topk,
                       int num_experts, int64_t capacity, int32_t* row_id_map, void* counts, int counts_i64,
                       void* workspace, hipStream_t s) {
  const int64_t n = tokens * topk, cus = num_cus();
  MoveArgs a;
  a.chunks16 = (int)(row_bytes / 16);
  const bool move = in && tokens > 0 && a.chunks16 <= (1 << 20) &&  // a batch's chunks are counted in 32 bits
                    (small_sort(n, topk) || place_moves_rows(tokens, topk, row_bytes));
  a.in = move ? (const i32x4_t*)in : nullptr;
  a.out = (i32x4_t*)out;
  a.indices = indices;
  a.row_id_map = row_id_map;
  a.counts = counts;
  a.counts_i64 = counts_i64;
  a.tokens = tokens;
  a.capacity = capacity;
  a.topk = topk;
  a.num_experts = num_experts;
  a.bits = 0;
  while ((1 << a.bits) < num_experts) ++a.bits;
  if (small_sort(n, topk)) {
    // rows: enough workgroups to fill the chip twice (each repeats the counting); the map alone: 512 assignments each
    const int64_t want = move ? 2 * cus : (n + 511) / 512;
    const int64_t per = want > 0 ? (tokens + want - 1) / want : 1;
    a.tokens_per_wg = (int)(per > 0 ? per : 1);
    const int64_t grid = tokens > 0 ? (tokens + a.tokens_per_wg - 1) / a.tokens_per_wg : 1;
    hipLaunchKernelGGL(moe_small_kernel<kPlaceThreads>, dim3((unsigned)grid), dim3(kPlaceThreads), 0, s, a);
  } else {
    const SortWorkspace w = carve(workspace, n, num_experts);
    hipLaunchKernelGGL(moe_count_kernel, dim3(w.chunks), dim3(kCountThreads), kCountThreads / 64 * num_experts * sizeof(uint16_t), s,
                       indices, n, num_experts, a.bits, (int)(w.chunk / (kCountThreads / 64)), w.table, w.rank);
    const bool scanned = (int64_t)w.chunks * num_experts > kTableEntries;
    if (scanned)
      hipLaunchKernelGGL(moe_scan_table_kernel, dim3((num_experts + 63) / 64), dim3(256), 0, s, w.table, w.chunks, num_experts, w.totals);
    // rows: four workgroups per CU, all resident; the map alone: 2048 assignments each
    const int64_t want = move ? 4 * cus : (n + 2047) / 2048;
    a.tokens_per_wg = (int)((tokens + want - 1) / want);
    hipLaunchKernelGGL(moe_place_kernel<kPlaceThreads>, dim3((unsigned)((tokens + a.tokens_per_wg - 1) / a.tokens_per_wg)), dim3(kPlaceThreads),
                       0, s, a, w.table, scanned ? w.totals : nullptr, w.rank, w.chunks, w.chunk);
  }
  if (int e = check_launch("moe_permute")) return e;
  return in && !move && tokens > 0 ? launch_moe_permute_rows(in, out, row_id_map, tokens, topk, row_bytes, s) : 0;
}

int launch_moe_permute_map(const int32_t* indices, int64_t tokens, int topk, int num_experts, int64_t capacity,
                           int32_t* row_id_map, void* counts, int counts_i64, void* workspace, hipStream_t s) {
  return launch_moe_permute(nullptr, nullptr, 0, indices, tokens, topk, num_experts, capacity, row_id_map, counts,
                            counts_i64, workspace, s);
}

// ---- the sort without a caller-provided workspace ---------------------------------------------------------------
// For callers that cannot allocate (HIP graph capture, serving loops): the sort's temporaries live in a fixed
// array in device memory that is part of the library's code object.  Sized for any problem the entry point
// accepts: 2^20 assignments, 1024 experts, the smallest chunks (table 4 MiB + rank 4 MiB + totals 4 KiB, and 4 KiB to spare).  Every GPU the
// library runs on holds its own copy at its own address until the process ends; all calls on one GPU share it, so
// calls that overlap on one GPU (different streams) race.  Nothing in it has to start at zero: the counting pass
// writes every table entry and rank that is read later, the scan of a large table its totals; the one-launch sort uses none of it.
constexpr int64_t kStaticMaxAssignments = 1ll << 20;
constexpr size_t kStaticScratchBytes = (size_t)kMaxExperts * (kStaticMaxAssignments / kCountThreads) * 4 + 2 * (size_t)kMaxExperts * 4 +
                                       (size_t)kStaticMaxAssignments * 4;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

// Device address of this GPU's copy of `scratch`, looked up once per device (the array's name is only a host-side
// handle for hipGetSymbolAddress; it is never passed to a kernel or a memory call).
static int static_scratch_ptr(void** out) {
  static std::mutex mu;
  static void* ptr[64] = {nullptr};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return check_launch("hipGetDevice");
  if (dev < 0 || dev >= 64) return set_error("device ordinal %d outside [0, 64)", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      (void)hipGetLastError();
      return set_error("hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
    }
    ptr[dev] = p;
  }
  *out = ptr[dev];
  return 0;
}

int64_t moe_static_max_assignments() { return kStaticMaxAssignments; }

int launch_moe_permute_map_static(const int32_t* indices, int64_t tokens, int topk, int num_experts, int64_t capacity,
                                  int32_t* row_id_map, void* counts, int counts_i64, hipStream_t s) {
  const int64_t n = tokens * topk;
  if (n > kStaticMaxAssignments)
    return set_error("num_tokens * topk = %lld exceeds the %lld assignments the built-in scratch array holds; "
                     "use tgg_moe_permute_map with a workspace", (long long)n, (long long)kStaticMaxAssignments);
  if (carve(nullptr, n, num_experts).bytes > kStaticScratchBytes)
    return set_error("sort temporaries of %zu bytes exceed the built-in scratch array (%zu bytes)",
                     carve(nullptr, n, num_experts).bytes, kStaticScratchBytes);
  void* ws = nullptr;
  if (int e = static_scratch_ptr(&ws)) return e;
  return launch_moe_permute_map(indices, tokens, topk, num_experts, capacity, row_id_map, counts, counts_i64, ws, s);
}

int launch_moe_permute_rows(const void* in, void* out, const int32_t* row_id_map, int64_t tokens, int topk,
                            int64_t row_bytes, hipStream_t s) {
  if (tokens == 0) return 0;
  hipLaunchKernelGGL(moe_permute_rows_kernel, dim3((unsigned)tokens), dim3(256), 0, s, (const i32x4_t*)in, (i32x4_t*)out,
                     row_id_map, tokens, topk, (int)(row_bytes / 16));
  return check_launch("moe_permute_rows");
}

// KU, the rows of a token that a wave requests before it uses the first (the topK loop runs in groups of KU): 2 and 4
// measure the same on top-8 rows, 8 is 3-5 % slower in the forward kernel and 11 % in the backward one (registers).
// The forward kernel one row at a time: from 400 MiB read and written on, where the rows come from memory rather than from
// the memory-side cache and are the faster the fewer are in flight at once (top-8 rows of 4 KB, four / one: 144 MiB 23.0 /
// 22.6 us, 288 MiB 46.5 / 46.9, 432 MiB 89.3 / 88.7, 1700 MiB 347.5 / 338.2; top-4 and top-6 alike).  Top-2 rows are 0.6 %
// faster in pairs at every size; rows below 1 KB (several tokens a workgroup) want all requests they can have (512 B, top-8,
// 864 MiB: 199.7 / 224.9).
static bool one_row_at_a_time(int64_t tokens, int topk, int c16) {
  return topk > 2 && c16 >= 64 && tokens * (topk + 1) * c16 * 16 > (400ll << 20);
}

template <int DT>
static void launch_unpermute_dt(const void* in, void* out, const int32_t* row_id_map, const float* prob, int64_t tokens,
                                int topk, int c16, hipStream_t s) {
  const int per_token = (c16 + 63) / 64;
  const int64_t wgs = (tokens * per_token + 3) / 4;
  const dim3 grid((unsigned)(wgs < (1 << 22) ? wgs : 1 << 22));  // a launch's threads stay below 2^32
  const uint32_t step_tokens = grid.x * 4 / per_token, step_pieces = grid.x * 4 % per_token;
  const int shift = (per_token & (per_token - 1)) == 0 ? __builtin_ctz(per_token) : -1;
#define TGG_LAUNCH(KU) \
  hipLaunchKernelGGL((moe_unpermute_kernel<DT, KU>), grid, dim3(256), 0, s, (const char*)in, (char*)out, \
                     row_id_map, prob, tokens, topk, c16, (uint32_t)per_token, shift, step_tokens, step_pieces)
  if (topk <= 1 || one_row_at_a_time(tokens, topk, c16)) TGG_LAUNCH(1);
  else if (topk <= 2) TGG_LAUNCH(2);
  else TGG_LAUNCH(4);
#undef TGG_LAUNCH
}

// The backward kernel one row at a time, stored before the forward row is read: where a row is one chunk for (nearly) every
// thread of the workgroup and the gradient has more than 64 MiB.  Rows of 4 KB, batches / one: top-8 of 8192 tokens 112.2 /
// 115.8 us, of 12288 172.2 / 172.5, of 24576 340.0 / 339.4, of 81920 1136 / 1115; top-4 of 29491 223.6 / 219.3; top-2 of 65536
// 258 / 247; top-1 of 28672 66.0 / 65.1.  Shorter rows leave threads idle, longer ones are several chunks a thread: batches
// are better there with top-8 (rows of 3.5 KB by 2 %, of 5.6 KB by 5 %, of 8 KB by 2.5 %).
static bool single_backward(int64_t tokens, int c16) { return c16 > 240 && c16 <= 256 && tokens * c16 * 16 > (64ll << 20); }

template <int DT>
static void launch_unpermute_bwd_dt(const void* grad, const void* fwd_in, const int32_t* row_id_map, const float* prob,
                                    void* act_grad, float* prob_grad, int64_t tokens, int topk, int c16, hipStream_t s) {
#define TGG_LAUNCH(KU, SINGLE) \
  hipLaunchKernelGGL((moe_unpermute_bwd_kernel<DT, KU, SINGLE>), dim3((unsigned)tokens), dim3(256), 0, s, (const char*)grad, \
                     (const char*)fwd_in, row_id_map, prob, (char*)act_grad, prob_grad, tokens, topk, c16)
  if (single_backward(tokens, c16)) TGG_LAUNCH(1, true);
  else if (topk <= 1) TGG_LAUNCH(1, false);
  else if (topk <= 2) TGG_LAUNCH(2, false);
  else TGG_LAUNCH(4, false);
#undef TGG_LAUNCH
}

int launch_moe_unpermute(const void* in, void* out, const int32_t* row_id_map, const float* prob, int64_t tokens,
                         int topk, int64_t row_bytes, int dt, hipStream_t s) {
  if (tokens == 0) return 0;
  const int c16 = (int)(row_bytes / 16);
  if (dt == DT_BF16) launch_unpermute_dt<DT_BF16>(in, out, row_id_map, prob, tokens, topk, c16, s);
  else if (dt == DT_F16) launch_unpermute_dt<DT_F16>(in, out, row_id_map, prob, tokens, topk, c16, s);
  else launch_unpermute_dt<DT_F32>(in, out, row_id_map, prob, tokens, topk, c16, s);
  return check_launch("moe_unpermute");
}

int launch_moe_unpermute_bwd(const void* grad, const void* fwd_in, const int32_t* row_id_map, const float* prob,
                             void* act_grad, float* prob_grad, int64_t tokens, int topk, int64_t row_bytes, int dt,
                             hipStream_t s) {
  if (tokens == 0) return 0;
  const int c16 = (int)(row_bytes / 16);
  if (dt == DT_BF16) launch_unpermute_bwd_dt<DT_BF16>(grad, fwd_in, row_id_map, prob, act_grad, prob_grad, tokens, topk, c16, s);
  else if (dt == DT_F16) launch_unpermute_bwd_dt<DT_F16>(grad, fwd_in, row_id_map, prob, act_grad, prob_grad, tokens, topk, c16, s);
  else launch_unpermute_bwd_dt<DT_F32>(grad, fwd_in, row_id_map, prob, act_grad, prob_grad, tokens, topk, c16, s);
  return check_launch("moe_unpermute_bwd");
}

}  // namespace tgg
