// Building blocks shared by the four-wave gfx950 kernels (gemm_w4.hip, gemm_wgrad.hip): multiplies and fragment reads as
// single inline-assembly statements, which the compiler keeps in source order and only allocates registers for.
#pragma once
#include "fast_common.hpp"
#include <utility>

namespace tgg {

template <int DT> TGG_DEV void mfma_acc(f32x4_t& acc, const i32x4_t& w, const i32x4_t& x) {
  if (DT == DT_BF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
}

// The same with a zero addend: the first K step of a tile starts its accumulators afresh
template <int DT> TGG_DEV void mfma_new(f32x4_t& acc, const i32x4_t& w, const i32x4_t& x) {
  if (DT == DT_BF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc) : "v"(w), "v"(x));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(acc) : "v"(w), "v"(x));
}

// 16-byte fragment of a K-contiguous operand
template <int OFF> TGG_DEV void lds_read_b128(i32x4_t& dst, uint32_t addr) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF) : "memory");
}
// fragment of a token-row operand: two transposing 8-byte reads (K 0..3 and 4..7 of the lane's column)
template <int OFF0, int OFF1> TGG_DEV void lds_read_tr(i32x4_t& dst, uint32_t addr) {
  i32x2_t lo, hi;
  asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\tds_read_b64_tr_b16 %1, %2 offset:%4"
               : "=&v"(lo), "=&v"(hi) : "v"(addr), "n"(OFF0), "n"(OFF1) : "memory");
  dst = __builtin_shufflevector(lo, hi, 0, 1, 2, 3);
}
#define TGG_TIE8(f) "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7])

// A 16-byte output store of a lane and the wait states behind it (two must pass before the data registers may be overwritten).
// NT: non-temporal, for rows that begin on a multiple of 64 bytes.  Elsewhere the ends of a row segment share a line
// with the segments beside it, which are stored a few multiplies apart; non-temporal, such a line goes out piece by piece, which costs
// memory-bound launches up to half their time, while lines that stay in L2 are completed there first (figures: gemm_wgrad.hip).
inline bool rows_of_whole_64_bytes(const GemmParams& p) { return p.N % 32 == 0 && ((uintptr_t)p.C & 63) == 0; }
template <bool NT, int NOP> TGG_DEV void store_b128(const i32x4_t& v, int off, const i32x4_t& rs) {
  if constexpr (NT) asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen nt\n\ts_nop %3" : : "v"(v), "v"(off), "s"(rs), "n"(NOP) : "memory");
  else asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen\n\ts_nop %3" : : "v"(v), "v"(off), "s"(rs), "n"(NOP) : "memory");
}

// Division of 32-bit values by a divisor that is fixed for the launch, on the scalar unit.  m = floor(2^32 / d) + 1: the
// estimate n m / 2^32 is the quotient or one more for every 32-bit n.
struct FixedDiv {
  uint32_t d, m;
  TGG_DEV explicit FixedDiv(int d_) : d((uint32_t)d_), m(d_ > 1 ? 0xffffffffu / (uint32_t)d_ + 1 : 0) {}
  TGG_DEV uint32_t div(uint32_t n) const {
    if (d == 1) return n;
    const uint32_t q = __umulhi(n, m);
    return q * d > n ? q - 1 : q;
  }
};

// f(integral_constant<int, n>) for n = 0 .. N - 1: the gaps of a K step's multiplies
template <class F, int... N> TGG_DEV void for_each_of(const F& f, std::integer_sequence<int, N...>) { (f(std::integral_constant<int, N>()), ...); }
template <int N, class F> TGG_DEV void for_each(const F& f) { for_each_of(f, std::make_integer_sequence<int, N>()); }

// A tile of a K-grouped launch (256x256 outputs of one group), and its lookup from a tile id: sched_tile with the divisions by
// values fixed for the launch done on the scalar unit.
struct KgTile {
  int g, m0, n0;  // g = -1: there are no more tiles
  int slot;       // launches cut along K (kg_split.hpp): the part's place in the workspace, -1: the group is in one part
  int klen;       // tokens of the segment
  int64_t k0;     // its first token
};

template <class Table>
struct KgTiles {
  const Table& t;
  int tiles_m, nc, full_chunks, tail_width, per_group, total;
  FixedDiv by_group, by_chunk, by_nc, by_tail;
  const int32_t* meta;  // launches cut along K: what part an entry of the table is, else null
  TGG_DEV KgTiles(const GemmParams& p, const Table& t_, int groups, const int32_t* meta_)
      : t(t_), tiles_m((int)((p.m_total + 255) / 256)), nc(sched_chunk_width((p.N + 255) / 256, p.n_chunk)),
        full_chunks((p.N + 255) / 256 / nc), tail_width((p.N + 255) / 256 - full_chunks * nc), per_group(tiles_m * ((p.N + 255) / 256)),
        total(groups * per_group), by_group(per_group), by_chunk(tiles_m * nc), by_nc(nc), by_tail(tail_width > 0 ? tail_width : 1), meta(meta_) {}
  TGG_DEV KgTile look_up(int id) const {
    KgTile r;
    r.g = -1;
    r.m0 = r.n0 = r.klen = 0;
    r.slot = -1;
    r.k0 = 0;
    if (id < total) {
      const int slot = (int)by_group.div((uint32_t)id), at = id - slot * per_group;
      int c = (int)by_chunk.div((uint32_t)at);  // as sched_split
      const bool tail = c >= full_chunks;
      c = tail ? full_chunks : c;
      const int width = tail ? tail_width : nc, q = at - c * tiles_m * nc;
      const int mt = (int)(tail ? by_tail.div((uint32_t)q) : by_nc.div((uint32_t)q));
      r.m0 = mt * 256;
      r.n0 = (c * nc + q - mt * width) * 256;
      r.g = __builtin_amdgcn_readfirstlane(t.tile0[slot]);
      r.klen = __builtin_amdgcn_readfirstlane(t.rows[r.g]);
      r.k0 = (int64_t)uniform64((uint64_t)t.row0[r.g]);
      if (meta) {
        const int part = __builtin_amdgcn_readfirstlane(meta[r.g]);
        r.g = part & 0xffff;
        r.slot = (part >> 16) - 1;
      }
    }
    return r;
  }
};

// Where a four-wave workgroup's tiles of a K-grouped launch come from: the work queue of sched.hpp (largest groups first, one
// counter per XCD) or, without one, the fixed walk.  Wave 0 draws: request() goes out some K steps before take(), whose
// caller has waited for it; the answer sits in v255, which is named in the instruction text because a value in
// flight across K steps must not be known to the compiler (assembly_checks.py scans the assembly for any other use;
// the kernels' own waits list it as clobbered).  take() leaves the tile id in LDS for the other waves, in front of a
// barrier.  A counter's value stands for a tile id (sched_queue_id); once it stands for none, the wave looks at all
// counters at once and goes on with the next one that has tiles left.
struct KgDraw {
  int32_t* queue;
  volatile int32_t* next_id;  // two words of LDS, by the parity of the tile's position
  int total, R, lane, xq;
  int exhausted = 0;          // counters that a draw has found without a tile, one bit each
  bool spread, queued, live;  // eight counters or one; a queue was given; tiles are still being drawn (wave 0)
  FixedDiv by_r;
  TileWalk walk;
  TGG_DEV KgDraw(const GemmParams& p, int32_t* next_id_, int total_, int wave, int lane_)
      : queue(p.queue), next_id(next_id_), total(total_), R((int)gridDim.x >> 3), lane(lane_), xq((gridDim.x & 7) == 0 ? (int)(blockIdx.x & 7) : 0),
        spread((gridDim.x & 7) == 0), queued(p.queue != nullptr), live(p.queue != nullptr && wave == 0), by_r(R > 0 ? R : 1), walk(sched_walk(total_, false)) {
    if (wave == 0 && lane < 2) next_id[lane] = total;  // what the other waves find once nothing is drawn any more
  }
  TGG_DEV int id_of(int n) const {
    if (!spread) return n;
    const int pass = (int)by_r.div((uint32_t)n);
    return (pass * 8 + ((pass & 1) ? 7 - xq : xq)) * R + n - pass * R;
  }
  TGG_DEV int steal() {  // the next tile of another counter, `total` where there is none
    while (spread) {  // eight rounds at most: a round ends the search or marks a counter
      exhausted |= 1 << xq;
      const int seen = lane < 8 ? __hip_atomic_load(queue + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
      const int left = sched_queue_left(seen, total, R) & ~exhausted;
      if (left == 0) break;
      xq = sched_queue_next(left, xq);
      int n = 0;
      if (lane == 0) n = atomicAdd(queue + xq, 1);
      const int id = id_of(__builtin_amdgcn_readfirstlane(n));
      if (id < total) return id;
    }
    return total;
  }
  TGG_DEV void request() {
    if (live && lane == 0) {
      int32_t* const at = queue + xq;
      asm volatile("global_atomic_add v255, %0, %1, %2 sc0" : : "v"(0), "v"(1), "s"(at) : "memory", "v255");
    }
  }
  TGG_DEV void take(int pos) {
    if (live) {
      int got;
      asm volatile("v_readfirstlane_b32 %0, v255" : "=s"(got) : : "memory", "v255");
      int id = id_of(got);
      if (__builtin_expect(id >= total, 0)) {
        id = steal();
        live = id < total;
      }
      if (lane == 0) next_id[pos & 1] = id;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  }
  TGG_DEV int tile_at(int pos) const {  // the id of the workgroup's pos-th tile, `total` behind its last
    if (queued) return __builtin_amdgcn_readfirstlane(next_id[pos & 1]);
    const int64_t id = walk.first + (int64_t)pos * walk.stride;
    return id < walk.end ? (int)id : total;
  }
  TGG_DEV void finish() const {
    if (queued && threadIdx.x == 0) sched_queue_finish(queue);
  }
};

}  // namespace tgg
