// Four-wave FP8 (OCP e4m3fn / e5m2) grouped GEMM kernel for gfx950, K-contiguous operands, per-channel scales:
//   out[r, n] = (sum_k a[r, k] b[g, n, k]) * scale_m[r] * scale_n[g*N + n]
// K-grouped (weight gradient: x [M, Ktot], y [N, Ktot], a token range per group).
//
// One workgroup per CU, four waves, one per SIMD; tile 256x256, every wave owns a 128x128 block of 16x16x128 MFMA tiles with its
// 256 accumulator registers in AGPRs.  Against the eight-wave kernel (gemm_fp8.hip: 128x64 per wave) a slab needs a third fewer LDS
// reads per multiply, which there take as long as the multiplies, and the epilogue rides on multiplies.  A slab is 128
// bytes of every row = one K step; two slab buffers of 64 KB.
//
// A multiply keeps the matrix pipe busy for 32 cycles, so about six other instructions fit between two.  The operands' sixteen
// fragments of eight registers stay single: a slab's 64 multiplies run in sixteen groups of four (four row blocks times one column
// block), in quadrants, so that fragments are done with one after the other and the next ones are read in their place at least
// three groups (384 cycles) before they are used.  A0-3 = row blocks 0-3, ' = of the next slab:
//   group   0-3: A0-3 x B0..B3     4-7: A0-3 x B4..B7     8-11: A4-7 x B7..B4     12-15: A4-7 x B0..B3
//   reads   0: B3   1: B6 B7   2-5: A4..A7   | barrier |   8-11: A0'..A3'   12: B4' B5'   13-15: B0' B1' B2'
// LDS reads return in order, so a group waits with a count that leaves the younger ones in flight.  In front of group 8 the
// wave waits for its reads of the current slab and its copies of the next one and passes the workgroup barrier: the
// current slab's buffer is free, and its sixteen copies of the slab after the next are requested one every other multiply
// in groups 8-15.  The buffers alternate by a toggled address bit, so any number of slabs per tile will do (two at least: of
// nothing, if need be).
//
// The epilogue needs no LDS staging: B's rows sit in LDS in the order of gemm_w4.hip, so that a lane's results of the eight column
// blocks are eight neighbouring outputs of a row.  Row blocks 0-3 are complete after group 7 of a tile's last slab and leave between
// the multiplies of its groups 8-15; row blocks 4-7 leave in groups 0-7 of the next tile's first slab, where they are not
// touched.  The tile's 256 + 256 scales are copied to LDS in its first slab.
//
// Against the eight-wave kernel: 32 groups of 3072 x 4096 with 128 / 256 / 512 / 1024 / 4096 tokens on average 208 / 235 / 307 / 474 / 1511 ->
// 170 / 194 / 258 / 419 / 1269 us (2.6 PFLOP/s).  Without a fetch (nothing copied) the last one takes 798 us, with zeros for operands no less than with
// random ones: what bounds it is how fast 128-byte lines of distant rows come from HBM and L2, not power.  Without the touches
// (below) 466 and 1474 us.
#include "launch.hpp"
#include "kg_split.hpp"

namespace tgg {

namespace {

struct Fp8W4Cfg {
  static constexpr int BM = 256, BN = 256, THREADS = 256, KS = 128;
  static constexpr int A_BYTES = BM * KS, B_BYTES = BN * KS, STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int SCHED_OFF = 2 * STAGE_BYTES;
  static constexpr int NEXT_OFF = SCHED_OFF + (((int)sizeof(SchedTableT<kFastMaxGroups>) + 255) & ~255);
  static constexpr int SCALE_OFF = NEXT_OFF + 256;  // the tile's row scales, then its column scales
  static constexpr int SINK_OFF = SCALE_OFF + (BM + BN) * 4;  // where touched lines' words go, 256 bytes a wave
  static constexpr int META_OFF = SINK_OFF + 4 * 256;  // launches cut along K: what the table's entries are
  static constexpr int SMEM_BYTES = META_OFF + kFastMaxGroups * 4;
  static_assert(STAGE_BYTES == 0x10000, "the slab buffers alternate by one address bit");
  static_assert(SMEM_BYTES <= 160 * 1024, "LDS budget");
};

template <int FA, int FB> TGG_DEV void mfma8_acc(f32x4_t& acc, const i32x8_t& a, const i32x8_t& b) {
  asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:%3 blgp:%4" : "+a"(acc) : "v"(a), "v"(b), "n"(FA), "n"(FB));
}
template <int FA, int FB> TGG_DEV void mfma8_new(f32x4_t& acc, const i32x8_t& a, const i32x8_t& b) {
  asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0 cbsz:%3 blgp:%4" : "=a"(acc) : "v"(a), "v"(b), "n"(FA), "n"(FB));
}

// one fragment: 16-byte chunks lg and lg + 4 of a row's 128 bytes (see gemm_fp8.hip)
template <int OFF> TGG_DEV void read_frag8(i32x8_t& dst, uint32_t at0, uint32_t at1) {
  i32x4_t lo, hi;
  asm volatile("ds_read_b128 %0, %2 offset:%4\n\tds_read_b128 %1, %3 offset:%4" : "=&v"(lo), "=&v"(hi) : "v"(at0), "v"(at1), "n"(OFF) : "memory");
  dst = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

typedef SplitCost<128, 2, 18, 8> Fp8SplitCost;

// FA / FB: 0 = e4m3fn, 1 = e5m2 (format codes of the f8f6f4 multiply).  SPLIT: segments may be cut along K, see gemm_wgrad.hip; the
// kernel that adds the parts up applies the scales.
template <int FA, int FB, int OUT, bool SPLIT>
__global__ __launch_bounds__(Fp8W4Cfg::THREADS) void fp8_w4_kernel(const GemmParams p) {
  typedef Fp8W4Cfg C;
  typedef Operand<256, true> Op;  // a slab of either operand: 256 rows of 128 bytes

  extern __shared__ __attribute__((aligned(1024))) char smem[];
  auto& sched = *reinterpret_cast<SchedTableT<kFastMaxGroups>*>(smem + C::SCHED_OFF);
  sched_init<C::BM>(p, sched);
  if (!sched_kg_gate_open(p, sched)) {
    if (SPLIT && blockIdx.x == 0 && (int)threadIdx.x < p.G) reinterpret_cast<int32_t*>(p.split_ws)[2 * threadIdx.x + 1] = 0;  // there are no parts
    return;
  }
  int32_t* const meta = SPLIT ? reinterpret_cast<int32_t*>(smem + C::META_OFF) : nullptr;
  int groups = p.G;
  if constexpr (SPLIT) groups = __builtin_amdgcn_readfirstlane(split_plan<Fp8SplitCost>(p, sched, meta, (int)((p.m_total + 255) / 256) * ((p.N + 255) / 256)));

  const uint32_t smem_addr = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm0 = (wave >> 1) * 128, wn0 = (wave & 1) * 128;
  const int l16 = lane & 15, lg = lane >> 4;
  const int ld = (int)p.k_total;  // bytes between consecutive rows of either operand

  // Copy k (0..7) of an operand's slab by this wave is copy instruction wave + 4 k: LDS rows 8 (wave + 4 k) ... + 7.  A's rows are in order,
  // B's permuted as in gemm_w4.hip: LDS row 128 h + 16 j + c holds column 128 h + 8 c + j of the tile.
  int vo_a[8], vo_b[8];
  static_assert(Op::NPAT == 2, "the swizzle pattern of copy wave + 4 k is that of copy wave");
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int r_local = lane / Op::CPR;
    const int col = 128 * (k >> 2) + 8 * (8 * (wave & 1) + r_local) + 2 * (k & 3) + (wave >> 1);
    vo_a[k] = Op::lane_voff(lane, wave % Op::NPAT, ld) + (wave + 4 * k) * Op::RPI * ld;
    vo_b[k] = Op::lane_voff(lane, wave % Op::NPAT, ld) + (col - r_local) * ld;
  }
  const int my_chunk = Op::lane_chunk(lane, wave % Op::NPAT);  // which 16 bytes of its row's 128 this lane copies
  const int fsw = (l16 / 2) % 8;
  uint32_t a_rd[2], b_rd[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int at = l16 * 128 + (((lg + 4 * h) ^ fsw) << 4);
    a_rd[h] = smem_addr + wm0 * 128 + at;
    b_rd[h] = smem_addr + C::A_BYTES + wn0 * 128 + at;
  }

  // ---- the copy stream -------------------------------------------------------------------------------------------------------
  // The cursor is two slabs ahead of the multiplies.  A tile's windows (descriptors) are fixed, the offset along K travels in the copies'
  // scalar offset, which the windows' range check counts in; chunks beyond the tile's range along K are not fetched.
  const KgTiles<SchedTableT<kFastMaxGroups>> tiles(p, sched, groups, meta);
  KgDraw draw(p, reinterpret_cast<int32_t*>(smem + C::NEXT_OFF), tiles.total, wave, lane);
  auto steps_of = [&](const KgTile& t) __attribute__((always_inline)) {
    const int steps = (t.klen + C::KS - 1) / C::KS;
    return steps < 2 ? 2 : steps;
  };
  struct Feed {
    i32x4_t ra, rb;
    int klen, koff, left;
  };
  auto feed_of = [&](const KgTile& t) __attribute__((always_inline)) {
    Feed f;
    const int m_left = (int)p.m_total - t.m0, n_left = p.N - t.n0;
    f.ra = make_rsrc((uint64_t)p.A + (uint64_t)((int64_t)t.m0 * ld + t.k0), (int64_t)(m_left < C::BM ? m_left : C::BM) * ld - t.k0);
    f.rb = make_rsrc((uint64_t)p.B + (uint64_t)((int64_t)t.n0 * ld + t.k0), (int64_t)(n_left < C::BN ? n_left : C::BN) * ld - t.k0);
    f.klen = t.klen;
    f.koff = 0;
    f.left = t.g < 0 ? 0x7fffffff : steps_of(t);
    return f;
  };
  Feed feed, nxt;
  int koff = 0, mask = 0;  // of the slab being requested; mask: kNoFetch in the lanes that fetch nothing
  auto step_feed = [&]() __attribute__((always_inline)) {
    const bool wrap = feed.left == 0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      feed.ra[q] = wrap ? nxt.ra[q] : feed.ra[q];
      feed.rb[q] = wrap ? nxt.rb[q] : feed.rb[q];
    }
    feed.klen = wrap ? nxt.klen : feed.klen;
    koff = wrap ? 0 : feed.koff;
    feed.left = (wrap ? nxt.left : feed.left) - 1;
    feed.koff = koff + C::KS;
    mask = koff + my_chunk * 16 >= feed.klen ? kNoFetch : 0;  // K-grouped ranges are multiples of 16 (kg_gate)
  };
  const uint32_t wave_buf = smem_addr + wave * 1024;
  uint32_t cp_buf = wave_buf;  // this wave's first copy in the buffer that is being filled
  auto copy_m0 = [&](auto Kc) __attribute__((always_inline)) {
    constexpr int k = decltype(Kc)::value;
    const uint32_t buf = cp_buf;
    asm volatile("s_add_u32 m0, %0, %1" : : "s"(buf), "n"((k >> 3) * C::A_BYTES + (k & 7) * 4096) : "memory", "m0", "scc");
  };
  auto copy = [&](auto Kc) __attribute__((always_inline)) {
    constexpr int k = decltype(Kc)::value;
    const int v = (k < 8 ? vo_a[k & 7] : vo_b[k & 7]) | mask, off = koff;
    const i32x4_t r = k < 8 ? feed.ra : feed.rb;
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" : : "v"(v), "s"(r), "s"(off) : "memory");
  };
  // the scales of a tile's rows 64 wave .. + 63 and of its columns
  auto copy_scales = [&](const KgTile& t) __attribute__((always_inline)) {
    const int m_left = (int)p.m_total - t.m0, n_left = p.N - t.n0, v = lane * 4 + wave * 256;
    const i32x4_t rm = make_rsrc32((uint64_t)(p.scale_m + t.g * p.scale_m_sg + t.m0), (m_left < C::BM ? m_left : C::BM) * 4);
    const i32x4_t rn = make_rsrc32((uint64_t)(p.scale_n + (int64_t)t.g * p.N + t.n0), (n_left < C::BN ? n_left : C::BN) * 4);
    const uint32_t at = smem_addr + C::SCALE_OFF + wave * 256;
    asm volatile("s_nop 4\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds\n\ts_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dword %1, %3, 0 offen lds"
                 : : "s"(at), "v"(v), "s"(rm), "s"(rn), "n"(C::BM * 4) : "memory", "m0", "scc");
  };

  // A slab takes 128 bytes of rows that lie far apart, one line of each, which HBM serves slowly and late.  So once in two slabs the
  // rows' next two lines are touched (one word of each, into a sink in LDS) and wait in L2 when they are copied, the first two of a
  // tile at the start of the tile before, the next two when the copies, a slab and a half before the tile, have come to its second.  The
  // workgroups of an XCD that run together share their panels (the tiles of a run of 32 neighbours: nc columns by 32 / nc rows, or as
  // many as a group has), and each touches its part of them only: all of it by everybody costs more than it gains, and so does
  // a panel that nobody shares (outputs of a single column or row of tiles: 51 groups of 1316 x 208, 2900 tokens 125 -> 117 us, 2 of 208 x 4648, 8500
  // tokens 251 -> 230; parts for 32 / nc rows where a group has fewer: 71 of 1334 x 488, 2600 tokens 270 -> 262).
  // Rows a multiple of many KB apart crowd into few sets of L2, and touched lines leave it again before they are copied: 128 groups of 3072 x 4096,
  // 5120 tokens each, 655360 codes a row: 6161 us, untouched 6185, with twice the traffic; 655744 a row: 5658 and 6201.  32 groups, 1024 tokens
  // on average, 32768 a row: 435 and 461; 32896: 403 and 455.
  const int parts_b = max(1, min(tiles.tiles_m, 32 / tiles.nc));
  const int rows_a = tiles.nc > 1 ? (C::BM + tiles.nc - 1) / tiles.nc : 0, rows_b = parts_b > 1 ? (C::BN + parts_b - 1) / parts_b : 0;
  struct Part { int a, b; };  // the lane's offsets, kNoFetch beyond the workgroup's part
  auto part_of = [&](const KgTile& t) __attribute__((always_inline)) {
    const int mt = t.m0 >> 8, nt = t.n0 >> 8, part_a = nt - (int)tiles.by_nc.div((uint32_t)nt) * tiles.nc, part_b = mt % parts_b;
    const int thread = wave * 64 + lane;
    return Part{thread < rows_a ? (part_a * rows_a + thread) * ld : kNoFetch, thread < rows_b ? (part_b * rows_b + thread) * ld : kNoFetch};
  };
  auto touch = [&](const i32x4_t& r, int v0, int off, int klen) __attribute__((always_inline)) {
    const int v = off < klen ? v0 : kNoFetch;
    const uint32_t at = smem_addr + C::SINK_OFF + wave * 256;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dword %1, %2, %3 offen lds" : : "s"(at), "v"(v), "s"(r), "s"(off) : "memory", "m0");
  };
  auto touch_two = [&](const Feed& f, const Part& part, int off) __attribute__((always_inline)) {  // the lines at off and behind
    if (wave * 64 < rows_a) { touch(f.ra, part.a, off, f.klen); touch(f.ra, part.a, off + C::KS, f.klen); }
    if (wave * 64 < rows_b) { touch(f.rb, part.b, off, f.klen); touch(f.rb, part.b, off + C::KS, f.klen); }
  };
  Part part = {kNoFetch, kNoFetch};
  // ---- fragments and accumulators ----------------------------------------------------------------------------------------------
  i32x8_t fa[8], fb[8];
  f32x4_t acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto read_a = [&](auto Ic) __attribute__((always_inline)) { read_frag8<decltype(Ic)::value * 2048>(fa[decltype(Ic)::value], a_rd[0], a_rd[1]); };
  auto read_b = [&](auto Jc) __attribute__((always_inline)) { read_frag8<decltype(Jc)::value * 2048>(fb[decltype(Jc)::value], b_rd[0], b_rd[1]); };
  auto toggle = [&](uint32_t& at) __attribute__((always_inline)) { asm volatile("v_xor_b32 %0, 0x10000, %0" : "+v"(at)); };

  // ---- epilogue ------------------------------------------------------------------------------------------------------------------
  i32x4_t pend_rs = make_rsrc32(0, 0);
  int pend_cols = 0;
  const float* const scale_m = reinterpret_cast<const float*>(smem + C::SCALE_OFF);
  struct Epi { f32x4_t cs[2], rs; int off; };  // the lane's eight column scales, its four row scales of the strip, its output offset
  auto epi_begin = [&](Epi& e) __attribute__((always_inline)) {
    int el = lane;
    asm volatile("" : "+v"(el));
    const int col = (el & 15) * 8;
    e.off = col < pend_cols ? ((el >> 4) * 4 * p.N + col) * 2 : kNoFetch;
    const f32x4_t* const c = reinterpret_cast<const f32x4_t*>(scale_m + C::BM + wn0 + col);
    e.cs[0] = c[0];
    e.cs[1] = c[1];
    asm volatile("" ::: "memory");
  };
  auto epi_rows = [&](Epi& e, int i) __attribute__((always_inline)) {
    e.rs = *reinterpret_cast<const f32x4_t*>(scale_m + wm0 + 16 * i + 4 * lg);
    asm volatile("" ::: "memory");
  };
  // outputs 4 h .. 4 h + 3 of the lane's eight in row r of strip i, not before this point in the instruction stream
  auto epi_half = [&](const Epi& e, int i, int r, int h) __attribute__((always_inline)) {
    asm volatile("" : "+a"(acc[i][4 * h]), "+a"(acc[i][4 * h + 1]), "+a"(acc[i][4 * h + 2]), "+a"(acc[i][4 * h + 3]));
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = acc[i][4 * h + q][r] * e.rs[r] * e.cs[h][q];
    uint2 x;
    x.x = pack2<OUT>(v[0], v[1]);
    x.y = pack2<OUT>(v[2], v[3]);
    asm volatile("" : "+v"(x.x), "+v"(x.y));
    return x;
  };
  auto epi_store = [&](const Epi& e, int i, int r, const uint2& x, const uint2& y) __attribute__((always_inline)) {
    i32x4_t v;
    v[0] = (int)x.x; v[1] = (int)x.y; v[2] = (int)y.x; v[3] = (int)y.y;
    const int off = e.off + (16 * i + r) * p.N * 2;
    // the data registers of a 16-byte store must not be overwritten within two wait states (assembly_checks.py)
    asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen nt\n\ts_nop 1" : : "v"(v), "v"(off), "s"(pend_rs) : "memory");
  };
  auto epi_flush = [&]() __attribute__((always_inline)) {  // row blocks 4-7 of the workgroup's last tile
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" : "+a"(acc[4][3]), "+a"(acc[5][3]), "+a"(acc[6][3]), "+a"(acc[7][3]));
    Epi e;
    epi_begin(e);
#pragma unroll
    for (int i = 4; i < 8; ++i) {
      epi_rows(e, i);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint2 x = epi_half(e, i, r, 0), y = epi_half(e, i, r, 1);
        epi_store(e, i, r, x, y);
      }
    }
  };

  // ---- prologue: slabs 0 and 1 of the first tile, the fragments that group 0 expects ---------------------------------------------------
#define TGG_F8_I(k) std::integral_constant<int, k>()
#define TGG_F8_EACH16(f) f(0) f(1) f(2) f(3) f(4) f(5) f(6) f(7) f(8) f(9) f(10) f(11) f(12) f(13) f(14) f(15)
  __syncthreads();
  draw.request();
  wait_vmcnt<0>();
  draw.take(0);
  __syncthreads();
  KgTile cur = tiles.look_up(draw.tile_at(0)), following = cur;
  feed = feed_of(cur);
  nxt = feed;
  draw.request();
  for (int s = 0; s < 2; ++s) {
    step_feed();
    asm volatile("s_nop 4" ::: "memory");
#define TGG_F8_P(k) copy_m0(TGG_F8_I(k)); asm volatile("s_nop 0" ::: "memory"); copy(TGG_F8_I(k));
    TGG_F8_EACH16(TGG_F8_P)
#undef TGG_F8_P
    cp_buf ^= C::STAGE_BYTES;
  }
  wait_vmcnt<0>();
  draw.take(1);
  __syncthreads();
  read_a(TGG_F8_I(0)); read_a(TGG_F8_I(1)); read_a(TGG_F8_I(2)); read_a(TGG_F8_I(3));
  read_b(TGG_F8_I(4)); read_b(TGG_F8_I(5)); read_b(TGG_F8_I(0)); read_b(TGG_F8_I(1)); read_b(TGG_F8_I(2));

  // One slab.  EPI 0: an inner one of a tile, 1: its first, 2: its last.  STORES: output stores behind the copies of the next slab.
  auto slab = [&](auto EPIc, auto STORESc, int pos) __attribute__((always_inline)) {
    constexpr int EPI = decltype(EPIc)::value, STORES = decltype(STORESc)::value;
    Epi e = {};
    uint2 ex = {0, 0};
    // unit u = 4 (strip of the half) + r, halves 2 u and 2 u + 1, spread over the half slab's gaps behind its third multiply
    auto epi_gap = [&](auto Nc, auto S0c) __attribute__((always_inline)) {
      constexpr int n = decltype(Nc)::value, S0 = decltype(S0c)::value;
      if constexpr (n == 0) epi_begin(e);
      for_each<32>([&](auto Uc) __attribute__((always_inline)) {
        constexpr int half = decltype(Uc)::value, u = half / 2;
        if constexpr (3 + half * 28 / 32 == n) {
          if constexpr (half % 8 == 0) epi_rows(e, S0 + u / 4);
          if constexpr (half % 2 == 0) ex = epi_half(e, S0 + u / 4, u % 4, 0);
          else epi_store(e, S0 + u / 4, u % 4, ex, epi_half(e, S0 + u / 4, u % 4, 1));
        }
      });
    };
    for_each<64>([&](auto Nc) __attribute__((always_inline)) {
      constexpr int n = decltype(Nc)::value, g = n / 4, q = g / 4;
      constexpr int j = q == 0 ? g : q == 1 ? g : q == 2 ? 15 - g : g - 12;
      constexpr int ii = (g & 1) ? 3 - n % 4 : n % 4, i = (q < 2 ? 0 : 4) + ii;  // snake order
      if constexpr (n % 4 == 0) {  // the group's fragments have arrived
        if constexpr (g == 0) asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(fa[0]), "+v"(fa[1]), "+v"(fa[2]), "+v"(fa[3]), "+v"(fb[0]) : : "memory");
        if constexpr (g == 1) asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(fb[1]) : : "memory");
        if constexpr (g == 2) asm volatile("s_waitcnt lgkmcnt(6)" : "+v"(fb[2]) : : "memory");
        if constexpr (g == 3) asm volatile("s_waitcnt lgkmcnt(6)" : "+v"(fb[3]), "+v"(fb[4]), "+v"(fb[5]) : : "memory");
        if constexpr (g == 6) asm volatile("s_waitcnt lgkmcnt(8)" : "+v"(fb[6]), "+v"(fb[7]) : : "memory");
        if constexpr (g == 8) {
          asm volatile("s_waitcnt vmcnt(%4) lgkmcnt(0)" : "+v"(fa[4]), "+v"(fa[5]), "+v"(fa[6]), "+v"(fa[7]) : "n"(STORES) : "memory", "v255");
          if constexpr (EPI == 2) draw.take(pos + 2);
          asm volatile("s_barrier" ::: "memory");
          if constexpr (EPI == 1) copy_scales(cur);
        }
      }
      if constexpr (EPI == 1) mfma8_new<FA, FB>(acc[i][j], fa[i], fb[j]);
      else mfma8_acc<FA, FB>(acc[i][j], fa[i], fb[j]);
      if constexpr (n % 4 == 0) {
        if constexpr (g == 0) read_b(TGG_F8_I(3));
        if constexpr (g == 1) { read_b(TGG_F8_I(6)); read_b(TGG_F8_I(7)); }
        if constexpr (g >= 2 && g < 6) read_a(TGG_F8_I(g + 2));
        if constexpr (g == 6) { toggle(a_rd[0]); toggle(a_rd[1]); toggle(b_rd[0]); toggle(b_rd[1]); step_feed(); }
        if constexpr (g >= 8 && g < 12) read_a(TGG_F8_I(g - 8));
        if constexpr (g == 12) { read_b(TGG_F8_I(4)); read_b(TGG_F8_I(5)); }
        if constexpr (g >= 13) read_b(TGG_F8_I(g - 13));
      }
      if constexpr (n >= 32 && n % 2 == 0) copy_m0(TGG_F8_I((n - 32) / 2));
      if constexpr (n >= 32 && n % 2 == 1) copy(TGG_F8_I((n - 33) / 2));
      if constexpr (n == 63) {
        // the first two lines of a tile have been touched before, and its last slab requests the next tile's second
        if (EPI != 2 && (koff & C::KS) != 0) touch_two(feed, part, koff + C::KS);
      }
      if constexpr (EPI == 1 && n < 32) epi_gap(Nc, TGG_F8_I(4));
      if constexpr (EPI == 2 && n >= 32) epi_gap(TGG_F8_I(n - 32), TGG_F8_I(0));
    });
    cp_buf ^= C::STAGE_BYTES;
  };
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<int, 16> S16;
  for (int pos = 0; cur.g >= 0; ++pos) {
    following = tiles.look_up(draw.tile_at(pos + 1));
    nxt = feed_of(following);
    touch_two(nxt, part_of(following), 0);
    part = part_of(cur);
    const int steps = steps_of(cur);
    if (steps == 2) draw.request();
    // the launch's first slab finds the slab behind it landed; later first slabs have the sixteen stores of row blocks 4-7 behind the copies
    slab(I1(), S16(), pos);
    for (int k = 2; k < steps; ++k) {
      if (k + 1 == steps) draw.request();  // the answer is taken a slab and a half later
      slab(I0(), I0(), pos);
    }
    const int64_t rows_left = p.m_total - cur.m0 - wm0;
    pend_rs = make_rsrc32((uint64_t)p.C + (uint64_t)((((int64_t)cur.g * p.m_total + cur.m0 + wm0) * (int64_t)p.N + cur.n0 + wn0) * 2),
                          rows_left > 0 && (!SPLIT || cur.slot < 0) ? (int)(rows_left < 128 ? rows_left : 128) * p.N * 2 : 0);
    pend_cols = p.N - cur.n0 - wn0;
    slab(I2(), I0(), pos);
    if constexpr (SPLIT) {
      if (cur.slot >= 0) store_part(acc, p.split_ws, (int64_t)cur.slot * tiles.per_group + (cur.m0 >> 8) * ((p.N + 255) >> 8) + (cur.n0 >> 8), wave, lane);
    }
    touch_two(feed, part_of(following), 2 * C::KS);
    cur = following;
  }
  epi_flush();
  draw.finish();
  wait_vmcnt<0>();  // trailing copies that fetch nothing still write LDS
#undef TGG_F8_I
#undef TGG_F8_EACH16
}

template <int FA, int FB, int OUT, bool SPLIT>
int launch_cfg(const GemmParams& p, hipStream_t s) {
  static bool attr_set[64] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  const bool listed = dev >= 0 && dev < 64;
  auto kern = fp8_w4_kernel<FA, FB, OUT, SPLIT>;
  if (!listed || !attr_set[dev]) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Fp8W4Cfg::SMEM_BYTES) != hipSuccess)
      return check_launch("hipFuncSetAttribute(fp8_w4)");
    if (listed) attr_set[dev] = true;
  }
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(Fp8W4Cfg::THREADS), Fp8W4Cfg::SMEM_BYTES, s, p);
  return check_launch("fp8_w4");
}

}  // namespace

// What its table and offsets allow, but for outputs of a single column of tiles over long segments, which wait for the rows of A, shared by
// nobody, and get them no sooner here.  650 random launches of 64-6144 columns and 16-16000 tokens a group, operands in no cache: 0.94 of the
// eight-wave kernel's time in the mean (0.69-1.11) with N > 256, 0.95 with N <= 256 and fewer than 1000 tokens, 1.04 with 1000 and more
// (0.89-1.16: 89 groups of 1850 x 136, 2100 tokens 183 us and 157 there, 4 of 4251 x 144, 1400 tokens 46 and 41).
bool fp8_w4_supported(const GemmParams& p, bool any_size) {
  if (p.mode != MODE_KG_COUNT) return false;
  if (p.G > Fp8W4Cfg::THREADS || (p.N & 7) != 0 || (p.k_total & 15) != 0) return false;
  // a tile's window of either operand, and a wave's block of the output, within 32-bit offsets below the out-of-range marker
  if (p.k_total * 256 >= (1ll << 30) || (int64_t)p.N * 2 * 128 >= (1ll << 30)) return false;
  if (p.G * ((p.m_total + 255) / 256) * (((int64_t)p.N + 255) / 256) >= (1ll << 31)) return false;
  return any_size || p.N > Fp8W4Cfg::BN || p.k_total < 1000 * (int64_t)p.G;
}

int64_t fp8_w4_split_bytes(const GemmParams& p) { return fp8_w4_supported(p, true) ? split_bytes(p, 4000, 16000) : 0; }

template <bool SPLIT>
static int launch_formats(const GemmParams& p, int ta, int tb, hipStream_t s) {
  if (ta == DT_E4M3) return tb == DT_E4M3 ? launch_cfg<0, 0, DT_BF16, SPLIT>(p, s) : launch_cfg<0, 1, DT_BF16, SPLIT>(p, s);
  return tb == DT_E4M3 ? launch_cfg<1, 0, DT_BF16, SPLIT>(p, s) : launch_cfg<1, 1, DT_BF16, SPLIT>(p, s);
}

int launch_fp8_w4(const GemmParams& p, int ta, int tb, hipStream_t s) {
  if (!p.split_ws) return launch_formats<false>(p, ta, tb, s);
  if (int e = launch_formats<true>(p, ta, tb, s)) return e;
  return launch_split_sum<DT_BF16, true>(p, s);
}

}  // namespace tgg
