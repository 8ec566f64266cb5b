// Four-wave bf16/fp16 grouped GEMM kernel for gfx950: the large-problem path of the M-grouped and masked entry points
// (B as [G, N, K] or as [G, K, N]).
//
// One workgroup per CU, four waves, one per SIMD; tile 256x256, K slab 64; every wave owns a 128x128 block of
// 16x16x32 MFMA tiles with its 256 accumulator registers in AGPRs.  Against the eight-wave kernel (gemm_fast.hip,
// 128x64 per wave) a K step needs a third fewer LDS fragment reads per multiply.  With a single wave per SIMD there
// is nobody to interleave with, so the instruction order *is* the schedule: the slab loop is a sequence of
// inline-assembly statements (multiplies, fragment reads, copies, waits), which the compiler keeps in source order and
// only allocates registers for.  What the order has to respect (measured with a stream of multiplies and one kind
// of instruction between them): a wave issues in order and a multiply keeps the matrix pipe busy for 16 cycles, so
// one or two other instructions between two multiplies cost nothing, three or four cost 4-10 cycles of pipe time,
// and a 16-byte-per-lane LDS write costs 13 cycles on its own (33 next to fragment reads).  Hence: never more than
// two instructions in a gap of the slab loop proper, m0 written a multiply ahead of the copy that needs it, every per-copy address in a
// register or an immediate, and the per-slab bookkeeping down to an offset and three selects per cursor.
//
// Per slab r (two LDS slab buffers, r % 2; two register sets for A chunks), per wave:
//   K step 0   64 multiplies on fragment set 0; meanwhile the 16 fragments of K step 1 are read into set 1, the A
//              chunks of slab r+1 go from their register set to LDS and the A chunks of slab r+3 are requested
//              into that set
//   wait for the fragment reads and for this wave's B copies of slab r+1, workgroup barrier
//   K step 1   64 multiplies on set 1; meanwhile the fragments of slab r+1 / K step 0 are read into set 0 and
//              this wave's B copies of slab r+2 go straight to LDS, into the buffer of slab r
// Within a K step the sixteen fragment reads follow the first sixteen multiplies, one each; the LDS writes with their
// reloads, or the copies, follow from the seventeenth multiply on, one every fourth or fifth multiply (fragment
// reads and 16-byte LDS writes slow each other down when they alternate).
// A is the operand that streams from memory (B panels are shared through L2), so it is requested two slabs
// earlier than an LDS buffer is free for it: worth 3 % over copying it straight to LDS a slab ahead, although
// the LDS writes cost more than that copy would.  The slabs of all of a workgroup's tiles form one stream; each
// of the two cursors carries the buffer descriptor of its tile's window and an offset along K.
//
// A tile of at most 128 rows (a group's last one, mostly) is a half tile: the two wave rows take 64 rows each, four row blocks per wave, and a K step is 32
// multiplies; its results leave behind its last K step.  So that a wave's fragments may lie elsewhere in the two kinds, all fragments and
// accumulators are named registers.  Before, the zeros that such a tile's windows deliver were multiplied (masked launches: waves without rows
// sat the tile out).  128 groups, 32768 rows, same box: N = 1536, K = 2048 274 -> 265 us, as [K, N] N = 2048, K = 1536 287 -> 278; 32 groups,
// 16384 rows, N = 2048, K = 2880 220 -> 215; headline and masked decode the same.
//
// The epilogue rides on multiplies: the upper half of a wave's block is converted and stored between the multiplies
// of the tile's last K step, the lower half between those of the next tile's first K step, whose multiplies start
// from a zero addend instead of the accumulators (see "epilogue" below).  With B as [G, N, K] the results never pass
// through LDS: the rows of a B slab sit in LDS in an order that makes each lane's results of the eight column blocks
// eight neighbouring outputs of a row.  Measured on the headline shape: staging a tile's results in LDS costs 9 % of
// a launch in LDS bandwidth however it is spread over those two K steps (fragment reads already take half of it);
// exchanging halves between lane groups instead gives 16 rows x 64 bytes per store, whose lanes four by four lie in
// different rows, and costs 6 % more than staging; the permuted slab rows give 4 rows x 256 bytes per store and
// cost nothing.  What remains of the epilogue is the write traffic itself (6 % of a launch against stores that
// write nothing).
//
// Headline shape (G = 128, M = 655360, N = 1536, K = 2048), same box: 3.03 ms against 3.30 ms for the eight-wave
// kernel; K = 768 shape 1.77 against 1.97 ms; masked decode (G = 128, up to 512 rows per group, N = 4096, K = 1536)
// 0.51 against 0.56 ms.  Large M-grouped launches of 512 rows a group and more take this kernel (w4_supported); masked launches of that size, M-grouped
// ones of smaller groups and those of at most four rounds that are likely to be its enqueue it together with the eight-wave kernel, and the sizes decide on
// the device which of the two runs (GemmParams::wide_gate).  Launches of few tiles have gone to gemm_deep.hip before this is asked; the rest are
// the eight-wave kernels'.
//
// What the compiler does not know about assembly statements, and how it is handled here:
//   * fragments and accumulators are named in the instruction text and waited for by the K step's wait statement; the compiler's own allocation
//     is kept below them (amdgpu_num_vgpr; the build fails where its assembly shows any other use, assembly_checks.py);
//   * the A chunks are in flight across loop iterations and paths that join: their registers (v[192:255]) are named
//     in the instruction text too;
//   * the multiplies write AGPRs: the epilogue's conversions read a block's accumulators no sooner
//     than three multiplies after the multiply that wrote them (a multiply takes 16 cycles to issue and delivers
//     within two more), except where a flush follows a tile directly: there the last row block's accumulators pass
//     through a statement of idle cycles first.  Accumulators are never the target of a load.
#include "launch.hpp"
#include "w4_common.hpp"

namespace tgg {

namespace {

enum : int { W4_NT = 0, W4_NN = 1 };
constexpr int BK4 = 64;

#define TGG_W4_ACC_CLOBBER "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", "a16", "a17", "a18", "a19", "a20", "a21", \
  "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", \
  "a44", "a45", "a46", "a47", "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", "a64", "a65", \
  "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", \
  "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", \
  "a110", "a111", "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127", "a128", "a129", "a130", "a131", \
  "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", \
  "a154", "a155", "a156", "a157", "a158", "a159", "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", \
  "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191", "a192", "a193", "a194", "a195", "a196", "a197", \
  "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", \
  "a220", "a221", "a222", "a223", "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", "a240", "a241", \
  "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"
#define TGG_W4_I(k) std::integral_constant<int, (k)>()

// Registers by number (see "fragments and accumulators"): FA, FB the fragments' first VGPR, AT the accumulators' first AGPR.
template <int DT, bool FRESH, int AT, int X, int Y> TGG_DEV void acc_mfma() {
  if constexpr (DT == DT_BF16 && FRESH) asm volatile("v_mfma_f32_16x16x32_bf16 a[%c0:%c1], v[%c2:%c3], v[%c4:%c5], 0" : : "n"(AT), "n"(AT + 3), "n"(X), "n"(X + 3), "n"(Y), "n"(Y + 3));
  else if constexpr (DT == DT_BF16) asm volatile("v_mfma_f32_16x16x32_bf16 a[%c0:%c1], v[%c2:%c3], v[%c4:%c5], a[%c0:%c1]" : : "n"(AT), "n"(AT + 3), "n"(X), "n"(X + 3), "n"(Y), "n"(Y + 3));
  else if constexpr (FRESH) asm volatile("v_mfma_f32_16x16x32_f16 a[%c0:%c1], v[%c2:%c3], v[%c4:%c5], 0" : : "n"(AT), "n"(AT + 3), "n"(X), "n"(X + 3), "n"(Y), "n"(Y + 3));
  else asm volatile("v_mfma_f32_16x16x32_f16 a[%c0:%c1], v[%c2:%c3], v[%c4:%c5], a[%c0:%c1]" : : "n"(AT), "n"(AT + 3), "n"(X), "n"(X + 3), "n"(Y), "n"(Y + 3));
}
template <int V, int OFF> TGG_DEV void frag_read_b128(uint32_t addr) {
  asm volatile("ds_read_b128 v[%c1:%c2], %0 offset:%c3" : : "v"(addr), "n"(V), "n"(V + 3), "n"(OFF) : "memory");
}
template <int V, int OFF0, int OFF1> TGG_DEV void frag_read_tr(uint32_t addr) {  // two transposing 8-byte reads (K 0..3 and 4..7 of the lane's column)
  asm volatile("ds_read_b64_tr_b16 v[%c1:%c2], %0 offset:%c5\n\tds_read_b64_tr_b16 v[%c3:%c4], %0 offset:%c6"
               : : "v"(addr), "n"(V), "n"(V + 1), "n"(V + 2), "n"(V + 3), "n"(OFF0), "n"(OFF1) : "memory");
}
template <int AT> TGG_DEV float acc_read() {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, a%c1" : "=v"(v) : "n"(AT));
  return v;
}
template <int AT> TGG_DEV void acc_zero() {
  asm volatile("v_accvgpr_write_b32 a%c0, 0\n\tv_accvgpr_write_b32 a%c1, 0\n\tv_accvgpr_write_b32 a%c2, 0\n\tv_accvgpr_write_b32 a%c3, 0" : : "n"(AT), "n"(AT + 1), "n"(AT + 2), "n"(AT + 3));
}

struct W4Cfg {
  static constexpr int BM = 256, BN = 256, NWAVES = 4, THREADS = 256;
  static constexpr int A_BYTES = BM * BK4 * 2, B_BYTES = BN * BK4 * 2, STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int NI_A = A_BYTES / 1024, NI_B = B_BYTES / 1024;
  static constexpr int TM = 8, TN = 8;                       // 16x16 blocks per wave: 128 x 128
  static constexpr int EPI_PITCH = 4 * 32 + 16;              // epilogue staging (B as [G, K, N] only); a piece: 16 rows x 64 outputs, row pitch in bytes
  static constexpr int EPI_PIECE = 16 * EPI_PITCH;
  static constexpr int EPI_WAVE_BYTES = 2 * EPI_PIECE;       // two pieces alternate
  static constexpr int SCHED_OFF = 2 * STAGE_BYTES;
  static constexpr int EPI_OFF = SCHED_OFF + (((int)sizeof(SchedTableT<kFastMaxGroups>) + 255) & ~255);
  static constexpr int SMEM_BYTES = EPI_OFF + NWAVES * EPI_WAVE_BYTES;
  static_assert(SMEM_BYTES <= 160 * 1024, "LDS budget");
};

// A is the operand that takes the long way through registers ("staged", s), B is copied straight to LDS ("direct",
// d).  Staging B instead makes no difference even where the weights are what streams from memory (masked decode:
// 0.526 ms either way).
// TAIL: K is any multiple of 8 from 192 on, and N, for B as [G, K, N], any multiple of 8.  A tile's last slabs are cut short (or
// added, for an even number of four at least): lanes whose chunk of a K-contiguous row starts at or beyond K get an out-of-range
// offset, and token rows beyond K lie behind the window's end.  An instantiation of its own: the plain one needs no mask.
template <int DT, int LAYOUT, bool TAIL>
__global__ __launch_bounds__(W4Cfg::THREADS) __attribute__((amdgpu_num_vgpr(64))) void gemm_w4_kernel(const GemmParams p) {
  typedef W4Cfg C;
  constexpr int S_OFF = 0, D_OFF = C::A_BYTES;  // the operands' places in a slab buffer
  constexpr bool B_KMAJOR = LAYOUT == W4_NT;  // NN: B is [G, K, N], its slab 64 token rows of 512 bytes
  typedef Operand<C::BM, true> Op;            // the A slab, and B's when K-contiguous: 256 rows of 128 bytes
  typedef Operand<C::BN, B_KMAJOR> OpB;

  extern __shared__ __attribute__((aligned(1024))) char smem[];
  auto& sched = *reinterpret_cast<SchedTableT<kFastMaxGroups>*>(smem + C::SCHED_OFF);
  sched_init<C::BM>(p, sched);
  // a launch that pays only with sizes for 256x256 tiles (GemmParams::wide_gate):
  // the same predicate on the same table decides there that the eight-wave launch behind this one has nothing to do
  if (p.wide_gate == 1 && !sched_wide_tiles_chosen<C::BM, C::BN>(p, sched)) return;
  const int num_tiles = (int)sched_num_tiles<C::BM, C::BN>(p, sched);

  const uint32_t smem_addr = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave_m = wave >> 1, wn0 = (wave & 1) * 128;
  const int l16 = lane & 15, lg = lane >> 4;

  const int ld = p.K * 2;  // row pitch of A and of B in bytes; K is a multiple of 128 (w4_supported) unless TAIL
  const int kt_all = TAIL ? max(4, (p.K + 2 * BK4 - 1) / (2 * BK4) * 2) : p.K / BK4;  // slabs per tile
  // Copy k (0..7) of an operand's slab by this wave is copy instruction wave + 4 k of the slab: rows 8 (wave + 4 k) ...
  // + 7.  Its per-lane source offset within the tile's window is fixed for the launch and kept in a register; the slab's offset along K travels in the
  // instruction's scalar offset, which the range check of the window counts in: rows behind the valid ones stay behind its end.  One register for all
  // copies, with their distances from the first added to the scalar offset in front of each, costs 1.5 % of a launch (64 groups, 126593 rows, N = 4096,
  // K = 3072: 2.43 against 2.38 ms); the empty statements keep the compiler from computing the offsets anew instead.
  int vo[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    vo[k] = Op::lane_voff(lane, wave % Op::NPAT, ld) + (wave + 4 * k) * Op::RPI * ld;
    asm volatile("" : "+v"(vo[k]));
  }
  static_assert(Op::NPAT == 2, "the swizzle pattern of copy wave + 4 k is that of copy wave");
  // NN: B's copies have offsets of their own (two token rows of 512 bytes per copy, row pitch 2 N)
  const int ld_b = (B_KMAJOR ? p.K : p.N) * 2;
  // NT: B's rows land in LDS permuted: LDS row 128 h + 16 j + c of the slab (column block j of a wave's half h, lane
  // column c of the multiply) holds column 128 h + 8 c + j of the tile, so that a lane's results of the eight column
  // blocks are eight neighbouring outputs of a row and leave as one 16-byte store without passing through LDS.
  // LDS row 8 (wave + 4 k) + lane / 8: h = k / 4, j = 2 (k % 4) + wave / 2, c = 8 (wave % 2) + lane / 8
  int vo_b[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    vo_b[k] = B_KMAJOR ? Op::lane_voff(lane, wave % Op::NPAT, ld) + (8 * (8 * (wave & 1) + lane / Op::CPR) + (wave >> 1) - lane / Op::CPR + 128 * (k >> 2) + 2 * (k & 3)) * ld
                       : OpB::lane_voff(lane, (wave + 4 * k) % OpB::NPAT, ld_b) + (wave + 4 * k) * OpB::RPI * ld_b;
    asm volatile("" : "+v"(vo_b[k]));
  }

  // LDS addresses of the fragment reads relative to a slab buffer (see gemm_fast.hip for the layout)
  uint32_t a_rd[2], b_rd[B_KMAJOR ? 2 : 8];
  auto set_a_rd = [&](int ks, const Tile& t) __attribute__((always_inline)) {  // for a tile's fragments of K step ks: the wave's rows are those of its height
    a_rd[ks] = smem_addr + (wave_m * (t.rows <= C::BM / 2 ? 64 : 128) + l16) * 128 + (((4 * ks + lg) ^ ((l16 / 2) % 8)) << 4);
  };
  if (B_KMAJOR) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) b_rd[ks] = smem_addr + C::A_BYTES + (wn0 + l16) * 128 + (((4 * ks + lg) ^ ((l16 / 2) % 8)) << 4);
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // per column block: token row 8 lg + e, 16-byte chunk of the lane's columns, swizzled
      const int e = l16 >> 2, c = l16 & 3;
      const int chunk = ((wn0 + 16 * j) / 8 + (c >> 1)) ^ (e * 4) ^ ((lg & 1) * 2);
      b_rd[B_KMAJOR ? 0 : j] = smem_addr + C::A_BYTES + (lg * 8 + e) * (C::BN * 2) + chunk * 16 + (c & 1) * 8;
    }
  }

  // ---- the copy stream --------------------------------------------------------------------------------------------
  // The slabs of all of this workgroup's tiles form one stream.  While slab r is multiplied, the B copies of slab
  // r + 2 go straight to LDS (into the buffer of slab r, free after the barrier in the middle of the slab) and the A
  // chunks of slab r + 3 are loaded into registers, from where the chunks of slab r + 1, loaded two slabs earlier,
  // have just been written to LDS: A is the operand that comes from memory, B panels are shared through L2.
  // Each of the two cursors holds the window (buffer descriptor) of the tile it is in and its offset along K.
  struct Win { i32x4_t rs, rd; };  // staged operand, directly copied operand
  auto window = [&](const Tile& t, bool live) __attribute__((always_inline))  {
    Win w;
    const int n_left = p.N - t.n0;
    w.rs = make_rsrc32((uint64_t)p.A + (uint64_t)(t.row0 * ld), live ? t.rows * ld : 0);  // only the tile's valid rows
    if (B_KMAJOR) w.rd = make_rsrc32((uint64_t)p.B + (uint64_t)(((int64_t)t.g * p.N + t.n0) * ld), live ? (n_left < C::BN ? n_left : C::BN) * ld : 0);
    // NN: the tile's 256 columns of the group's K rows, to the end of the last one.  What a row segment reads beyond its row are the
    // next row's first columns, for outputs that are not stored.
    else w.rd = make_rsrc32((uint64_t)p.B + (uint64_t)(((int64_t)t.g * p.K * p.N + t.n0) * 2), live ? p.K * ld_b - t.n0 * 2 : 0);
    return w;
  };
  const TileWalk walk64 = sched_walk(num_tiles, p.tile_split != 0);
  struct { int first, end, stride; } walk = {(int)walk64.first, (int)walk64.end, (int)walk64.stride};
  // A last round of at most half an XCD's workgroups is cut into half tiles, one each: tile ids from tail_first on count halves there.  The launch
  // ends with the time of a half tile in place of a whole one (8 groups, 11560 rows, N = 1536, K = 4096: 169 -> 153 us; 128 groups, 32768 rows,
  // N = 1536, K = 2048: 259 -> 250).  A longer last round is left whole: cut, it would be more than one half tile for some workgroup, as long as the whole.
  int tail_first = walk.end;
  if (p.tile_split != 0 && (gridDim.x & 7) == 0) {
    const int per_xcd = (int)gridDim.x >> 3, begin = walk.first - (int)(blockIdx.x >> 3), rest = (walk.end - begin) % per_xcd;
    if (2 * rest <= per_xcd) {
      tail_first = walk.end - rest;
      walk.end = tail_first + 2 * rest;
    }
  }
  const int row_bytes = __builtin_amdgcn_readfirstlane(ld);
  int hint_g = -1;
  auto tile_at = [&](int id, Tile& t) __attribute__((always_inline))  {  // false: the walk has ended
    if (id >= walk.end) { t.g = 0; t.row0 = 0; t.rows = 0; t.n0 = 0; t.k0 = t.k1 = 0; return false; }
    Tile v = sched_tile<C::BM, C::BN>(p, sched, id < tail_first ? id : tail_first + ((id - tail_first) >> 1), hint_g);
    if (id >= tail_first) {  // rows 0 .. 127 of the tile or those behind, if any
      const int at = ((id - tail_first) & 1) * (C::BM / 2), left = v.rows - at;
      v.row0 += at;
      v.rows = left < 0 ? 0 : (left < C::BM / 2 ? left : C::BM / 2);
    }
    // the same in every lane; in scalar registers, so that what depends on it branches as a wave
    t.g = __builtin_amdgcn_readfirstlane(v.g);
    t.row0 = (int64_t)uniform64((uint64_t)v.row0);
    t.rows = __builtin_amdgcn_readfirstlane(v.rows);
    t.n0 = __builtin_amdgcn_readfirstlane(v.n0);
    t.k0 = t.k1 = 0;
    hint_g = t.g;
    return true;
  };

  // The staged A chunks live in v[192:255] (two sets of eight), named in the instruction text like all fragments and accumulators.
#define TGG_W4_GA(c, f) \
  if (c == 0) { f("224", "227") } else if (c == 1) { f("228", "231") } else if (c == 2) { f("232", "235") } else if (c == 3) { f("236", "239") } \
  else if (c == 4) { f("240", "243") } else if (c == 5) { f("244", "247") } else if (c == 6) { f("248", "251") } else if (c == 7) { f("252", "255") } \
  else if (c == 8) { f("192", "195") } else if (c == 9) { f("196", "199") } else if (c == 10) { f("200", "203") } else if (c == 11) { f("204", "207") } \
  else if (c == 12) { f("208", "211") } else if (c == 13) { f("212", "215") } else if (c == 14) { f("216", "219") } else { f("220", "223") }
#define TGG_W4_GA_CLOBBER "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199", "v200", "v201", "v202", "v203", "v204", "v205", "v206", "v207", \
  "v208", "v209", "v210", "v211", "v212", "v213", "v214", "v215", "v216", "v217", "v218", "v219", "v220", "v221", "v222", "v223", "v224", "v225", "v226", "v227", \
  "v228", "v229", "v230", "v231", "v232", "v233", "v234", "v235", "v236", "v237", "v238", "v239", "v240", "v241", "v242", "v243", "v244", "v245", "v246", "v247", \
  "v248", "v249", "v250", "v251", "v252", "v253", "v254", "v255"
  int mask_s = 0, mask_d = 0;  // TAIL: kNoFetch in the lanes whose chunk of the cursor's slab lies beyond K
  const int chunk_off = Op::lane_chunk(lane, wave % Op::NPAT) * 16;
  const uint32_t s_wr = smem_addr + S_OFF + wave * 1024 + lane * 16;  // LDS address of this lane's 16 bytes of A copy 0 (buffer 0)
  // A chunk k of the slab at offset koff of window ra -> register set SET
  auto load_s = [&](auto Kc, auto SETc, const i32x4_t& ra, int koff) __attribute__((always_inline))  {
    constexpr int k = decltype(Kc)::value, kq = k + 8 * decltype(SETc)::value;
    const int v = TAIL ? vo[k] | mask_s : vo[k];
#define TGG_W4_F(lo, hi) asm volatile("buffer_load_dwordx4 v[" lo ":" hi "], %0, %1, %2 offen" : : "v"(v), "s"(ra), "s"(koff) : "memory", TGG_W4_GA_CLOBBER);
    TGG_W4_GA(kq, TGG_W4_F)
#undef TGG_W4_F
  };
  // register set SET, chunk k -> LDS (wr_addr: s_wr + the buffer's offset)
  auto write_s = [&](auto Kc, auto SETc, uint32_t wr_addr) __attribute__((always_inline))  {
    constexpr int k = decltype(Kc)::value, kq = k + 8 * decltype(SETc)::value;
#define TGG_W4_F(lo, hi) asm volatile("ds_write_b128 %0, v[" lo ":" hi "] offset:%1" : : "v"(wr_addr), "n"(k * 4096) : "memory", TGG_W4_GA_CLOBBER);
    TGG_W4_GA(kq, TGG_W4_F)
#undef TGG_W4_F
  };
  // B copy k of the slab at offset koff of window rb, straight to LDS, in two statements a multiply apart: the LDS
  // address goes to m0 first (a copy to LDS needs a wait state after a write of m0; the multiply in between is one)
  auto copy_d_m0 = [&](auto Kc, uint32_t buf_addr) __attribute__((always_inline))  {
    constexpr int k = decltype(Kc)::value;
    asm volatile("s_add_u32 m0, %0, %1" : : "s"(buf_addr), "n"(D_OFF + 4 * k * 1024) : "memory", "m0", "scc");
  };
  auto copy_d = [&](auto Kc, const i32x4_t& rb, int koff) __attribute__((always_inline))  {
    constexpr int k = decltype(Kc)::value;
    const int v = TAIL && B_KMAJOR ? vo_b[k] | mask_d : vo_b[k];
    // (the staged chunks' registers are listed here too: the compiler must not hold a value in them in a K step without loads either)
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" : : "v"(v), "s"(rb), "s"(koff) : "memory", TGG_W4_GA_CLOBBER);
  };
  // a slab's A copy k straight to LDS (prologue only)
  auto copy_direct = [&](auto Kc, auto ISBc, const i32x4_t& ra, int koff, uint32_t buf_addr) __attribute__((always_inline))  {
    constexpr int k = decltype(Kc)::value;
    const int v = decltype(ISBc)::value ? vo_b[k] : vo[k];
    asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
                 : : "s"(buf_addr), "n"(4 * k * 1024), "v"(v), "s"(ra), "s"(koff) : "memory", "m0", "scc");
  };
  const uint32_t wave_buf = smem_addr + wave * 1024;  // copy `wave` of buffer 0's A slab

  // ---- fragments and accumulators --------------------------------------------------------------------------------
  // All of them are named in the instruction text: block (i, j)'s accumulators a[32 i + 4 j : + 3], A's fragment i of set s v[64 + 32 s + 4 i : + 3], B's
  // fragment j v[128 + 32 s + 4 j : + 3].  Full and half tiles leave and find different parts of them in use, and where such
  // paths join the compiler moves what it knows of from register to register.  Its own allocation ends below v64 (amdgpu_num_vgpr)
  // and has no AGPR (they are clobbered at every K step's end; assembly_checks.py looks at the assembly).
  for_each<64>([&](auto Bc) __attribute__((always_inline)) { acc_zero<4 * decltype(Bc)::value>(); });

  // read number q (0..15) of the fragments of K step KS of the slab at byte offset `buf_off`, into set SET: B fragments first
  // (the next step needs all of them at once), then A fragments in the order of use
  auto read_frag = [&](auto KSc, auto Qc, auto SETc, uint32_t buf_off) __attribute__((always_inline)) {
    constexpr int KS = decltype(KSc)::value, Q = decltype(Qc)::value, SET = 32 * decltype(SETc)::value;
    if constexpr (Q < 8 && B_KMAJOR) frag_read_b128<128 + SET + 4 * Q, Q * 2048>(b_rd[KS] + buf_off);
    else if constexpr (Q < 8) frag_read_tr<128 + SET + 4 * Q, KS * 32 * (C::BN * 2), KS * 32 * (C::BN * 2) + 4 * (C::BN * 2)>(b_rd[Q] + buf_off);
    else frag_read_b128<64 + SET + 4 * (Q - 8), (Q - 8) * 2048>(a_rd[KS] + buf_off);
  };
  // ---- epilogue ------------------------------------------------------------------------------------------------------
  // With one wave per SIMD nothing else would keep the matrix pipe busy while a wave converts and stores its 128x128
  // block, so the work sits in the gaps between multiplies: strips 0-3 (a strip: one 16-row block, 128 columns) during
  // the tile's last K step, each after its last multiply, strips 4-7 during the first K step of the workgroup's next
  // tile, each before the multiply that starts it afresh (that K step multiplies with a zero addend); a wave without
  // a next tile to multiply stores strips 4-7 in a flush.  Half a block's conversion per gap on average keeps the
  // gaps within what a multiply hides.
  // B as [G, N, K]: the multiply takes A's fragment as its first operand, so a lane holds rows 16 i + 4 lg + r
  // (r = 0..3) of one column per block, and the permuted slab rows (vo_b) make that column 8 l16 + j for block j:
  // the lane's eight blocks of a strip are 16 contiguous bytes of an output row, 16 lanes cover 256 bytes of it, and
  // a store instruction writes 4 rows x 256 bytes.
  // B as [G, K, N] (fragments come from transposing reads, which tie a lane's column to its number): B's fragment is
  // the first operand, a lane owns row l16 and columns 16 j + 4 lg + (0..3) of block (i, j); a strip goes through the
  // wave's LDS staging as two pieces of 64 columns and leaves as 16-byte stores covering 128-byte row segments.
  // The stores go through a buffer descriptor over the wave's block that ends with its last valid row; lanes whose
  // columns lie beyond N get an out-of-range offset: no branches.
  // Nothing pending = a descriptor of length zero.
  i32x4_t pend_rs = make_rsrc32(0, 0);
  int pend_cols = 0;
  bool pending = false;
  char* const stage = smem + C::EPI_OFF + wave * C::EPI_WAVE_BYTES;
  // per-lane staging addresses and output offset, recomputed where a first K step or a flush begins
  struct EpiLane { char* wr; const char* rd; int off[2]; };  // off[h]: output offset of the lane's 16 bytes in column half h of strip 0, out of range where those columns lie beyond N
  auto epi_lane = [&]() __attribute__((always_inline))  {
    int el = lane;
    asm volatile("" : "+v"(el));
    EpiLane e;
    e.wr = stage + (el & 15) * C::EPI_PITCH + (el >> 4) * 8;
    e.rd = stage + (el >> 3) * C::EPI_PITCH + (el & 7) * 16;
    const int off = ((el >> 3) * p.N + (el & 7) * 8) * 2, ch8 = (el & 7) * 8;
#pragma unroll
    for (int h = 0; h < 2; ++h) e.off[h] = (64 * h + ch8 < pend_cols) ? off + 128 * h : kNoFetch;
    return e;
  };
  // block (i, j) -> staging piece j / 4; not before this point in the instruction stream
  auto epi_cvt = [&](const EpiLane& e, auto Ic, auto Jc) __attribute__((always_inline))  {
    constexpr int j = decltype(Jc)::value, at = 32 * decltype(Ic)::value + 4 * j;
    *(uint2*)(e.wr + (j >> 2) * C::EPI_PIECE + (j & 3) * 32) = pack4<DT>(acc_read<at>(), acc_read<at + 1>(), acc_read<at + 2>(), acc_read<at + 3>());
    asm volatile("" ::: "memory");
  };
  auto epi_read = [&](const EpiLane& e, int h, i32x4_t (&v)[2]) {
#pragma unroll
    for (int it = 0; it < 2; ++it) v[it] = *(const i32x4_t*)(e.rd + h * C::EPI_PIECE + it * 8 * C::EPI_PITCH);
    asm volatile("" ::: "memory");
  };
  auto epi_store = [&](const EpiLane& e, int i, int h, int it, const i32x4_t& v, bool between_multiplies) __attribute__((always_inline))  {
    // (an out-of-range marker stays out of range with the rows' offset added: both are far below 2^31)
    const int off = e.off[h] + (16 * i + 8 * it) * p.N * 2;
    // Two wait states must pass before a 16-byte store's data registers may be overwritten, and the compiler, which
    // considers them free after this statement, reuses them at once: between multiplies the multiply that follows is
    // one wait state (TAIL: a mask may come between them), the flush has none.  No wait states in front: the descriptor sits in scalar registers since the
    // end of the tile.  Both hazards are checked on the kept assembly (assembly_checks.py).
    if (between_multiplies && !TAIL) asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen nt\n\ts_nop 0" : : "v"(v), "v"(off), "s"(pend_rs) : "memory");
    else asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen nt\n\ts_nop 1" : : "v"(v), "v"(off), "s"(pend_rs) : "memory");
  };
  // NT: no staging.  A lane holds rows 16 i + 4 lg + r (r = 0..3) of column 8 l16 + j of the wave's block in
  // accumulator block (i, j), component r: the eight blocks of a strip give eight neighbouring outputs of a row.
  auto epi_lane_t = [&]() __attribute__((always_inline))  {
    int el = lane;
    asm volatile("" : "+v"(el));
    const int col = (el & 15) * 8;
    return col < pend_cols ? ((el >> 4) * 4 * p.N + col) * 2 : kNoFetch;
  };
  // outputs 4 h .. 4 h + 3 of the lane's eight in row r of strip i, converted; not before this point in the instruction stream
  auto epi_half_t = [&](auto Ic, auto Rc, auto Hc) __attribute__((always_inline))  {
    constexpr int at = 32 * decltype(Ic)::value + 16 * decltype(Hc)::value + decltype(Rc)::value;
    uint2 x;
    x.x = pack2<DT>(acc_read<at>(), acc_read<at + 4>());
    x.y = pack2<DT>(acc_read<at + 8>(), acc_read<at + 12>());
    asm volatile("" : "+v"(x.x), "+v"(x.y));
    return x;
  };
  auto epi_store_t = [&](int lane_off, int i, int r, const uint2& x, const uint2& y, bool between_multiplies) __attribute__((always_inline))  {
    i32x4_t v;
    v[0] = (int)x.x; v[1] = (int)x.y; v[2] = (int)y.x; v[3] = (int)y.y;
    const int off = lane_off + (16 * i + r) * p.N * 2;
    if (between_multiplies && !TAIL) asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen nt\n\ts_nop 0" : : "v"(v), "v"(off), "s"(pend_rs) : "memory");
    else asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen nt\n\ts_nop 1" : : "v"(v), "v"(off), "s"(pend_rs) : "memory");
  };
  // strips S0 .. S0 + 3 without multiplies to hide them under
  auto epi_strips = [&](auto S0c) __attribute__((always_inline))  {
    constexpr int S0 = decltype(S0c)::value;
    // the last row block's multiplies may have just been issued: give them time before the registers are read
    asm volatile("s_nop 15\n\ts_nop 7" : : : "memory");
    if constexpr (B_KMAJOR) {
      const int lane_off = epi_lane_t();
      for_each<16>([&](auto Uc) __attribute__((always_inline)) {
        constexpr int i = S0 + decltype(Uc)::value / 4, r = decltype(Uc)::value % 4;
        const uint2 x = epi_half_t(TGG_W4_I(i), TGG_W4_I(r), TGG_W4_I(0)), y = epi_half_t(TGG_W4_I(i), TGG_W4_I(r), TGG_W4_I(1));
        epi_store_t(lane_off, i, r, x, y, false);
      });
    } else {
      const EpiLane e = epi_lane();
      for_each<4>([&](auto Qc) __attribute__((always_inline)) {
        constexpr int i = S0 + decltype(Qc)::value;
        for_each<8>([&](auto Jc) __attribute__((always_inline)) { epi_cvt(e, TGG_W4_I(i), Jc); });
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          i32x4_t v[2];
          epi_read(e, h, v);
          epi_store(e, i, h, 0, v[0], false);
          epi_store(e, i, h, 1, v[1], false);
        }
      });
    }
  };
  // what a full tile has left pending
  auto epi_flush = [&]() __attribute__((always_inline))  {
    if (pending) epi_strips(std::integral_constant<int, 4>());
    pending = false;
    pend_rs[2] = 0;
  };


  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<bool, true> Yes;
  typedef std::integral_constant<bool, false> No;
  typedef std::integral_constant<int, 3> I3;
  typedef std::integral_constant<int, 4> I4;
  typedef std::integral_constant<int, 8> I8;

  // the two cursors of the copy stream and the tile after the one being multiplied
  i32x4_t rs_c, rd_c;
  int koff_s, koff_d;
  Win nxt;
  Tile nxt_tile;
  const int k_bytes = TAIL ? __builtin_amdgcn_readfirstlane(kt_all * 128) : row_bytes;  // a tile's extent along K in bytes: where a cursor moves on to the next tile
  // A cursor moves on to the next slab in four parts, one to a gap between two multiplies: where all of them stand in one gap the matrix pipe idles.
  bool wrap = false;
  auto advance_s = [&](int part) __attribute__((always_inline))  {
    __builtin_amdgcn_sched_barrier(0);
    if (part == 0) {
      wrap = koff_s + 128 == k_bytes;
      koff_s = wrap ? 0 : koff_s + 128;
    } else {
      rs_c[part - 1] = wrap ? nxt.rs[part - 1] : rs_c[part - 1];
      if (TAIL && part == 3) mask_s = koff_s + chunk_off >= row_bytes ? kNoFetch : 0;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int d_step = B_KMAJOR ? 128 : __builtin_amdgcn_readfirstlane(64 * ld_b);         // B's slab offset per slab ...
  const int d_bytes = B_KMAJOR ? k_bytes : __builtin_amdgcn_readfirstlane((TAIL ? kt_all * BK4 : p.K) * ld_b);   // ... and where it reaches the next tile
  auto advance_d = [&](int part) __attribute__((always_inline))  {
    __builtin_amdgcn_sched_barrier(0);
    if (part == 0) {
      wrap = koff_d + d_step == d_bytes;
      koff_d = wrap ? 0 : koff_d + d_step;
    } else {
      rd_c[part - 1] = wrap ? nxt.rd[part - 1] : rd_c[part - 1];
      if (TAIL && B_KMAJOR && part == 3) mask_d = koff_d + chunk_off >= row_bytes ? kNoFetch : 0;
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // One K step: 64 multiplies on fragment set CUR (when MUL); the 16 fragments of K step NKS of the slab at nb_off go
  // to the other set, one read after each of the first sixteen multiplies; the LDS writes and the loads and copies follow
  // behind them (reads and staged writes apart in time: 2.5 % over interleaving them through the whole K step; the
  // loads must not slip much later, a quarter of a slab less lead costs 6 %).  Outside the two K steps that carry
  // the epilogue at most two other instructions sit between two multiplies: a wave issues in order, and what exceeds
  // the sixteen cycles of a multiply leaves the matrix pipe idle.
  // ROLE 0: prologue (reads only, waits for everything).
  // ROLE 1: a slab's first K step.  The A chunks of the next slab go from register set SET to LDS (wr_addr) and the
  //         chunks of the slab three ahead are requested into the same set; ends with the wait for the B copies of
  //         the next slab (eight younger loads, and the 16 stores of a tile's first K step, may stay in flight; loads
  //         and stores complete in order, so the A chunks written here -- requested two slabs ago -- have arrived
  //         since the previous such wait).
  // ROLE 2: second K step: the B copies of the slab two ahead, into the buffer at cp_addr.
  // EPI 1: the first K step of a tile -- multiplies start from zero, strips 4-7 of the tile before are stored between
  //        them.  EPI 2: the last K step of a tile -- strips 0-3 are stored between its multiplies.
  // NS: row blocks of the tile per wave, eight, or four in a tile of at most 128 rows (no epilogue rides on its 32 multiplies; EPI 3:
  // they start from zero).  RD: fragments of A to read for the next K step.
  auto kstep = [&](auto CURc, auto NKSc, auto NSc, auto RDc, auto ROLEc, uint32_t nb_off, auto EPIc, uint32_t wr_addr, auto SETc, uint32_t cp_addr) __attribute__((always_inline))  {
    constexpr int CUR = decltype(CURc)::value, NKS = decltype(NKSc)::value, ROLE = decltype(ROLEc)::value, NS = decltype(NSc)::value, RD = decltype(RDc)::value;
    constexpr bool MUL = NS > 0;
    constexpr int EPI = decltype(EPIc)::value == 3 ? 0 : decltype(EPIc)::value;
    constexpr bool FRESH = decltype(EPIc)::value == 1 || decltype(EPIc)::value == 3;
    static_assert(!EPI || NS == 8, "the epilogue rides on the multiplies of a full tile");
    constexpr int G1 = NS == 4 ? 8 + RD : 16, D1 = NS == 4 ? 2 : 4, L1 = NS == 4 ? 1 : 2;  // LDS writes: first gap, distance, distance of the reload behind
    constexpr int G2 = 16, D2 = NS == 4 ? 2 : 5;                                             // copies likewise
    EpiLane e = {nullptr, nullptr, {0, 0}};
    i32x4_t vv[2][2];
    if (EPI && !B_KMAJOR) e = epi_lane();
    int lane_off = 0;
    uint2 ex = {0, 0};
    if (EPI && B_KMAJOR) lane_off = epi_lane_t();
    // NT: unit u = 4 (strip - first strip) + r in the gaps in front of multiplies T0 + 3 u and T0 + 3 u + 1: a strip of
    // the tile's last K step is complete three multiplies before its first unit, a strip of the first K step is
    // started afresh after its last unit
    constexpr int EPI_T0 = EPI == 2 ? 11 : 0;
    // EPI 2 (a tile's last K step) converts and stores strips 0-3 of the tile, EPI 1 (the next tile's first) strips
    // 4-7: block bb of the half in the gap in front of multiply G0 + 7 bb / 4, at least four multiplies after the
    // multiply that completed it and before the one that starts it afresh; a piece (four blocks) is read back in the
    // gap of its last block and stored two and four gaps later.
    constexpr int EPI_S0 = EPI == 2 ? 0 : 4, EPI_G0 = EPI == 2 ? 4 : 0;
    for_each<(NS == 4 ? 32 : 64)>([&](auto Nc) __attribute__((always_inline)) {
      constexpr int n = decltype(Nc)::value, i = n / 8, j = (i & 1) ? 7 - n % 8 : n % 8;  // snake order: one operand register changes per multiply
      if constexpr (EPI != 0 && B_KMAJOR) {
        constexpr int u = (n - EPI_T0) / 3;
        if constexpr (n >= EPI_T0 && u < 16) {
          if constexpr ((n - EPI_T0) % 3 == 0) ex = epi_half_t(TGG_W4_I(EPI_S0 + u / 4), TGG_W4_I(u % 4), TGG_W4_I(0));
          if constexpr ((n - EPI_T0) % 3 == 1) {
            const uint2 ey = epi_half_t(TGG_W4_I(EPI_S0 + u / 4), TGG_W4_I(u % 4), TGG_W4_I(1));
            epi_store_t(lane_off, EPI_S0 + u / 4, u % 4, ex, ey, true);
          }
        }
      }
      if constexpr (EPI != 0 && !B_KMAJOR) {
        for_each<32>([&](auto Bc) __attribute__((always_inline)) {
          constexpr int bb = decltype(Bc)::value, g = EPI_G0 + 7 * bb / 4, si = EPI_S0 + bb / 8, sj = (si & 1) ? 7 - bb % 8 : bb % 8;
          if constexpr (g == n) epi_cvt(e, TGG_W4_I(si), TGG_W4_I(sj));
          if constexpr ((bb & 3) == 3 && g == n) epi_read(e, sj >> 2, vv[(bb >> 2) & 1]);
        });
        for_each<32>([&](auto Bc) __attribute__((always_inline)) {
          constexpr int bb = decltype(Bc)::value, g = EPI_G0 + 7 * bb / 4, si = EPI_S0 + bb / 8, sj = (si & 1) ? 7 - bb % 8 : bb % 8;
          if constexpr ((bb & 3) == 3 && g + 2 == n) epi_store(e, si, sj >> 2, 0, vv[(bb >> 2) & 1][0], true);
          if constexpr ((bb & 3) == 3 && g + 4 == n) epi_store(e, si, sj >> 2, 1, vv[(bb >> 2) & 1][1], true);
        });
      }
      if constexpr (MUL) {
        constexpr int fa = 64 + 32 * CUR + 4 * i, fb = 128 + 32 * CUR + 4 * j;
        if constexpr (B_KMAJOR) acc_mfma<DT, FRESH, 32 * i + 4 * j, fa, fb>();
        else acc_mfma<DT, FRESH, 32 * i + 4 * j, fb, fa>();
      }
      if constexpr (n < 8 + RD) read_frag(TGG_W4_I(NKS), Nc, TGG_W4_I(CUR ^ 1), nb_off);
      if constexpr (ROLE == 1) {
        constexpr int w = n - G1, l = n - G1 - L1;
        if constexpr (w >= 0 && w % D1 == 0 && w / D1 < 8) write_s(TGG_W4_I(w / D1), SETc, wr_addr);
        if constexpr (l >= 0 && l % D1 == 0 && l / D1 < 8) load_s(TGG_W4_I(l / D1), SETc, rs_c, koff_s);
        constexpr int part = n - (NS == 4 ? 28 : 56);  // behind the last load
        if constexpr (part >= 0 && part < 4) advance_s(part);
      }
      if constexpr (ROLE == 2) {
        constexpr int m = n - G2, c = n - G2 - 1;
        if constexpr (m >= 0 && m % D2 == 0 && m / D2 < 8) copy_d_m0(TGG_W4_I(m / D2), cp_addr);
        if constexpr (c >= 0 && c % D2 == 0 && c / D2 < 8) copy_d(TGG_W4_I(c / D2), rd_c, koff_d);
        if constexpr (NS == 4) {
          if constexpr (n == 31) for_each<4>([&](auto Pc) __attribute__((always_inline)) { advance_d(decltype(Pc)::value); });
        } else {
          constexpr int part = n - 56;
          if constexpr (part >= 0 && part < 4) advance_d(part);
        }
      }
    });
    if constexpr (ROLE == 2) asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory", TGG_W4_ACC_CLOBBER);
    else if constexpr (ROLE == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(EPI ? 24 : 8) : "memory", TGG_W4_ACC_CLOBBER);
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : : : "memory", TGG_W4_ACC_CLOBBER);
  };

  // ---- prologue: slab 0 lands in buffer 0, slabs 1 and 2 are requested, the first fragments are read -----------------
  Tile cur;
  tile_at(walk.first, cur);
  {
    const Win w0 = window(cur, walk.first < walk.end);
    const bool more = tile_at(walk.first + walk.stride, nxt_tile);
    nxt = window(nxt_tile, more);
    rs_c = w0.rs;
    rd_c = w0.rd;
  }
#define TGG_W4_EACH(f) f(0) f(1) f(2) f(3) f(4) f(5) f(6) f(7)
#define TGG_W4_P0(c) copy_direct(std::integral_constant<int, c>(), No(), rs_c, 0, wave_buf + S_OFF); \
                     copy_direct(std::integral_constant<int, c>(), Yes(), rd_c, 0, wave_buf + D_OFF);
  TGG_W4_EACH(TGG_W4_P0)
#undef TGG_W4_P0
  wait_vmcnt<0>();
  __syncthreads();
#define TGG_W4_P1(c) load_s(std::integral_constant<int, c>(), I1(), rs_c, 128);
  TGG_W4_EACH(TGG_W4_P1)
#undef TGG_W4_P1
#define TGG_W4_P2(c) copy_direct(std::integral_constant<int, c>(), Yes(), rd_c, d_step, wave_buf + C::STAGE_BYTES + D_OFF);
  TGG_W4_EACH(TGG_W4_P2)
#undef TGG_W4_P2
#define TGG_W4_P3(c) load_s(std::integral_constant<int, c>(), I0(), rs_c, 256);
  TGG_W4_EACH(TGG_W4_P3)
#undef TGG_W4_P3
  koff_s = 3 * 128;  // at least four slabs per tile (w4_supported): both cursors are still in the first tile
  koff_d = 2 * d_step;
  if (TAIL) {
    mask_s = koff_s + chunk_off >= row_bytes ? kNoFetch : 0;
    if (B_KMAJOR) mask_d = koff_d + chunk_off >= row_bytes ? kNoFetch : 0;
  }
  set_a_rd(0, cur);
  set_a_rd(1, cur);
  kstep(I1(), I0(), I0(), I8(), I0(), 0u, I0(), 0u, I0(), 0u);  // reads K step 0 of buffer 0 into set 0, multiplies nothing, waits for everything

  for (int tile_id = walk.first; tile_id < walk.end; tile_id += walk.stride) {
    const bool half = cur.rows <= C::BM / 2;  // a tile of at most 128 rows: 64 per wave, half the multiplies
    const int wm0 = wave_m * (half ? 64 : 128);
    const bool active = wm0 < cur.rows && cur.n0 + wn0 < p.N;  // this wave's block of the tile has rows and columns
    const int rows_left = cur.rows - wm0, most = half ? 64 : 128;
    const i32x4_t out_rs = make_rsrc32((uint64_t)p.C + (uint64_t)(((cur.row0 + wm0) * (int64_t)p.N + cur.n0 + wn0) * 2),
                                       active ? (rows_left < most ? rows_left : most) * p.N * 2 : 0);
    const int out_cols = __builtin_amdgcn_readfirstlane(active ? p.N - cur.n0 - wn0 : 0);
    // One slab.  EP: 1 the first of a full tile, whose first K step starts the accumulators afresh and carries strips 4-7 of the tile before,
    // 2 the last of a full tile, whose second K step carries strips 0-3, 3 the first of a half tile; PAR: parity of the slab = its LDS buffer; the A
    // chunks of the next slab wait in register set 1 - PAR.  RD: fragments of A to read for the slab behind.
    auto slab = [&](auto NSc, auto EPc, auto PARc, auto RDc) __attribute__((always_inline)) {
      constexpr int EP = decltype(EPc)::value, PAR = decltype(PARc)::value;
      typedef std::integral_constant<int, EP == 1 || EP == 3 ? EP : 0> Ep0;
      typedef std::integral_constant<int, EP == 2 ? 2 : 0> Ep1;
      typedef std::integral_constant<int, 1 - PAR> SetN;
      constexpr uint32_t cur_off = PAR * C::STAGE_BYTES, nxt_off = C::STAGE_BYTES - cur_off;
      kstep(I0(), I1(), NSc, NSc, I1(), cur_off, Ep0(), s_wr + nxt_off, SetN(), 0u);
      // set 1 is complete, this wave has read all it needs of the current slab, its copies of the next slab have landed
      asm volatile("s_barrier" ::: "memory");
      kstep(I1(), I0(), NSc, RDc, I2(), nxt_off, Ep1(), 0u, I0(), wave_buf + cur_off);
    };
    if (__builtin_expect(half, 0)) {
      epi_flush();
      slab(I4(), I3(), I0(), I4());  // an even number of slabs per tile, at least four: every tile starts in buffer 0
      slab(I4(), I0(), I1(), I4());
      for (int kt = 4; kt < kt_all; kt += 2) {
        slab(I4(), I0(), I0(), I4());
        slab(I4(), I0(), I1(), I4());
      }
      slab(I4(), I0(), I0(), I4());
      set_a_rd(0, nxt_tile);
      slab(I4(), I0(), I1(), I8());
      pend_rs = out_rs;
      pend_cols = out_cols;
      epi_strips(I0());
      pend_rs[2] = 0;
    } else {
      slab(I8(), I1(), I0(), I8());
      slab(I8(), I0(), I1(), I8());
      for (int kt = 4; kt < kt_all; kt += 2) {
        slab(I8(), I0(), I0(), I8());
        slab(I8(), I0(), I1(), I8());
      }
      // what the tile's last K step, the next tile's first K step and a flush store: nothing for a wave whose block of
      // the tile has no rows or no columns
      pend_rs = out_rs;
      pend_cols = out_cols;
      pending = true;
      slab(I8(), I0(), I0(), I8());
      set_a_rd(0, nxt_tile);
      slab(I8(), I2(), I1(), I8());
    }
    set_a_rd(1, nxt_tile);
    // both cursors are in the next tile by now: it becomes the current one, and the one after it is looked up
    cur = nxt_tile;
    const bool more = tile_at(tile_id + 2 * walk.stride, nxt_tile);
    nxt = window(nxt_tile, more);
  }
  epi_flush();
  wait_vmcnt<0>();  // trailing zero-length copies still write LDS
#undef TGG_W4_EACH
#undef TGG_W4_GA
#undef TGG_W4_GA_CLOBBER
}

template <int DT, int LAYOUT, bool TAIL>
int launch_w4(const GemmParams& p, hipStream_t s) {
  static bool attr_set[64] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  const bool listed = dev >= 0 && dev < 64;
  auto kern = gemm_w4_kernel<DT, LAYOUT, TAIL>;
  if (!listed || !attr_set[dev]) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, W4Cfg::SMEM_BYTES) != hipSuccess)
      return check_launch("hipFuncSetAttribute(gemm_w4)");
    if (listed) attr_set[dev] = true;
  }
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(W4Cfg::THREADS), W4Cfg::SMEM_BYTES, s, p);
  return check_launch("gemm_w4");
}

// see TAIL
bool needs_tail(const GemmParams& p, int layout) { return p.K % 128 != 0 || p.K < 256 || (layout == W4_NN && (p.N & 255) != 0); }

}  // namespace

// More than two rounds of 256x256 tiles whatever the group sizes turn out to be: at least ceil(m_total / 256) row tiles.
static bool w4_large(const GemmParams& p) {
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  return ((p.m_total + 255) / 256) * ((p.N + 127) / 128) > 4 * (int64_t)grid;
}

// Whether 256-row tiles pay depends on the group sizes, which only the device knows.  With 512 rows and more per group on
// average they do; a masked launch (counts anywhere up to its row stride), one with smaller groups or one of fewer rounds is
// enqueued together with the eight-wave kernel, and the two decide from the sizes which of them runs.  The average is that of the operand, whose rows the
// groups may own in part only (a buffer of fixed size, a padded layout of small groups).  Filled whole, launches of 200-511 rows a group take 0.95 of the
// eight-wave kernel's time by this kernel alone and 0.97 decided on the device; filled to a tenth and less 1.05-1.14 alone (15 random ones, up to
// 1.21).  Large ones of longer groups 0.93-0.98 alone, however much of them is filled (56 random ones, a fiftieth to the whole).
bool w4_decided_on_device(const GemmParams& p) {
  return p.mode == MODE_MASKED || p.m_total < 512 * (int64_t)p.G || !w4_large(p);
}

// The four-wave kernel takes large M-grouped and masked launches, and M-grouped ones of 128 rows and more per group whose likely tiles
// (every group's last one half full) cost two rounds of K = 2048 or more and would not be chosen for 128-row tiles
// (sched_wide_tiles_chosen).  Of 574 of those, drawn at random with operands in no cache, 554 were its by their sizes as well and
// took 0.91 of the eight-wave kernel's time (0.92 with a tail, 0.85-1.01; before half tiles) with the launch that returns in it; 20 were not and lost 4-6 us, 1.03.
// Large ones with a tail: 0.93.  32 groups of 1635 rows, N = 1536, K = 3208: 549 -> 487 us; 8 of 1700, N = 3296, K = 1256: 136 -> 123.
// Smaller launches stay with the eight-wave kernels, which choose narrower tiles on the device.
bool w4_supported(const GemmParams& p, int dt, int layout, bool any_size) {
  if (dt != DT_BF16 && dt != DT_F16) return false;
  if (layout != W4_NT && layout != W4_NN) return false;
  // NN: a group's B, with the rows that the tail may add, within 2 GiB
  if (layout == W4_NN && ((int64_t)p.K + 128) * p.N * 2 >= (1ll << 31)) return false;
  if (p.mode != MODE_MG && p.mode != MODE_MG_PAD && p.mode != MODE_MASKED) return false;
  // launches whose groups may be small are decided on the device (w4_decided_on_device), by a predicate that needs
  // one thread of this kernel per group; besides, with more groups than threads one of them makes the whole table, 0.12-0.2 us a group, which the eight-wave
  // kernels' 512 threads do together (367 groups of 256 rows, N = 512, K = 768: 106 us there, 171 here)
  if (w4_decided_on_device(p) && p.G > W4Cfg::THREADS) return false;
  if (p.q_fmt != 0 || p.G > kFastMaxGroups) return false;
  if ((p.N & 7) != 0 || p.K < 8 || (p.K & 7) != 0) return false;
  if ((int64_t)p.K * 2 * 256 >= (1ll << 30)) return false;
  if ((int64_t)p.N * 2 * 128 >= (1ll << 30)) return false;  // a wave's block of the output within the epilogue's 32-bit offsets, out-of-range marker included
  if (p.K < 192) return false;  // the first three slabs of a tile are whole
  // masked launches with a tail: the launch that returns costs more than this kernel gains (120 random ones from K = 776 on, counts up to 0.05-0.4 of the
  // slots 1.035 of the eight-wave kernels' time alone, up to 0.7 and all of them 0.995)
  if (p.mode == MODE_MASKED && needs_tail(p, layout)) return false;
  if (any_size) return true;
  // a short K spends more on the slab that makes the tail's number even than the eight-wave kernel loses (4 groups of 13000 rows, N = 3096,
  // K = 512, [K, N]: 195 us there, 202 here; 16 of 1200, N = 3072, K = 536: 79 and 81)
  if (needs_tail(p, layout) && p.K < 768) return false;
  // and so does, up to K = 1024, the launch that returns where only N is cut, whose slabs the eight-wave kernel has whole as well (17 random ones 1.014 of
  // its time alone, up to 1.07; K = 1152-1500 0.995; K no multiple of 128: 0.98)
  if (layout == W4_NN && p.K % 128 == 0 && p.K <= 1024 && needs_tail(p, layout) && w4_decided_on_device(p)) return false;
  if (w4_large(p)) return true;
  if (p.mode == MODE_MASKED || p.m_total < 128 * (int64_t)p.G) return false;
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  const int64_t tiles_n = (p.N + 255) / 256;
  const int64_t full_2 = (2 * ((p.m_total + 255) / 256) + p.G) * tiles_n, half_2 = (2 * ((p.m_total + 127) / 128) + p.G) * tiles_n;  // twice the likely tiles
  const int64_t rounds_full = (full_2 + 2 * grid - 1) / (2 * grid), rounds_half = (half_2 + 2 * grid - 1) / (2 * grid);
  // (Fewer rounds are no safe choice: launches of 256 rows a group and more take 0.91 of the eight-wave kernel's time from 1.15 rounds of likely tiles on
  // and from 0.7 to 0.9 of one where the groups fill the operand, but 1.03 with half of it filled, up to 1.24, and 1.1 with a tenth, up to 1.29: its narrower
  // tiles fit what is left.  Decided on the device they would pay 4 us for 30-100.)
  return full_2 * p.K >= 2 * 4096 * (int64_t)grid && rounds_half * 3 > rounds_full * 4;
}

template <int DT, int LAYOUT>
int launch_w4_layout(const GemmParams& p, hipStream_t s) {
  return needs_tail(p, LAYOUT) ? launch_w4<DT, LAYOUT, true>(p, s) : launch_w4<DT, LAYOUT, false>(p, s);
}

int launch_w4_16bit(const GemmParams& p, int dt, int layout, hipStream_t s) {
  if (layout == W4_NT) return dt == DT_BF16 ? launch_w4_layout<DT_BF16, W4_NT>(p, s) : launch_w4_layout<DT_F16, W4_NT>(p, s);
  return dt == DT_BF16 ? launch_w4_layout<DT_BF16, W4_NN>(p, s) : launch_w4_layout<DT_F16, W4_NN>(p, s);
}

}  // namespace tgg
