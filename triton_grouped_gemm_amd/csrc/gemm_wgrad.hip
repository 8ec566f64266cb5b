// Four-wave bf16/fp16 K-grouped GEMM kernel for gfx950 (weight gradient): C[g] = A[tokens of g, :]^T . B[tokens of g, :],
// A [Ktot, Mdim], B [Ktot, N], C [G, Mdim, N].
//
// One workgroup per CU, four waves, one per SIMD; tile 256x256, every wave owns a 128x128 block of 16x16x32 MFMA tiles with
// its 256 accumulator registers in AGPRs (see gemm_w4.hip for why, and for the rules that the order of the instructions
// follows).  A K step is 32 tokens, and so is a slab: 16 KB of A and 16 KB of B, token rows of 512 bytes, four slab buffers
// in LDS.  Per K step q, per wave:
//   64 multiplies on fragment set q % 2; meanwhile the 16 fragments of slab q + 1 are read into the other set (two
//   transposing 8-byte reads each) and this wave's eight copies of slab q + 4 go straight to LDS, into the buffer of slab q;
//   wait for the fragment reads and for this wave's copies of slab q + 2, workgroup barrier.
// The copies have between two and three K steps to land, where two 64-token buffers leave them one or two: what
// a launch with short segments waits for is memory (it writes 128 KB of output per tile, and loads queue behind stores).
// Token rows are 512 bytes whatever the slab's depth, so that the shallow slabs cost no extra requests here (operands whose
// rows run along K would fetch half lines), and a segment's last slab is padded to 32 tokens and not to 64.
//
// The epilogue rides on multiplies as in gemm_w4.hip: strips 0-3 of a wave's block are converted and stored between the
// multiplies of the tile's last K step, strips 4-7 between those of the next tile's first, whose multiplies start from a
// zero addend.  Against the eight-wave kernel (gemm_fast.hip, TN), 128 groups of 2048 x 1536 with 64 /
// 128 / 256 / 512 / 1024 tokens on average, operands in no cache: 190 / 237 / 325 / 488 / 815 -> 179 / 212 / 287 / 432 / 721 us (5120 tokens:
// 3434 -> 3042, 1.36 PFLOP/s).  What bounds it: from about 512 tokens on the matrix pipe (0.73 us a K step with all CUs multiplying,
// 0.53 on a quarter of them, i.e. power) and 1.5 us a tile for the epilogue's conversions and LDS staging; below, memory (256 tokens: 1.04 GB,
// 204 us at the copy rate): reads that come from HBM wait behind the writes, so the next tile's are requested a tile ahead (below).
// A tile has an even number of K steps, four at least (of nothing where the segment ends sooner: the
// copy stream is four slabs ahead of the multiplies, so it is in the tile being multiplied or in the next one, and every
// tile starts on the same parity).
//
// Tiles come from KgDraw (w4_common.hpp); the request for the tile after the next goes out four K steps before a tile's end, and its
// answer, in order with the copies, has arrived by the wait that ends the tile.
#include "launch.hpp"
#include "kg_split.hpp"

namespace tgg {

namespace {

struct WgradCfg {
  static constexpr int BM = 256, BN = 256, THREADS = 256, KS = 32;
  static constexpr int OP_BYTES = KS * 512, SLAB_BYTES = 2 * OP_BYTES, SLABS = 4;
  static constexpr int EPI_PITCH = 4 * 32 + 16;         // epilogue staging; a piece: 16 rows x 64 outputs, row pitch in bytes
  static constexpr int EPI_PIECE = 16 * EPI_PITCH;
  static constexpr int EPI_WAVE_BYTES = 2 * EPI_PIECE;  // two pieces alternate
  static constexpr int SCHED_OFF = SLABS * SLAB_BYTES;
  static constexpr int NEXT_OFF = SCHED_OFF + (((int)sizeof(SchedTableT<kFastMaxGroups>) + 255) & ~255);  // drawn tile ids, two words
  static constexpr int EPI_OFF = NEXT_OFF + 256;
  static constexpr int SINK_OFF = EPI_OFF + 4 * EPI_WAVE_BYTES;  // where touched lines' words go, 256 bytes a wave
  static constexpr int META_OFF = SINK_OFF + 4 * 256;  // launches cut along K: what the table's entries are
  static constexpr int SMEM_BYTES = META_OFF + kFastMaxGroups * 4;
  static constexpr int TOUCH = 256;  // tokens of the next tile that are touched
  static_assert(SMEM_BYTES <= 160 * 1024, "LDS budget");
  static_assert(TOUCH >= KS && TOUCH >= BM / 2, "wgrad_supported bounds the slab's and the stores' windows by the touched rows'");
};

typedef SplitCost<64, 3, 20, 8> WgradSplitCost;

// NT: see store_b128.  128 groups of 2048 x N, operands in no cache, 32 / 128 / 256 / 1024 tokens a group: N = 1544 non-temporal 463 / 456 /
// 444 / 888 us, else 202 / 236 / 314 / 823 (the eight-wave kernel, non-temporal: 435 / 392 / 400 / 967); N = 1552 379 / 374 / 357 / 855 and 199 / 231 /
// 310 / 814; N = 1568, whole 64 bytes, 184 / 194 / 306 / 800 and 188 / 227 / 310 / 811; N = 1536 146 / 167 / 252 / 688 and 165 / 191 / 272 / 703.
// SPLIT: segments may be cut along K (kg_split.hpp).  An instantiation of its own: tiles of parts leave as fp32 behind their last K step
// (they are long), and the plain one needs no look at what a tile is.
template <int DT, bool NT, bool SPLIT>
__global__ __launch_bounds__(WgradCfg::THREADS) void gemm_wgrad_kernel(const GemmParams p) {
  typedef WgradCfg C;
  typedef Operand<256, false> Op;  // a slab of either operand: token rows of 512 bytes (here 32 of them)

  extern __shared__ __attribute__((aligned(1024))) char smem[];
  auto& sched = *reinterpret_cast<SchedTableT<kFastMaxGroups>*>(smem + C::SCHED_OFF);
  sched_init<C::BM>(p, sched);
  int32_t* const meta = SPLIT ? reinterpret_cast<int32_t*>(smem + C::META_OFF) : nullptr;
  int groups = p.G;
  if constexpr (SPLIT) groups = __builtin_amdgcn_readfirstlane(split_plan<WgradSplitCost>(p, sched, meta, (int)((p.m_total + 255) / 256) * ((p.N + 255) / 256)));

  const uint32_t smem_addr = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm0 = (wave >> 1) * 128, wn0 = (wave & 1) * 128;
  const int l16 = lane & 15, lg = lane >> 4;
  const int a_ld = (int)p.m_total * 2, b_ld = p.N * 2;  // token row pitches in bytes

  // Copy k (0..3) of an operand's slab by this wave is copy instruction wave + 4 k of the slab: token rows 2 (wave + 4 k), + 1.
  int vo_a[4], vo_b[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    vo_a[k] = Op::lane_voff(lane, (wave + 4 * k) % Op::NPAT, a_ld) + (wave + 4 * k) * Op::RPI * a_ld;
    vo_b[k] = Op::lane_voff(lane, (wave + 4 * k) % Op::NPAT, b_ld) + (wave + 4 * k) * Op::RPI * b_ld;
  }
  // LDS addresses of the fragment reads (gemm_fast.hip has the layout).  A slab buffer's number is (pair, parity): the parity
  // goes into the instruction's offset, the pair is toggled in the address once in two K steps.
  uint32_t a_rd[8], b_rd[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int e = l16 >> 2, c = l16 & 3, sw = (e * 4) ^ ((lg & 1) * 2), row = (lg * 8 + e) * 512 + (c & 1) * 8;
    a_rd[i] = smem_addr + row + ((((wm0 + 16 * i) / 8 + (c >> 1)) ^ sw) << 4);
    b_rd[i] = smem_addr + C::OP_BYTES + row + ((((wn0 + 16 * i) / 8 + (c >> 1)) ^ sw) << 4);
  }

  const KgTiles<SchedTableT<kFastMaxGroups>> tiles(p, sched, groups, meta);
  KgDraw draw(p, reinterpret_cast<int32_t*>(smem + C::NEXT_OFF), tiles.total, wave, lane);
  auto steps_of = [&](const KgTile& t) __attribute__((always_inline)) {
    const int steps = (t.klen + 2 * C::KS - 1) / (2 * C::KS) * 2;
    return steps < C::SLABS ? C::SLABS : steps;
  };

  // ---- the copy stream ---------------------------------------------------------------------------------------------
  // The slabs of all of this workgroup's tiles form one sequence; the cursor is four slabs ahead of the multiplies.  Tokens
  // beyond the segment read as zero through the descriptor's length.
  struct Feed {
    uint64_t a_base, b_base;  // the next slab
    int rem;                  // tokens of the segment from there on
    int a_off, b_off;         // the tile's columns within a token row, bytes
    int left;                 // slabs of the tile still to be requested
  };
  auto feed_of = [&](const KgTile& t) __attribute__((always_inline)) {
    Feed f;
    f.rem = t.klen;
    f.left = t.g < 0 ? 0x7fffffff : steps_of(t);
    f.a_off = t.m0 * 2;
    f.b_off = t.n0 * 2;
    f.a_base = (uint64_t)p.A + (uint64_t)(t.k0 * a_ld + f.a_off);
    f.b_base = (uint64_t)p.B + (uint64_t)(t.k0 * b_ld + f.b_off);
    return f;
  };
  Feed feed, nxt;
  i32x4_t ra, rb;
  auto rsrc = [&](uint64_t base, int bytes) __attribute__((always_inline)) {  // make_rsrc32 of values that are in scalar registers
    return i32x4_t{(int)(uint32_t)base, (int)(uint32_t)(base >> 32) & 0xffff, bytes < 0 ? 0 : bytes, 0x00020000};
  };
  auto step_feed = [&]() __attribute__((always_inline)) {  // descriptors of the next slab; the cursor moves behind it
    const bool wrap = feed.left == 0;
    feed.a_base = wrap ? nxt.a_base : feed.a_base;
    feed.b_base = wrap ? nxt.b_base : feed.b_base;
    feed.rem = wrap ? nxt.rem : feed.rem;
    feed.a_off = wrap ? nxt.a_off : feed.a_off;
    feed.b_off = wrap ? nxt.b_off : feed.b_off;
    feed.left = (wrap ? nxt.left : feed.left) - 1;
    int rows = feed.rem < 0 ? 0 : feed.rem;
    asm("" : "+s"(rows));  // two scalar instructions and not a vector one whose result would have to be read back
    rows = rows > C::KS ? C::KS : rows;
    ra = rsrc(feed.a_base, rows * a_ld - feed.a_off);
    rb = rsrc(feed.b_base, rows * b_ld - feed.b_off);
    feed.rem -= C::KS;
    feed.a_base += (uint64_t)(C::KS * a_ld);
    feed.b_base += (uint64_t)(C::KS * b_ld);
  };
  const uint32_t wave_buf = smem_addr + wave * 1024;  // copy `wave` of buffer 0's A slab
  auto copy_m0 = [&](auto Kc, uint32_t buf) __attribute__((always_inline)) {
    constexpr int k = decltype(Kc)::value;
    asm volatile("s_add_u32 m0, %0, %1" : : "s"(buf), "n"((k >> 2) * C::OP_BYTES + (k & 3) * 4096) : "memory", "m0", "scc");
  };
  auto copy = [&](auto Kc) __attribute__((always_inline)) {
    constexpr int k = decltype(Kc)::value;
    const int v = k < 4 ? vo_a[k & 3] : vo_b[k & 3];
    const i32x4_t r = k < 4 ? ra : rb;
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(v), "s"(r) : "memory");
  };

  // While a tile is multiplied and the one before it is stored, the next tile's lines are brought into L2: one word of each of its
  // first 256 tokens' lines (four per token row and operand) goes into a sink in LDS.  The workgroups of an XCD that run
  // together share their panels (the tiles of a run of 32 neighbours: nc columns by 32 / nc rows), and each touches its part of
  // them only.  128 groups of 2048 x 1536, 64 / 128 / 256 / 512 tokens, operands in no cache: 201 / 243 / 312 / 450 -> 179 / 212 / 287 / 432 us.
  // Touched during the tile's own K steps (a few slabs ahead of the copies) the lines come hardly sooner than the copies (313 us with 256 tokens) and
  // long segments lose 2 %; the next tile's touched two K steps later: 200 / 226 / 292 / 441.
  const int sharers_b = tiles.nc < 32 ? 32 / tiles.nc : 1;
  const int lines_a = (4 * C::TOUCH + tiles.nc - 1) / tiles.nc, lines_b = (4 * C::TOUCH + sharers_b - 1) / sharers_b;
  auto touch = [&](uint64_t base, int off, int klen, int ld, int part, int lines) __attribute__((always_inline)) {
    const i32x4_t r = make_rsrc32(base, (klen < C::TOUCH ? klen : C::TOUCH) * ld - off);
    const uint32_t at = smem_addr + C::SINK_OFF + wave * 256;
    for (int n0 = wave * 64; n0 < lines; n0 += C::THREADS) {
      const int n = n0 + lane, line = part * lines + n;
      const int v = n < lines ? (line >> 2) * ld + (line & 3) * 128 : kNoFetch;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dword %1, %2, 0 offen lds" : : "s"(at), "v"(v), "s"(r) : "memory", "m0");
    }
  };
  auto touch_tile = [&](const KgTile& t, const Feed& f) __attribute__((always_inline)) {
    const int mt = t.m0 >> 8, nt = t.n0 >> 8;
    touch(f.a_base, f.a_off, t.klen, a_ld, nt - (int)tiles.by_nc.div((uint32_t)nt) * tiles.nc, lines_a);
    touch(f.b_base, f.b_off, t.klen, b_ld, mt % sharers_b, lines_b);
  };
  // ---- fragments and accumulators ------------------------------------------------------------------------------------
  i32x4_t fa[2][8], fb[2][8];
  f32x4_t acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto toggle = [&](uint32_t& at) __attribute__((always_inline)) { asm volatile("v_xor_b32 %0, 0x10000, %0" : "+v"(at)); };
  // read number q (0..15) of a slab's fragments: B's first, the next K step needs all of them at once; PAR: the slab's parity
  auto read_frag = [&](auto PARc, auto Qc, i32x4_t (&sa)[8], i32x4_t (&sb)[8]) __attribute__((always_inline)) {
    constexpr int Q = decltype(Qc)::value, off = decltype(PARc)::value * C::SLAB_BYTES;
    if (Q < 8) lds_read_tr<off, off + 4 * 512>(sb[Q & 7], b_rd[Q & 7]);
    else lds_read_tr<off, off + 4 * 512>(sa[Q & 7], a_rd[Q & 7]);
  };

  // ---- epilogue (see gemm_w4.hip, B as [G, K, N]): a lane owns row l16 and columns 16 j + 4 lg + (0..3) of block (i, j); a strip
  // goes through the wave's LDS staging as two pieces of 64 columns and leaves as 16-byte stores of 128-byte row segments
  i32x4_t pend_rs = make_rsrc32(0, 0);
  int pend_cols = 0;
  char* const stage = smem + C::EPI_OFF + wave * C::EPI_WAVE_BYTES;
  struct EpiLane { char* wr; const char* rd; int off[2]; };
  auto epi_lane = [&]() __attribute__((always_inline)) {
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
  auto epi_cvt = [&](const EpiLane& e, int i, int j) __attribute__((always_inline)) {
    asm volatile("" : "+a"(acc[i][j]));
    *(uint2*)(e.wr + (j >> 2) * C::EPI_PIECE + (j & 3) * 32) = pack4<DT>(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
    asm volatile("" ::: "memory");
  };
  auto epi_read = [&](const EpiLane& e, int h, i32x4_t (&v)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < 2; ++it) v[it] = *(const i32x4_t*)(e.rd + h * C::EPI_PIECE + it * 8 * C::EPI_PITCH);
    asm volatile("" ::: "memory");
  };
  auto epi_store = [&](const EpiLane& e, int i, int h, int it, const i32x4_t& v, bool between_multiplies) __attribute__((always_inline)) {
    const int off = e.off[h] + (16 * i + 8 * it) * p.N * 2;
    if (between_multiplies) store_b128<NT, 0>(v, off, pend_rs);  // the multiply that follows is the second wait state
    else store_b128<NT, 1>(v, off, pend_rs);
  };
  auto epi_flush = [&]() __attribute__((always_inline)) {  // strips 4-7 of the workgroup's last tile
    asm volatile("s_nop 15\n\ts_nop 7" : "+a"(acc[7][0]), "+a"(acc[7][1]), "+a"(acc[7][2]), "+a"(acc[7][3]),
                 "+a"(acc[7][4]), "+a"(acc[7][5]), "+a"(acc[7][6]), "+a"(acc[7][7]));
    const EpiLane e = epi_lane();
#pragma unroll
    for (int i = 4; i < 8; ++i) {
#pragma unroll
      for (int j = 0; j < 8; ++j) epi_cvt(e, i, j);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        i32x4_t v[2];
        epi_read(e, h, v);
        epi_store(e, i, h, 0, v[0], false);
        epi_store(e, i, h, 1, v[1], false);
      }
    }
  };

  // ---- prologue ------------------------------------------------------------------------------------------------------
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<int, 16> W16;
  typedef std::integral_constant<int, 32> W32;
  typedef std::integral_constant<int, 48> W48;
  __syncthreads();
  draw.request();
  wait_vmcnt<0>();
  draw.take(0);
  __syncthreads();
  KgTile cur = tiles.look_up(draw.tile_at(0)), following = cur;
  feed = feed_of(cur);
  nxt = feed;
  draw.request();
#define TGG_WG_EACH8(f) f(0) f(1) f(2) f(3) f(4) f(5) f(6) f(7)
  for (int s = 0; s < C::SLABS; ++s) {
    step_feed();
    const uint32_t buf = wave_buf + s * C::SLAB_BYTES;
#define TGG_WG_P(c) copy_m0(std::integral_constant<int, c>(), buf); asm volatile("s_nop 0" ::: "memory"); copy(std::integral_constant<int, c>());
    TGG_WG_EACH8(TGG_WG_P)
#undef TGG_WG_P
  }
  wait_vmcnt<0>();
  draw.take(1);
  __syncthreads();
#define TGG_WG_RD(q) read_frag(I0(), std::integral_constant<int, q>(), fa[0], fb[0]);
  TGG_WG_EACH8(TGG_WG_RD)
  TGG_WG_RD(8) TGG_WG_RD(9) TGG_WG_RD(10) TGG_WG_RD(11) TGG_WG_RD(12) TGG_WG_RD(13) TGG_WG_RD(14) TGG_WG_RD(15)
#undef TGG_WG_RD
#undef TGG_WG_EACH8
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : TGG_TIE8(fa[0]), TGG_TIE8(fb[0]) : : "memory");  // slab 0 is in registers: its buffer is free

  uint32_t cp_off = 0;  // the slab buffer that the K step copies into
  // One K step on fragment set CUR (the parity of the slab).  EPI 0: a tile's inner one, 1: its first, 2: its last, without the
  // barrier.  WAIT: the memory operations that may be in flight at its end, see below.
  auto kstep = [&](auto CURc, auto EPIc, auto WAITc) __attribute__((always_inline)) {
    constexpr int CUR = decltype(CURc)::value, EPI = decltype(EPIc)::value, WAIT = decltype(WAITc)::value;
    typedef std::integral_constant<int, CUR ^ 1> NextPar;
    EpiLane e = {nullptr, nullptr, {0, 0}};
    i32x4_t vv[2][2];
    if (EPI) e = epi_lane();
    const uint32_t buf = wave_buf + cp_off;
    constexpr int EPI_S0 = EPI == 2 ? 0 : 4, EPI_G0 = EPI == 2 ? 4 : 0;
    for_each<64>([&](auto Nc) __attribute__((always_inline)) {
      constexpr int n = decltype(Nc)::value, i = n / 8, j = (i & 1) ? 7 - n % 8 : n % 8;  // snake order: one operand register changes per multiply
      if constexpr (EPI != 0) {  // block bb of the half in the gap in front of multiply G0 + 7 bb / 4, as in gemm_w4.hip
#pragma unroll
        for (int bb = 0; bb < 32; ++bb) {
          const int g = EPI_G0 + 7 * bb / 4, si = EPI_S0 + bb / 8, sj = (si & 1) ? 7 - bb % 8 : bb % 8;
          if (g == n) epi_cvt(e, si, sj);
          if ((bb & 3) == 3 && g == n) epi_read(e, sj >> 2, vv[(bb >> 2) & 1]);
        }
#pragma unroll
        for (int bb = 3; bb < 32; bb += 4) {
          const int g = EPI_G0 + 7 * bb / 4, si = EPI_S0 + bb / 8, sj = (si & 1) ? 7 - bb % 8 : bb % 8;
          if (g + 2 == n) epi_store(e, si, sj >> 2, 0, vv[(bb >> 2) & 1][0], true);
          if (g + 4 == n) epi_store(e, si, sj >> 2, 1, vv[(bb >> 2) & 1][1], true);
        }
      }
      if constexpr (EPI == 1) mfma_new<DT>(acc[i][j], fb[CUR][j], fa[CUR][i]);
      else mfma_acc<DT>(acc[i][j], fb[CUR][j], fa[CUR][i]);
      if constexpr (n < 16) read_frag(NextPar(), Nc, fa[CUR ^ 1], fb[CUR ^ 1]);
      if constexpr (n == 4) step_feed();
      constexpr int c0 = n - 17;  // copies: m0 in one gap, the copy in the next, one every four multiplies
      if constexpr (c0 >= 0 && c0 < 32 && c0 % 4 == 0) copy_m0(std::integral_constant<int, c0 / 4>(), buf);
      if constexpr (c0 >= 0 && c0 < 32 && c0 % 4 == 1) copy(std::integral_constant<int, c0 / 4>());
      if constexpr (CUR == 0 && c0 >= 0 && c0 < 32 && c0 % 4 == 2) toggle(a_rd[c0 / 4]);
      if constexpr (CUR == 0 && c0 >= 0 && c0 < 32 && c0 % 4 == 3) toggle(b_rd[c0 / 4]);
    });
    cp_off = (cp_off + C::SLAB_BYTES) & (C::SLABS * C::SLAB_BYTES - 1);
    // This wave's copies of slab q + 2, requested two K steps ago, have landed: younger are the sixteen copies of this K step and
    // the one before, and their stores (sixteen in a tile's last K step and in the next tile's first; loads and stores complete in order).
    asm volatile("s_waitcnt vmcnt(%16) lgkmcnt(0)" : TGG_TIE8(fa[CUR ^ 1]), TGG_TIE8(fb[CUR ^ 1]) : "n"(WAIT) : "memory", "v255");
    if constexpr (EPI != 2) asm volatile("s_barrier" ::: "memory");
  };

  for (int pos = 0; cur.g >= 0; ++pos) {
    following = tiles.look_up(draw.tile_at(pos + 1));
    nxt = feed_of(following);
    touch_tile(following, nxt);
    const int steps = steps_of(cur);
    if (steps == 4) draw.request();
    kstep(I0(), I1(), W48());  // behind the last K step of the tile before; the launch's first three K steps find their slabs landed
    kstep(I1(), I0(), W32());
    for (int k = 4; k < steps; k += 2) {
      if (k + 2 >= steps) draw.request();  // four K steps before the answer is taken, no sooner: who draws late draws fairly
      kstep(I0(), I0(), W16());
      kstep(I1(), I0(), W16());
    }
    // what the tile's last K step, the next tile's first and a flush store
    const int64_t rows_left = p.m_total - cur.m0 - wm0;
    pend_rs = make_rsrc32((uint64_t)p.C + (uint64_t)((((int64_t)cur.g * p.m_total + cur.m0 + wm0) * (int64_t)p.N + cur.n0 + wn0) * 2),
                          rows_left > 0 && (!SPLIT || cur.slot < 0) ? (int)(rows_left < 128 ? rows_left : 128) * p.N * 2 : 0);
    pend_cols = p.N - cur.n0 - wn0;
    kstep(I0(), I0(), W16());
    kstep(I1(), I2(), W32());
    if constexpr (SPLIT) {
      if (cur.slot >= 0) store_part(acc, p.split_ws, (int64_t)cur.slot * tiles.per_group + (cur.m0 >> 8) * ((p.N + 255) >> 8) + (cur.n0 >> 8), wave, lane);
    }
    draw.take(pos + 2);
    asm volatile("s_barrier" ::: "memory");
    cur = following;
  }
  epi_flush();
  draw.finish();
  wait_vmcnt<0>();  // trailing zero-length copies still write LDS
}

template <int DT, bool NT, bool SPLIT>
int launch_wgrad(const GemmParams& p, hipStream_t s) {
  static bool attr_set[64] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  const bool listed = dev >= 0 && dev < 64;
  auto kern = gemm_wgrad_kernel<DT, NT, SPLIT>;
  if (!listed || !attr_set[dev]) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, WgradCfg::SMEM_BYTES) != hipSuccess)
      return check_launch("hipFuncSetAttribute(gemm_wgrad)");
    if (listed) attr_set[dev] = true;
  }
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(WgradCfg::THREADS), WgradCfg::SMEM_BYTES, s, p);
  return check_launch("gemm_wgrad");
}

}  // namespace

// K-grouped launches of one and a half rounds of 256x256 tiles and more.  Smaller ones stay with the eight-wave kernel, which has
// narrower tiles and draws a tile later, i.e. more evenly: half a round, 384 / 1024 tokens a group (512 x 1024, 16 groups) 25 / 55 us there
// and 33 / 73 here; one and a half rounds (768 x 2048, 16 groups) 45 / 92 and 36 / 85.  More groups
// than this kernel has threads stay there too: their table takes longer to make (300 groups of 264 x 520, 256 tokens: 98 against 113 us).
// So do short segments where few workgroups run or no queue evens them out: a tile has four K steps at least here, one slab there, which is
// hidden while memory is the bound.  Time of this kernel over the eight-wave kernel's, 1600 random launches of 2-400 tokens a group: a queue and 64 CUs
// 1.05 below 64 tokens (100 and 128 CUs 1.0, all 0.8); no queue and 64-128 CUs 1.07-1.2 below 96 tokens, more of them 1.04 below 32 where N is a multiple
// of 32 (0.7 elsewhere).  128 groups of 1536 x 2816, 15 tokens, 64 CUs, no queue: 652 -> 491 us.
bool wgrad_supported(const GemmParams& p, int dt, bool any_size) {
  if (dt != DT_BF16 && dt != DT_F16) return false;
  if (p.mode != MODE_KG && p.mode != MODE_KG_COUNT) return false;
  if (p.G > WgradCfg::THREADS || (p.N & 7) != 0 || (p.m_total & 7) != 0) return false;
  // the token rows of either operand that are touched (a slab has fewer), and a wave's block of the output, within 32-bit offsets that stay
  // below the out-of-range marker
  if (p.m_total * 2 * WgradCfg::TOUCH >= (1ll << 30) || (int64_t)p.N * 2 * WgradCfg::TOUCH >= (1ll << 30)) return false;
  const int64_t tiles_m = (p.m_total + 255) / 256, tiles_n = (p.N + 255) / 256;
  if (p.G * tiles_m * tiles_n >= (1ll << 31)) return false;
  if (any_size) return true;
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  const int64_t tokens = p.k_total / p.G;
  if (p.queue ? 4 * grid <= num_cus() && tokens < 64 : 2 * grid <= num_cus() ? tokens < 96 : tokens < 32 && rows_of_whole_64_bytes(p)) return false;
  return 2 * p.G * tiles_m * tiles_n >= 3 * (int64_t)grid;
}

int64_t wgrad_split_bytes(const GemmParams& p, int dt) { return wgrad_supported(p, dt, true) ? split_bytes(p, 2000, 6400) : 0; }

int kg_split_slots(const GemmParams& p) { return split_room(p).slots; }

int launch_wgrad_16bit(const GemmParams& p, int dt, hipStream_t s) {
  if (p.split_ws) {
    const bool whole = rows_of_whole_64_bytes(p);
    if (int e = dt == DT_BF16 ? (whole ? launch_wgrad<DT_BF16, true, true>(p, s) : launch_wgrad<DT_BF16, false, true>(p, s))
                              : (whole ? launch_wgrad<DT_F16, true, true>(p, s) : launch_wgrad<DT_F16, false, true>(p, s))) return e;
    return dt == DT_BF16 ? launch_split_sum<DT_BF16, false>(p, s) : launch_split_sum<DT_F16, false>(p, s);
  }
  if (rows_of_whole_64_bytes(p)) return dt == DT_BF16 ? launch_wgrad<DT_BF16, true, false>(p, s) : launch_wgrad<DT_F16, true, false>(p, s);
  return dt == DT_BF16 ? launch_wgrad<DT_BF16, false, false>(p, s) : launch_wgrad<DT_F16, false, false>(p, s);
}

}  // namespace tgg
