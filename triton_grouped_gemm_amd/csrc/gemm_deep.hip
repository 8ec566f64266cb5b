// Bf16/fp16 grouped GEMM kernel for gfx950 launches of few tiles: small tiles, and a deep ring of K slabs.
//
// What bounds a launch whose tiles do not fill the chip is how fast the workgroups it has can draw their operands.  A compute unit keeps
// no more than about 36 KB of cache misses in flight, whatever its waves request: 57-62 GB/s from memory and 105-115 GB/s from the
// memory-side cache (measured with workgroups that only copy; from L2 it is 64 bytes a clock).  A 128x128 tile with K = 2048 is a
// megabyte of operands and takes one workgroup 18 us or more, however deep its pipeline.  So the tile is chosen on the device from the
// sizes, for the fewest bytes that one workgroup has to draw: rounds of the persistent workgroups times the bytes of a slab, for tiles of 64x64
// (16 KB a slab), 64x128 (24) and 128x128 (32).  The ring (eight, five and four slabs) keeps the copies that far ahead of the multiplies,
// also across tiles: the slabs of all of a workgroup's tiles form one stream.
//
// One workgroup per CU, four waves (2x2).  Per slab r (buffer r % ST):
//   K step 0   multiply on fragment set 0 while the fragments of K step 1 are read into set 1 and the second half of the copies of
//              slab r + ST - 1 goes out, into the buffer of slab r - 1
//   wait for this wave's copies of slab r + 1 and its fragment reads, workgroup barrier
//   K step 1   multiply on set 1 while the fragments of slab r + 1 / K step 0 are read into set 0 and the first half of the copies of
//              slab r + ST goes out, into the buffer of slab r (nobody reads it any more)
//
// 150 random launches of up to 8192 rows that take this kernel: 0.61 of the eight-wave kernel's time (0.39-0.89), the same bits.  4 groups of
// 320 rows, N = 512, K = 256 (64 tiles of 64x64): 10.0 -> 7.1 us, of which 4.5 are the host's; 4 of 768, N = 856, K = 2048 (168): 34 -> 17; 8 of
// 1086, N = 2048, K = 4072 (208 of 128x128): 96 -> 55; 16 of 1280, N = 1024, K = 512 (160 of 64x128): 14.3 -> 10.3.  In launches of several
// rounds a small tile's operands cost more than its fit gains (128 groups, 32768 rows, N = 1536, K = 2048: 256 us by the larger tiles, 381 here).
// FP8 with per-channel scales, 100 random launches of up to 8192 rows: 0.62 of the eight-wave kernel's time (0.42-0.87), the same bits.  4 groups of 270
// rows, N = 2048, K = 4096: 35 -> 16 us; 16 of 3393, N = 768, K = 768: 16.1 -> 12.7.
#include "launch.hpp"
#include "w4_common.hpp"

namespace tgg {

namespace {

enum : int { DEEP_NT = 0, DEEP_NN = 1, DEEP_FP8 = 2 };  // FP8: NT, K-contiguous codes, per-row and per-(group, column) scales
constexpr int BKD = 64;

template <int BM_, int BN_, int ST_>
struct DeepCfg {
  static constexpr int BM = BM_, BN = BN_, ST = ST_, NWAVES = 4, THREADS = 256;
  static constexpr int A_BYTES = BM * BKD * 2, B_BYTES = BN * BKD * 2, STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int CA = A_BYTES / 1024 / NWAVES, CB = B_BYTES / 1024 / NWAVES, NC = CA + CB;  // copies per wave and slab
  static constexpr int TM = BM / 32, TN = BN / 32;  // 16x16 blocks per wave: 2x2 waves
  static constexpr int EPI_PITCH = TN * 32 + 16;    // staged strip (B as [G, K, N]): 16 rows x 16 TN outputs
  static constexpr int EPI_WAVE_BYTES = 16 * EPI_PITCH;
  static constexpr int STORES_NT = TM * 4, STORES_NN = TM * TN / 2;  // store instructions per wave and tile
  static_assert(TN == 2 || TN == 4, "a lane's blocks of a row are one store (NT)");
  static_assert(NC % 2 == 0 && TM * TN >= NC / 2, "half a slab's copies go out during a K step");
  static_assert((ST - 2) * NC + STORES_NT < 64, "vmcnt range");
};

constexpr int kDeepSchedOff = 128 * 1024;  // the group table and, behind it, the epilogue's staging
constexpr int kDeepEpiOff = kDeepSchedOff + (((int)sizeof(SchedTableT<kFastMaxGroups>) + 255) & ~255);
constexpr int kDeepSmemBytes = kDeepEpiOff + 4 * DeepCfg<128, 128, 4>::EPI_WAVE_BYTES;
static_assert(kDeepSmemBytes <= 160 * 1024, "LDS budget");

// Copy of 16 bytes a lane, global -> LDS, of the slab at scalar offset koff (see copy_b128_to_lds)
TGG_DEV void copy_slab_b128(const i32x4_t& rsrc, uint32_t lds_addr, int voff, int koff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" : : "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(koff) : "memory", "m0");
}

// The whole kernel but for the group table, which the caller has built for tiles of C::BM rows.  DT: the outputs' type, and unless FP8 the operands';
// FA / FB: FP8, 0 = e4m3fn, 1 = e5m2 (format codes of the f8f6f4 multiply).
// FP8: a slab is 128 bytes of every row as well, but its multiplies take all 128 values at once (32 per lane: 16-byte chunks lg and lg + 4 of a row,
// see gemm_fp8.hip).  The two steps of a slab are the two halves of the wave's row blocks; the second one goes column block by
// column block, and the next slab's fragment takes the place of the one that has been used.
template <class C, int DT, int LAYOUT, int FA, int FB>
TGG_DEV void gemm_deep_body(const GemmParams& p) {
  constexpr bool FP8 = LAYOUT == DEEP_FP8;
  constexpr bool B_KMAJOR = LAYOUT != DEEP_NN;
  constexpr int ES = FP8 ? 1 : 2, KS = BKD * 2 / ES;  // bytes of an operand's value, values of a slab row
  typedef Operand<C::BM, true> OpA;
  typedef Operand<C::BN, B_KMAJOR> OpB;
  static_assert(C::NWAVES % OpA::NPAT == 0 && C::NWAVES % OpB::NPAT == 0, "a wave's copies share one swizzle pattern");
  static_assert(C::ST * C::STAGE_BYTES <= kDeepSchedOff, "LDS layout");

  extern __shared__ __attribute__((aligned(1024))) char smem[];
  auto& sched = *reinterpret_cast<SchedTableT<kFastMaxGroups>*>(smem + kDeepSchedOff);
  const int num_tiles = (int)sched_num_tiles<C::BM, C::BN>(p, sched);

  const uint32_t smem_addr = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm0 = (wave >> 1) * (C::BM / 2), wn0 = (wave & 1) * (C::BN / 2);
  const int l16 = lane & 15, lg = lane >> 4;

  const int ld = p.K * ES, ld_b = (B_KMAJOR ? p.K : p.N) * ES;
  const int kt_n = (p.K + KS - 1) / KS;
  // Source offsets of this wave's copies within the tile's window.  NT: B's rows land permuted, LDS row 16 TN h + 16 j + c of the slab
  // holds column 16 TN h + TN c + j of the tile, so that a lane's results of the TN column blocks are neighbouring outputs of a row.
  int vo_a[C::CA], vo_b[C::CB];
#pragma unroll
  for (int k = 0; k < C::CA; ++k) vo_a[k] = OpA::lane_voff(lane, wave % OpA::NPAT, ld) + (wave + 4 * k) * OpA::RPI * ld;
#pragma unroll
  for (int k = 0; k < C::CB; ++k) {
    if (B_KMAJOR) {
      const int r_local = lane / OpB::CPR, row = (wave + 4 * k) * OpB::RPI + r_local;
      const int col = (row & ~(16 * C::TN - 1)) + C::TN * (row & 15) + ((row >> 4) & (C::TN - 1));
      vo_b[k] = OpB::lane_voff(lane, wave % OpB::NPAT, ld) + (col - r_local) * ld;
    } else {
      vo_b[k] = OpB::lane_voff(lane, wave % OpB::NPAT, ld_b) + (wave + 4 * k) * OpB::RPI * ld_b;
    }
  }
  // K tail: lanes whose chunk of a K-contiguous row starts at or beyond K fetch nothing in a tile's last slab
  const int tail_chunks = (p.K % KS) * ES / 16;
  const int tail = tail_chunks != 0 && OpA::lane_chunk(lane, wave % OpA::NPAT) >= tail_chunks ? kNoFetch : 0;

  // LDS offsets of the fragment reads, relative to a slab buffer
  int a_rd[2], b_rd[B_KMAJOR ? 2 : C::TN];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) a_rd[ks] = (wm0 + l16) * 128 + (((4 * ks + lg) ^ ((l16 / 2) % 8)) << 4);
  if (B_KMAJOR) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) b_rd[ks] = C::A_BYTES + (wn0 + l16) * 128 + (((4 * ks + lg) ^ ((l16 / 2) % 8)) << 4);
  } else {
#pragma unroll
    for (int j = 0; j < C::TN; ++j) {  // token row 8 lg + e (its swizzle is that of every other the lane reads: 32 ks and 4 rows on)
      const int e = l16 >> 2, c = l16 & 3;
      const int chunk = ((wn0 + 16 * j) / 8 + (c >> 1)) ^ OpB::token_swizzle(lg * 8 + e);
      b_rd[B_KMAJOR ? 0 : j] = C::A_BYTES + (lg * 8 + e) * (C::BN * 2) + chunk * 16 + (c & 1) * 8;
    }
  }
  auto load_a = [&](const char* s, int ks, int i) __attribute__((always_inline)) -> i32x4_t { return *(const i32x4_t*)(s + a_rd[ks] + i * 16 * 128); };
  auto load_b = [&](const char* s, int ks, int j) __attribute__((always_inline)) -> i32x4_t {
    if (B_KMAJOR) return *(const i32x4_t*)(s + b_rd[B_KMAJOR ? ks : 0] + j * 16 * 128);
    const char* q = s + b_rd[B_KMAJOR ? 0 : j] + ks * 32 * (C::BN * 2);
    const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr_t)q);
    const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr_t)(q + 4 * (C::BN * 2)));
    return __builtin_bit_cast(i32x4_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // ---- the copy stream: the cursor's tile window and offsets along K ----
  const TileWalk walk = sched_walk(num_tiles, p.tile_split != 0);
  const int w_first = (int)walk.first, w_end = (int)walk.end, w_stride = (int)walk.stride;
  if (w_first >= w_end) return;
  i32x4_t ra, rb;
  int koff_a = 0, koff_b = 0, left = 0;  // left: slabs of the cursor's tile not yet requested (0: there are no more tiles)
  int next_id = w_first;                 // the tile behind the cursor's
  const int step_b = B_KMAJOR ? BKD * 2 : __builtin_amdgcn_readfirstlane(BKD * ld_b);
  Tile seen;
  int seen_id = -1, seen_g = -1;
  auto seek = [&]() __attribute__((always_inline)) {
    koff_a = koff_b = 0;
    if (next_id < w_end) {
      const Tile t = sched_tile<C::BM, C::BN>(p, sched, next_id, seen_g);
      seen = t;
      seen_id = next_id;
      seen_g = t.g;
      const int n_left = p.N - t.n0;
      ra = make_rsrc32(uniform64((uint64_t)p.A + (uint64_t)(t.row0 * ld)), t.rows * ld);
      if (B_KMAJOR) rb = make_rsrc32(uniform64((uint64_t)p.B + (uint64_t)(((int64_t)t.g * p.N + t.n0) * ld)), (n_left < C::BN ? n_left : C::BN) * ld);
      // NN: to the end of the group's last token row; what a row segment reads beyond its row are columns that are not stored
      else rb = make_rsrc32(uniform64((uint64_t)p.B + (uint64_t)(((int64_t)t.g * p.K * p.N + t.n0) * 2)), p.K * ld_b - t.n0 * 2);
      left = kt_n;
      next_id += w_stride;
    } else {
      ra = make_rsrc32((uint64_t)p.A, 0);
      rb = make_rsrc32((uint64_t)p.A, 0);
      left = 0;
    }
    asm volatile("s_nop 4" : : "s"(ra), "s"(rb));  // wait states between a vector write of a scalar register and a copy that reads it
  };
  // copy k of the cursor's slab, into the buffer at `buf`
  auto copy_k = [&](int k, uint32_t buf) __attribute__((always_inline)) {
    const bool last = left == 1;
    if (k < C::CA) copy_slab_b128(ra, buf + (wave + 4 * k) * 1024, last ? vo_a[k] | tail : vo_a[k], koff_a);
    else copy_slab_b128(rb, buf + C::A_BYTES + (wave + 4 * (k - C::CA)) * 1024, last && B_KMAJOR ? vo_b[k - C::CA] | tail : vo_b[k - C::CA], koff_b);
  };
  auto advance = [&]() __attribute__((always_inline)) {
    if (left > 1) {
      koff_a += BKD * 2;
      koff_b += step_b;
      --left;
    } else if (left == 1) {
      seek();
    }
  };

  i32x4_t fa[2][C::TM], fb[2][C::TN];
  i32x8_t fa8[C::TM], fb8[C::TN];  // FP8
  f32x4_t acc[C::TM][C::TN];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::TM; ++i)
#pragma unroll
      for (int j = 0; j < C::TN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  auto read = [&](int set, const char* s, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < C::TN; ++j) fb[set][j] = load_b(s, ks, j);
#pragma unroll
    for (int i = 0; i < C::TM; ++i) fa[set][i] = load_a(s, ks, i);
    __builtin_amdgcn_sched_barrier(0);
  };
  // One K step on fragment set `set`; copies k0 .. k0 + NC / 2 - 1 of the cursor's slab go out between the multiplies
  auto step = [&](int set, int k0, uint32_t copy_buf) __attribute__((always_inline)) {
    constexpr int SP = C::TM * C::TN / (C::NC / 2);
#pragma unroll
    for (int i = 0; i < C::TM; ++i)
#pragma unroll
      for (int jj = 0; jj < C::TN; ++jj) {
        const int j = (i & 1) ? C::TN - 1 - jj : jj, n = i * C::TN + jj;
        const i32x4_t x = B_KMAJOR ? fa[set][i] : fb[set][j], y = B_KMAJOR ? fb[set][j] : fa[set][i];
        if (DT == DT_BF16) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x), __builtin_bit_cast(bf16x8_t, y), acc[i][j], 0, 0, 0);
        else acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, x), __builtin_bit_cast(f16x8_t, y), acc[i][j], 0, 0, 0);
        if (n % SP == 0 && n / SP < C::NC / 2) {
          __builtin_amdgcn_sched_barrier(0);
          copy_k(k0 + n / SP, copy_buf);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  // ---- FP8 ----
  auto frag8 = [&](const char* s, const int (&at)[2], int block) __attribute__((always_inline)) -> i32x8_t {
    const i32x4_t lo = *(const i32x4_t*)(s + at[0] + block * 16 * 128), hi = *(const i32x4_t*)(s + at[1] + block * 16 * 128);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto read8_a = [&](const char* s, int half) __attribute__((always_inline)) {
    if constexpr (FP8) {
#pragma unroll
      for (int i = half * C::TM / 2; i < (half + 1) * C::TM / 2; ++i) fa8[i] = frag8(s, a_rd, i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto read8_b = [&](const char* s, int j) __attribute__((always_inline)) {
    if constexpr (FP8) fb8[j] = frag8(s, b_rd, j);
  };
  // Half a slab's multiplies: row blocks of `half`; copies k0 .. k0 + NC / 2 - 1 go out between them.  The second half reads the next slab's
  // fragments of B (at `next`) behind the last use of this one's.
  auto step8 = [&](int half, int k0, uint32_t copy_buf, const char* next) __attribute__((always_inline)) {
    if constexpr (FP8) {
      constexpr int HM = C::TM / 2, SP = HM * C::TN / (C::NC / 2);
      static_assert(SP >= 1, "half a slab's copies go out during half its multiplies");
#pragma unroll
      for (int j = 0; j < C::TN; ++j) {
#pragma unroll
        for (int ii = 0; ii < HM; ++ii) {
          const int i = half * HM + ((j & 1) ? HM - 1 - ii : ii), n = j * HM + ii;
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fa8[i], fb8[j], acc[i][j], FA, FB, 0, 0, 0, 0);
          if (n % SP == 0 && n / SP < C::NC / 2) {
            __builtin_amdgcn_sched_barrier(0);
            copy_k(k0 + n / SP, copy_buf);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (half == 1) {
          __builtin_amdgcn_sched_barrier(0);
          read8_b(next, j);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  seek();
#pragma unroll 1
  for (int s = 0; s < C::ST - 1; ++s) {
#pragma unroll
    for (int k = 0; k < C::NC; ++k) copy_k(k, smem_addr + s * C::STAGE_BYTES);
    advance();
  }
#pragma unroll
  for (int k = 0; k < C::NC / 2; ++k) copy_k(k, smem_addr + (C::ST - 1) * C::STAGE_BYTES);
  clear();
  wait_vmcnt<(C::ST - 2) * C::NC + C::NC / 2>();
  __syncthreads();
  if constexpr (FP8) {
    read8_a(smem, 0);
#pragma unroll
    for (int j = 0; j < C::TN; ++j) read8_b(smem, j);
  } else {
    read(0, smem, 0);
  }
  int buf = 0, prev = (C::ST - 1) * C::STAGE_BYTES;  // byte offsets of the current slab's buffer and the one before it
  for (int tile_id = w_first; tile_id < w_end; tile_id += w_stride) {
    const Tile cur = tile_id == seen_id ? seen : sched_tile<C::BM, C::BN>(p, sched, tile_id);
    for (int kt = 0; kt < kt_n; ++kt) {
      const int nxt = buf == (C::ST - 1) * C::STAGE_BYTES ? 0 : buf + C::STAGE_BYTES;
      if constexpr (FP8) {
        read8_a(smem + buf, 1);
        step8(0, C::NC / 2, smem_addr + prev, nullptr);
      } else {
        read(1, smem + buf, 1);
        step(0, C::NC / 2, smem_addr + prev);
      }
      advance();
      // this wave's copies of the next slab have landed (a tile's stores, younger than those copies for ST - 2 slabs, may be in flight as well),
      // and it has read all it needs of this one
      if (kt < C::ST - 2 && tile_id != w_first) wait_vmcnt<(C::ST - 2) * C::NC + (B_KMAJOR ? C::STORES_NT : C::STORES_NN)>();
      else wait_vmcnt<(C::ST - 2) * C::NC>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __syncthreads();
      if constexpr (FP8) {
        read8_a(smem + nxt, 0);
        step8(1, 0, smem_addr + buf, smem + nxt);
      } else {
        read(0, smem + nxt, 0);
        step(1, 0, smem_addr + buf);
      }
      prev = buf;
      buf = nxt;
    }
    // ---- epilogue ----
    const int rows_left = cur.rows - wm0;
    const i32x4_t rc = make_rsrc32(uniform64((uint64_t)p.C + (uint64_t)(((cur.row0 + wm0) * (int64_t)p.N + cur.n0 + wn0) * 2)),
                                   (rows_left < C::BM / 2 ? rows_left : C::BM / 2) * p.N * 2);
    const int cols = p.N - cur.n0 - wn0;
    int el = lane;
    asm volatile("s_nop 4" : "+v"(el) : "s"(rc));
    const int e16 = el & 15, eg = el >> 4;
    if (B_KMAJOR) {
      const int off0 = C::TN * e16 < cols ? (4 * eg * p.N + C::TN * e16) * 2 : kNoFetch;
      float cs[C::TN];
      if constexpr (FP8) {  // the scales of the lane's columns; those of its rows block by block
#pragma unroll
        for (int j = 0; j < C::TN; ++j) cs[j] = C::TN * e16 < cols ? p.scale_n[(int64_t)cur.g * p.N + cur.n0 + wn0 + C::TN * e16 + j] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < C::TM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (FP8) {
            const int row = wm0 + 16 * i + 4 * eg + r;
            const float rs = row < cur.rows ? p.scale_m[cur.row0 + row] : 0.f;
#pragma unroll
            for (int j = 0; j < C::TN; ++j) acc[i][j][r] = acc[i][j][r] * rs * cs[j];
          }
          const int off = off0 + (16 * i + r) * p.N * 2;
          if constexpr (C::TN == 4) {
            const uint2 v = pack4<DT>(acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]);
            const i32x2_t w = {(int)v.x, (int)v.y};
            asm volatile("buffer_store_dwordx2 %0, %1, %2, 0 offen\n\ts_nop 1" : : "v"(w), "v"(off), "s"(rc) : "memory");
          } else {
            const uint32_t w = pack2<DT>(acc[i][0][r], acc[i][1][r]);
            asm volatile("buffer_store_dword %0, %1, %2, 0 offen\n\ts_nop 1" : : "v"(w), "v"(off), "s"(rc) : "memory");
          }
        }
    } else {
      char* const stage = smem + kDeepEpiOff + wave * C::EPI_WAVE_BYTES;
      constexpr int CPS = 2 * C::TN, PASSES = 16 * CPS / 64;
#pragma unroll
      for (int i = 0; i < C::TM; ++i) {
#pragma unroll
        for (int j = 0; j < C::TN; ++j)
          *(uint2*)(stage + e16 * C::EPI_PITCH + (16 * j + 4 * eg) * 2) = pack4<DT>(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
#pragma unroll
        for (int it = 0; it < PASSES; ++it) {
          const int idx = it * 64 + el, r = idx / CPS, ch = idx % CPS;
          const i32x4_t v = *(const i32x4_t*)(stage + r * C::EPI_PITCH + ch * 16);
          store_b128<false, 1>(v, ch * 8 < cols ? ((16 * i + r) * p.N + ch * 8) * 2 : kNoFetch, rc);
        }
      }
    }
    clear();
  }
  wait_vmcnt<0>();  // the trailing zero-length copies still write LDS
}

// The tile height of the table is 128; the small tiles take the half-height cut that sched_init leaves.
template <int DT, int LAYOUT, int FA = 0, int FB = 0>
__global__ __launch_bounds__(256) void gemm_deep_kernel(const GemmParams p) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  auto& sched = *reinterpret_cast<SchedTableT<kFastMaxGroups>*>(smem + kDeepSchedOff);
  const int32_t half_tile0 = sched_init<128>(p, sched);
  typedef DeepCfg<64, 64, 8> Small;
  typedef DeepCfg<64, 128, 5> Mid;
  typedef DeepCfg<128, 128, 4> Wide;
  const int wgs = (int)gridDim.x, rows64 = sched.tile0[p.G] + sched.pad_, rows128 = sched.tile0[p.G];
  const int cols64 = (p.N + 63) / 64, cols128 = (p.N + 127) / 128;
  auto rounds = [&](int64_t tiles) { return (int)((tiles + wgs - 1) / wgs); };
  const int small = rounds((int64_t)rows64 * cols64) * 16, mid = rounds((int64_t)rows64 * cols128) * 24, wide = rounds((int64_t)rows128 * cols128) * 32;
  if (wide <= mid && wide < small) {
    gemm_deep_body<Wide, DT, LAYOUT, FA, FB>(p);
  } else {
    sched_use_half_height(p, sched, half_tile0);
    if (small <= mid) gemm_deep_body<Small, DT, LAYOUT, FA, FB>(p);
    else gemm_deep_body<Mid, DT, LAYOUT, FA, FB>(p);
  }
}

template <int DT, int LAYOUT, int FA = 0, int FB = 0>
int launch_deep(const GemmParams& p, hipStream_t s) {
  static bool attr_set[64] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  const bool listed = dev >= 0 && dev < 64;
  auto kern = gemm_deep_kernel<DT, LAYOUT, FA, FB>;
  if (!listed || !attr_set[dev]) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kDeepSmemBytes) != hipSuccess)
      return check_launch("hipFuncSetAttribute(gemm_deep)");
    if (listed) attr_set[dev] = true;
  }
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), kDeepSmemBytes, s, p);
  return check_launch("gemm_deep");
}

}  // namespace

// Launches whose 128x128 tiles fit one round of the workgroups: for certain, or with a fifth to spare by the likely number of row tiles (a
// group's last one half full, one at least).  More rounds of small tiles lose to the larger tiles' kernels: 8 groups of 4096 rows, N = 1536,
// K = 2048 (432 tiles): 34 us there, 52 here; at 252 tiles 32.6 and 31.0.  Masked launches: counts anywhere up to the slots, so for certain only.
static bool few_tiles(const GemmParams& p) {
  int grid = num_cus();
  if (p.grid_limit > 0 && p.grid_limit < grid) grid = p.grid_limit;
  const int64_t cols = (p.N + 127) / 128;
  if (p.mode == MODE_MASKED) return p.G * ((p.m_stride + 127) / 128) * cols <= grid;
  const int64_t used = p.m_total < p.G ? p.m_total : p.G;  // groups that can have rows
  const int64_t most = (p.m_total + 127 * used) / 128, half_full = p.m_total / 128 + used / 2, likely = half_full > used ? half_full : used;
  return most * cols <= grid || 5 * likely * cols <= 4 * grid;
}

bool deep_supported(const GemmParams& p, int dt, int layout, bool any_size) {
  if (dt != DT_BF16 && dt != DT_F16) return false;
  if (layout != DEEP_NT && layout != DEEP_NN) return false;
  if (p.mode != MODE_MG && p.mode != MODE_MG_PAD && p.mode != MODE_MASKED) return false;
  if (p.G > 256 || p.q_fmt != 0) return false;
  if ((p.N & 7) != 0 || p.K < 8 || (p.K & 7) != 0) return false;
  if ((int64_t)p.K * 2 * 128 >= (1ll << 30) || (int64_t)p.N * 2 * 128 >= (1ll << 30)) return false;
  if (layout == DEEP_NN && ((int64_t)p.K + 64) * p.N * 2 >= (1ll << 30)) return false;
  return any_size || few_tiles(p);
}

// The same for FP8 operands with per-channel scales.
bool deep_fp8_supported(const GemmParams& p, bool any_size) {
  if (p.mode != MODE_MG || p.G > 256 || (p.N & 7) != 0 || p.K < 16 || (p.K & 15) != 0) return false;
  if ((int64_t)p.K * 128 >= (1ll << 30) || (int64_t)p.N * 2 * 128 >= (1ll << 30)) return false;
  return any_size || few_tiles(p);
}

template <int FA, int FB>
static int launch_deep_fp8_out(const GemmParams& p, int out_dt, hipStream_t s) {
  return out_dt == DT_F16 ? launch_deep<DT_F16, DEEP_FP8, FA, FB>(p, s) : launch_deep<DT_BF16, DEEP_FP8, FA, FB>(p, s);
}

int launch_deep_fp8(const GemmParams& p, int ta, int tb, int out_dt, hipStream_t s) {
  if (ta == DT_E4M3) return tb == DT_E4M3 ? launch_deep_fp8_out<0, 0>(p, out_dt, s) : launch_deep_fp8_out<0, 1>(p, out_dt, s);
  return tb == DT_E4M3 ? launch_deep_fp8_out<1, 0>(p, out_dt, s) : launch_deep_fp8_out<1, 1>(p, out_dt, s);
}

int launch_deep_16bit(const GemmParams& p, int dt, int layout, hipStream_t s) {
  if (layout == DEEP_NT) return dt == DT_BF16 ? launch_deep<DT_BF16, DEEP_NT>(p, s) : launch_deep<DT_F16, DEEP_NT>(p, s);
  return dt == DT_BF16 ? launch_deep<DT_BF16, DEEP_NN>(p, s) : launch_deep<DT_F16, DEEP_NN>(p, s);
}

}  // namespace tgg
