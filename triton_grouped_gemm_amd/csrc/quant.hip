// FP8 quantizers for gfx950: streaming, HBM-bound kernels.
//
//  * trans_quant128: per 128x128 block of a grouped bf16 matrix, quantise with one
//    fp32 scale, transpose, and place at the group's 128-padded column offset.
//  * token_cast128:  1x128 groups along K (activation recipe).
//  * block_cast128:  128x128 blocks, no transpose (weight recipe).
//
// Bit-exactness contract: scale and quotient/product are single IEEE fp32
// operations on the exact fp32 value of the bf16 input; fp32 -> fp8 is
// round-to-nearest-even after an explicit clamp (hardware v_cvt_pk_{fp8,bf8}_f32).
#include "common.hpp"
#include "sched.hpp"
#include "launch.hpp"

namespace tgg {

namespace {

TGG_DEV float bf16_bits_to_f32(uint32_t h) { return __builtin_bit_cast(float, h << 16); }

template <int FMT> TGG_DEV uint32_t cvt_pk(float a, float b, uint32_t old, bool hi) {
  if (FMT == DT_E4M3) return hi ? __builtin_amdgcn_cvt_pk_fp8_f32(a, b, old, true) : __builtin_amdgcn_cvt_pk_fp8_f32(a, b, old, false);
  return hi ? __builtin_amdgcn_cvt_pk_bf8_f32(a, b, old, true) : __builtin_amdgcn_cvt_pk_bf8_f32(a, b, old, false);
}

template <int FMT> TGG_DEV uint32_t cvt4(float a, float b, float c, float d) {
  uint32_t w = cvt_pk<FMT>(a, b, 0u, false);
  return cvt_pk<FMT>(c, d, w, true);
}

template <int FMT> struct FmtMax;
template <> struct FmtMax<DT_E4M3> { static constexpr float v = 448.0f; };
template <> struct FmtMax<DT_E5M2> { static constexpr float v = 57344.0f; };

TGG_DEV float clampf(float x, float lo, float hi) { return fminf(fmaxf(x, lo), hi); }

TGG_DEV float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// abs-max of 8 bf16 packed in a 16-byte vector
TGG_DEV float amax8(i32x4_t v) {
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = (uint32_t)v[i];
    m = fmaxf(m, fabsf(bf16_bits_to_f32(w & 0xffffu)));
    m = fmaxf(m, fabsf(bf16_bits_to_f32(w >> 16)));
  }
  return m;
}

// The same as an integer: the largest bf16 bit pattern without its sign, which orders like the magnitudes as long as
// none is a NaN (patterns above 0x7f80); two per instruction.
typedef __attribute__((ext_vector_type(2))) uint16_t u16x2_t;
TGG_DEV u16x2_t amax_bits(u16x2_t m, i32x4_t v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2_t, (uint32_t)v[i] & 0x7fff7fffu));
  return m;
}

// Correctly rounded f / s for many f and one s, r = the correctly rounded 1 / s: two corrections of f * r by its exact
// remainder.  The first leaves at most an ulp of error, from which the second rounds correctly (Markstein, "Computation
// of elementary functions on the IBM RISC System/6000 processor", 1990), as long as neither r nor the remainder leaves
// the range of normal numbers.  s is at least 1e-12, so a remainder does that only for quotients below 2^-63, whose FP8
// code is a zero of f's sign either way; f below kMaxFastValue keeps s and r in range.  The remainder is taken as q s - f:
// a zero f keeps its sign that way.  5 operations against the 10 of the compiler's division, one of those a reciprocal
// at a quarter of the rate.
constexpr float kMaxFastValue = 1e30f;
TGG_DEV float div_by(float f, float s, float r) {
  float q = f * r;
  q = __builtin_fmaf(-__builtin_fmaf(q, s, -f), r, q);
  return __builtin_fmaf(-__builtin_fmaf(q, s, -f), r, q);
}

// Row tile pm of the groups laid out by 128-row tiles: where its rows start and how many are valid; rows < 0 past the last
// tile.  Every wave finds it for itself, without LDS or barriers: a lane sums the sizes of up to 16 neighbouring groups,
// a scan over the lanes gives their first tiles, and the groups of the lane that holds pm are walked once more.  Sizes are
// clipped to the matrix as sched_init clips them.
TGG_DEV void find_row_tile(const GemmParams& p, int pm, int64_t& row0, int& rows) {
  const int lane = lane_id(), per = (p.G + 63) >> 6;
  const int g0 = min(p.G, lane * per), g1 = min(p.G, g0 + per);
  int64_t sum = 0;
  for (int g = g0; g < g1; ++g) sum += load_size(p.sizes, p.sizes_i64, g);
  int64_t start = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int64_t o = __shfl_up(start, d, 64);
    if (lane >= d) start += o;
  }
  start -= sum;
  auto tiles_of = [&](int64_t first, int64_t size, int64_t& valid) {
    valid = first >= p.m_total ? 0 : min(size, p.m_total - first);
    return (int)((valid + 127) >> 7);
  };
  int tiles = 0;
  int64_t at = start, valid;
  for (int g = g0; g < g1; ++g) {
    const int64_t size = load_size(p.sizes, p.sizes_i64, g);
    tiles += tiles_of(at, size, valid);
    at += size;
  }
  int first = tiles;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(first, d, 64);
    if (lane >= d) first += o;
  }
  first -= tiles;
  const uint64_t mine = __ballot(pm >= first && pm < first + tiles);
  rows = -1;
  row0 = 0;
  if (mine == 0) return;
  const int owner = __builtin_ctzll(mine);
  int left = pm - __builtin_amdgcn_readlane(first, owner);
  at = __shfl(start, owner, 64);
  for (int g = min(p.G, owner * per); g < p.G; ++g) {
    const int64_t size = load_size(p.sizes, p.sizes_i64, g);
    const int t = tiles_of(at, size, valid);
    if (left < t) {
      const int64_t r0 = at + (int64_t)left * 128;
      row0 = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)r0) | ((int64_t)__builtin_amdgcn_readfirstlane((int)(r0 >> 32)) << 32);
      rows = __builtin_amdgcn_readfirstlane((int)min((int64_t)128, valid - (int64_t)left * 128));
      return;
    }
    left -= t;
    at += size;
  }
}

// A block that holds an infinity, a NaN or values beyond 1e30, element by element from memory, with the maximum over the
// numbers alone and the division itself: leaves the codes in `codes` (layout below) and returns the scale.
template <int FMT>
TGG_DEV float trans_block_any(const uint16_t* x, int ld, int rows, uint8_t* codes, float* wmax) {
  constexpr float fmax_ = FmtMax<FMT>::v;
  const int tid = threadIdx.x, c = tid & 127;
  float amax = 0.f;
  for (int r = tid >> 7; r < rows; r += 2) amax = fmaxf(amax, fabsf(bf16_bits_to_f32(x[(int64_t)r * ld + c])));
  amax = wave_max(amax);
  __syncthreads();
  if ((tid & 63) == 0) wmax[tid >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  const float scale = clampf(amax / fmax_, 1e-12f, 3e38f);
  for (int r = tid >> 7; r < 128; r += 2) {
    const float f = r < rows ? bf16_bits_to_f32(x[(int64_t)r * ld + c]) : 0.f;
    codes[c * 128 + (((r >> 4) ^ ((c >> 3) & 7)) * 16) + (r & 15)] = (uint8_t)cvt_pk<FMT>(clampf(f / scale, -fmax_, fmax_), 0.f, 0u, false);
  }
  return scale;
}

// Output store: the codes are written once and not read here.
TGG_DEV void store_nt(void* dst, i32x4_t v) {
  // s_nop 1: the data registers of a 16-byte store must not be overwritten within two wait states, and the compiler
  // does not look inside this statement
  asm volatile("global_store_dwordx4 %0, %1, off nt\n\ts_nop 1" : : "v"(dst), "v"(v) : "memory");
}

// With more than 256 groups a workgroup takes four neighbouring blocks of its row tile one after another: the search for the
// rows walks 5 to 16 sizes a lane then, in three passes, and costs more than the block.  One block / four, 131072 x 4096
// values: 512 groups 503 / 395 us, 1024 groups 1036 / 487 (a table that 2048 persistent workgroups made once each: 623, 929);
// 524288 x 4096: 1550 / 1327, 2659 / 1448 (1605, 1895).  Eight and sixteen blocks leave the last workgroups more to do:
// 419 and 456 us with 512 groups, 467 and 509 with 1024.
constexpr int kManyGroups = 256, kManyCols = 4;

// One 128x128 block per workgroup, 256 threads.  Bound by memory: 3 bytes per element, rows of 256 bytes in, rows of 128
// bytes out.  A workgroup per block (COLS = 1) lets the hardware fill the chip evenly and beats 2048 workgroups that walk the blocks
// (a copy with this access pattern: 5.2 against 4.9 TB/s), which is why the block finds its rows without a table; streaming
// stores are worth another 3-15 %.  655360 x 4096 values 1770 -> 1598 us (4.59 -> 5.08 TB/s), 33001 x 4096 98 -> 82 us
// (4.5 -> 5.4 TB/s), of which the division's share is small: it overlaps the memory traffic of the other blocks of a CU.
// Read: thread (rr = tid/16, cv = tid%16) owns rows rr*8 .. rr*8+7, columns cv*8 .. cv*8+7.
// LDS holds the transposed codes: byte (c, r) at c*128 + ((r/16) ^ ((c/8)%8))*16 + r%16.
// padded (optional): the sizes rounded up to 128, in their own integer type.
template <int FMT, int COLS>
__global__ __launch_bounds__(256) void trans_quant128_kernel(const uint16_t* __restrict__ x, uint8_t* __restrict__ codes,
                                                            float* __restrict__ scales, GemmParams p, int64_t m_expand,
                                                            void* __restrict__ padded) {
  __shared__ __attribute__((aligned(16))) uint8_t codes_t[128 * 128];
  __shared__ float wmax[4];
  const int N = p.N;
  const int tiles_n = N >> 7;
  const int m_tiles_all = (int)(m_expand >> 7);
  const int tid = threadIdx.x;
  const int rr = tid >> 4, cv = tid & 15;
  constexpr float fmax_ = FmtMax<FMT>::v;
  if (padded && blockIdx.x == 0) {
    for (int g = tid; g < p.G; g += 256) {
      if (p.sizes_i64) ((int64_t*)padded)[g] = (((const int64_t*)p.sizes)[g] + 127) & ~(int64_t)127;
      else ((int32_t*)padded)[g] = (((const int32_t*)p.sizes)[g] + 127) & ~127;
    }
  }
  const unsigned runs = COLS > 1 ? ((unsigned)tiles_n + COLS - 1) / COLS : (unsigned)tiles_n;
  const int pm = (int)(blockIdx.x / runs), bn0 = (int)(blockIdx.x % runs) * COLS;
  if (pm >= m_tiles_all) return;
  int64_t row0;
  int rows;
  find_row_tile(p, pm, row0, rows);
  for (int bn = bn0; bn < (COLS > 1 ? min(tiles_n, bn0 + COLS) : bn0 + 1); ++bn) {
    uint8_t* out_base = codes + ((int64_t)bn * 128) * m_expand + (int64_t)pm * 128;
    if (rows < 0) {  // tail beyond the padded groups: zero codes, zero scale
      const i32x4_t z = {0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = (tid >> 3) + 32 * i, u = tid & 7;
        store_nt(out_base + (int64_t)c * m_expand + u * 16, z);
      }
      if (tid == 0) scales[(int64_t)bn * m_tiles_all + pm] = 0.f;
      continue;
    }
    i32x4_t v[8];
    u16x2_t top = {0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = rr * 8 + i;
      i32x4_t val = {0, 0, 0, 0};
      if (r < rows) val = *(const i32x4_t*)(x + (row0 + r) * (int64_t)N + bn * 128 + cv * 8);
      v[i] = val;
      top = amax_bits(top, val);
    }
    uint32_t bits = top[0] > top[1] ? top[0] : top[1];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const uint32_t o = (uint32_t)__shfl_xor((int)bits, off, 64);
      bits = o > bits ? o : bits;
    }
    if ((tid & 63) == 0) wmax[tid >> 6] = bf16_bits_to_f32(bits);
    __syncthreads();
    // the pattern's order survives the conversion to float, except that a NaN makes the sum one
    const float amax = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const bool numbers = wmax[0] + wmax[1] + wmax[2] + wmax[3] < 4.f * kMaxFastValue;
    float scale = clampf(amax / fmax_, 1e-12f, 3e38f);
    if (__builtin_expect(numbers, 1)) {
      const float inv = 1.0f / scale;
      // column j of this thread's 8x8 patch -> 8 consecutive r bytes
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float q[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t w = (uint32_t)v[i][j >> 1];
          const float f = __builtin_bit_cast(float, (j & 1) ? (w & 0xffff0000u) : (w << 16));
          q[i] = clampf(div_by(f, scale, inv), -fmax_, fmax_);
        }
        uint2 pk;
        pk.x = cvt4<FMT>(q[0], q[1], q[2], q[3]);
        pk.y = cvt4<FMT>(q[4], q[5], q[6], q[7]);
        const int c = cv * 8 + j;
        const int slot = (rr >> 1) ^ (cv & 7);
        *(uint2*)(codes_t + c * 128 + slot * 16 + (rr & 1) * 8) = pk;
      }
    } else {
      scale = trans_block_any<FMT>(x + row0 * (int64_t)N + bn * 128, N, rows, codes_t, wmax);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = (tid >> 3) + 32 * i, u = tid & 7;
      const i32x4_t o = *(const i32x4_t*)(codes_t + c * 128 + ((u ^ ((c >> 3) & 7)) * 16));
      store_nt(out_base + (int64_t)c * m_expand + u * 16, o);
    }
    if (tid == 0) scales[(int64_t)bn * m_tiles_all + pm] = scale;
  }
}

// 16 lanes per 1x128 group; each lane 8 elements.  A workgroup's 16 lane groups take 16 neighbouring groups
// along the axis the scales are contiguous in, so that the 16 scale stores of a step fill one 64-byte segment:
//   scales [rows, kblocks]  (mn_major = 0): 16 consecutive K blocks of one row
//   scales [kblocks, rows]  (mn_major = 1): the same K block of 16 consecutive rows
// Two steps are in flight per thread.
template <int FMT>
__global__ __launch_bounds__(256) void token_cast128_kernel(const uint16_t* __restrict__ x, uint8_t* __restrict__ codes,
                                                           float* __restrict__ scales, int64_t rows, int kblocks, int mn_major) {
  constexpr float fmax_ = FmtMax<FMT>::v;
  const int64_t groups = rows * kblocks;
  const int sub = threadIdx.x & 15, grp = threadIdx.x >> 4;
  // step s of the launch covers 16 groups; steps are numbered so that consecutive steps touch neighbouring memory
  const int64_t row_blocks = (rows + 15) / 16;
  const int64_t steps = mn_major ? row_blocks * kblocks : (groups + 15) / 16;
  auto group_of = [&](int64_t step, int64_t& g, int64_t& sidx) -> bool {
    if (mn_major) {
      const int64_t rb = step / kblocks;
      const int kb = (int)(step - rb * kblocks);
      const int64_t r = rb * 16 + grp;
      g = r * kblocks + kb;
      sidx = (int64_t)kb * rows + r;
      return r < rows;
    }
    g = step * 16 + grp;
    sidx = g;
    return g < groups;
  };
  auto quantise = [&](const i32x4_t v, int64_t g, int64_t sidx, bool ok) {
    float amax = amax8(v);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    amax = fmaxf(amax, 1e-4f);
    const float mult = (1.0f / amax) * fmax_;  // torch evaluates `448.0 / amax` as reciprocal * 448
    float f[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = (uint32_t)v[i];
      f[2 * i] = bf16_bits_to_f32(w & 0xffffu) * mult;
      f[2 * i + 1] = bf16_bits_to_f32(w >> 16) * mult;
    }
    uint2 pk;
    pk.x = cvt4<FMT>(f[0], f[1], f[2], f[3]);
    pk.y = cvt4<FMT>(f[4], f[5], f[6], f[7]);
    if (ok) {
      *(uint2*)(codes + g * 128 + sub * 8) = pk;
      if (sub == 0) scales[sidx] = amax / fmax_;
    }
  };
  const i32x4_t zero = {0, 0, 0, 0};
  for (int64_t s0 = (int64_t)blockIdx.x * 2; s0 < steps; s0 += (int64_t)gridDim.x * 2) {
    int64_t g0, g1, i0, i1;
    const bool ok0 = group_of(s0, g0, i0);
    const bool ok1 = s0 + 1 < steps && group_of(s0 + 1, g1, i1);
    const i32x4_t v0 = ok0 ? *(const i32x4_t*)(x + g0 * 128 + sub * 8) : zero;
    const i32x4_t v1 = ok1 ? *(const i32x4_t*)(x + g1 * 128 + sub * 8) : zero;
    quantise(v0, g0, i0, ok0);
    quantise(v1, g1, i1, ok1);
  }
}

// 128x128 blocks of a [batch, R, C] tensor (blocks never straddle batch entries).
template <int FMT>
__global__ __launch_bounds__(256) void block_cast128_kernel(const uint16_t* __restrict__ x, uint8_t* __restrict__ codes,
                                                           float* __restrict__ scales, int batch, int R, int C) {
  __shared__ float wmax[4];
  constexpr float fmax_ = FmtMax<FMT>::v;
  const int tr = (R + 127) >> 7, tc = (C + 127) >> 7;
  const int64_t total = (int64_t)batch * tr * tc;
  const int tid = threadIdx.x;
  const int rr = tid >> 4, cv = tid & 15;
  const bool vec_ok = (C & 7) == 0;
  for (int64_t tile = blockIdx.x; tile < total; tile += gridDim.x) {
    const int b = (int)(tile / (tr * tc));
    const int rem = (int)(tile % (tr * tc));
    const int r0 = (rem / tc) * 128, c0 = (rem % tc) * 128;
    const uint16_t* src = x + (int64_t)b * R * C;
    uint8_t* dst = codes + (int64_t)b * R * C;
    i32x4_t v[8];
    float amax = 0.f;
    const int c = c0 + cv * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = r0 + rr + 16 * i;
      i32x4_t val = {0, 0, 0, 0};
      if (r < R && c < C) {
        const uint16_t* s = src + (int64_t)r * C + c;
        if (vec_ok) {
          val = *(const i32x4_t*)s;
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (c + e < C) val[e >> 1] |= (int)((uint32_t)s[e] << ((e & 1) * 16));
        }
      }
      v[i] = val;
      amax = fmaxf(amax, amax8(val));
    }
    amax = wave_max(amax);
    __syncthreads();
    if ((tid & 63) == 0) wmax[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3])), 1e-4f);
    const float mult = (1.0f / amax) * fmax_;  // torch evaluates `448.0 / amax` as reciprocal * 448
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = r0 + rr + 16 * i;
      if (r >= R || c >= C) continue;
      float f[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = (uint32_t)v[i][e];
        f[2 * e] = bf16_bits_to_f32(w & 0xffffu) * mult;
        f[2 * e + 1] = bf16_bits_to_f32(w >> 16) * mult;
      }
      uint2 pk;
      pk.x = cvt4<FMT>(f[0], f[1], f[2], f[3]);
      pk.y = cvt4<FMT>(f[4], f[5], f[6], f[7]);
      uint8_t* d = dst + (int64_t)r * C + c;
      if (vec_ok) {
        *(uint2*)d = pk;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (c + e < C) d[e] = (uint8_t)(((e < 4) ? pk.x : pk.y) >> ((e & 3) * 8));
      }
    }
    if (tid == 0) scales[tile] = amax / fmax_;
  }
}

// [rows, cols] -> [cols, rows] for activation scales (cols = K / 128, a few dozen).  A workgroup takes 64 rows: one run
// of memory in, 64-float runs out, 64 columns at a time through LDS.
__global__ __launch_bounds__(256) void scales_transpose_kernel(const float* __restrict__ in, float* __restrict__ out,
                                                              int64_t rows, int cols) {
  __shared__ float t[64][65];
  const int64_t r0 = (int64_t)blockIdx.x * 64;
  const int n = (int)min((int64_t)64, rows - r0);
  for (int c0 = 0; c0 < cols; c0 += 64) {
    const int w = min(64, cols - c0);
    for (int i = threadIdx.x; i < n * w; i += 256) {
      const int r = i / w, c = i - r * w;
      t[c][r] = in[(r0 + r) * cols + c0 + c];
    }
    __syncthreads();
    const int r = threadIdx.x & 63;
    if (r < n)
      for (int c = threadIdx.x >> 6; c < w; c += 4) out[(int64_t)(c0 + c) * rows + r0 + r] = t[c][r];
    __syncthreads();
  }
}

template <int FMT>
__global__ void cvt_fp8_kernel(const float* __restrict__ in, uint8_t* __restrict__ out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (uint8_t)cvt_pk<FMT>(in[i], 0.f, 0u, false);
}

}  // namespace

int launch_trans_quant128(const void* x, void* codes, float* scales, const GemmParams& p, int64_t m_expand, void* padded,
                          int fmt, hipStream_t s) {
  const int64_t tiles = (m_expand >> 7) * (int64_t)(p.N >> 7);
  if (tiles >= (1ll << 24)) return set_error("a matrix of %lld 128 x 128 blocks is too large for one launch", (long long)tiles);
#define TGG_LAUNCH(FMT) \
  do { \
    if (many) hipLaunchKernelGGL((trans_quant128_kernel<FMT, kManyCols>), g, b, 0, s, (const uint16_t*)x, (uint8_t*)codes, scales, p, m_expand, padded); \
    else hipLaunchKernelGGL((trans_quant128_kernel<FMT, 1>), g, b, 0, s, (const uint16_t*)x, (uint8_t*)codes, scales, p, m_expand, padded); \
  } while (0)
  const bool many = p.G > kManyGroups;
  const int64_t runs = many ? (m_expand >> 7) * (((p.N >> 7) + kManyCols - 1) / kManyCols) : tiles;
  const dim3 g((unsigned)(runs > 0 ? runs : 1)), b(256);
  if (fmt == DT_E4M3) TGG_LAUNCH(DT_E4M3);
  else if (fmt == DT_E5M2) TGG_LAUNCH(DT_E5M2);
  else return set_error("unsupported fp8 format code %d", fmt);
#undef TGG_LAUNCH
  return check_launch("trans_quant128");
}

int launch_token_cast128(const void* x, void* codes, float* scales, int64_t rows, int kblocks, int mn_major, int fmt,
                         hipStream_t s) {
  const int64_t groups = rows * kblocks;
  if (groups == 0) return 0;
  int64_t grid = ((mn_major ? ((rows + 15) / 16) * kblocks : (groups + 15) / 16) + 1) / 2;
  const int64_t cap = (int64_t)num_cus() * 32;
  if (grid > cap) grid = cap;
  if (fmt == DT_E4M3)
    hipLaunchKernelGGL(token_cast128_kernel<DT_E4M3>, dim3((unsigned)grid), dim3(256), 0, s, (const uint16_t*)x,
                       (uint8_t*)codes, scales, rows, kblocks, mn_major);
  else if (fmt == DT_E5M2)
    hipLaunchKernelGGL(token_cast128_kernel<DT_E5M2>, dim3((unsigned)grid), dim3(256), 0, s, (const uint16_t*)x,
                       (uint8_t*)codes, scales, rows, kblocks, mn_major);
  else
    return set_error("unsupported fp8 format code %d", fmt);
  return check_launch("token_cast128");
}

int launch_block_cast128(const void* x, void* codes, float* scales, int batch, int R, int C, int fmt, hipStream_t s) {
  const int64_t tiles = (int64_t)batch * ((R + 127) / 128) * ((C + 127) / 128);
  if (tiles == 0) return 0;
  int64_t grid = (int64_t)num_cus() * 8;
  if (grid > tiles) grid = tiles;
  if (fmt == DT_E4M3)
    hipLaunchKernelGGL(block_cast128_kernel<DT_E4M3>, dim3((unsigned)grid), dim3(256), 0, s, (const uint16_t*)x,
                       (uint8_t*)codes, scales, batch, R, C);
  else if (fmt == DT_E5M2)
    hipLaunchKernelGGL(block_cast128_kernel<DT_E5M2>, dim3((unsigned)grid), dim3(256), 0, s, (const uint16_t*)x,
                       (uint8_t*)codes, scales, batch, R, C);
  else
    return set_error("unsupported fp8 format code %d", fmt);
  return check_launch("block_cast128");
}

// Sum of the sizes, each taken as int32 and rounded up to block_m (floor division, also of negative ones), to host memory that the
// GPU writes over the bus: the total, then the word that says it is there.
__global__ __launch_bounds__(64) void padded_total_kernel(const void* sizes, int is64, int G, int64_t block_m, int64_t* host) {
  int64_t sum = 0;
  for (int g = threadIdx.x; g < G; g += 64) {
    const int64_t v = is64 ? (int64_t)(int32_t)((const int64_t*)sizes)[g] : (int64_t)((const int32_t*)sizes)[g];
    const int64_t up = v + block_m - 1;
    sum += (up >= 0 ? up / block_m : -((block_m - 1 - up) / block_m)) * block_m;
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) sum += __shfl_xor(sum, d, 64);
  if (threadIdx.x == 0) {
    __hip_atomic_store(host, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(host + 1, (int64_t)1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

int launch_padded_total(const void* sizes, int is64, int G, int64_t block_m, int64_t* host, hipStream_t s) {
  hipLaunchKernelGGL(padded_total_kernel, dim3(1), dim3(64), 0, s, sizes, is64, G, block_m, host);
  return check_launch("padded_total");
}

int launch_scales_transpose(const float* in, float* out, int64_t rows, int cols, hipStream_t s) {
  if (rows == 0 || cols == 0) return 0;
  hipLaunchKernelGGL(scales_transpose_kernel, dim3((unsigned)((rows + 63) / 64)), dim3(256), 0, s, in, out, rows, cols);
  return check_launch("scales_transpose");
}

int launch_cvt_fp8(const float* in, void* out, int64_t n, int fmt, hipStream_t s) {
  if (n == 0) return 0;
  const unsigned grid = (unsigned)((n + 255) / 256);
  if (fmt == DT_E4M3) hipLaunchKernelGGL(cvt_fp8_kernel<DT_E4M3>, dim3(grid), dim3(256), 0, s, in, (uint8_t*)out, n);
  else if (fmt == DT_E5M2) hipLaunchKernelGGL(cvt_fp8_kernel<DT_E5M2>, dim3(grid), dim3(256), 0, s, in, (uint8_t*)out, n);
  else return set_error("unsupported fp8 format code %d", fmt);
  return check_launch("cvt_fp8");
}

}  // namespace tgg
