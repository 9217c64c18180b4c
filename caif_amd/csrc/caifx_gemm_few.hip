// Forward dequant-GEMM whose tiles all run at once: a few dozen to some hundred activation rows, or more of a small weight,
// Y = X * W^T over int8 or packed int4 codes, 16-bit compute.
//
// A workgroup of eight waves owns up to 112 rows x 64 columns of Y.  The waves split the reduction, units of 128 (int4) or 64 (int8)
// elements in turn, and share nothing until their partial tiles are added at the end: no barrier and no staging through LDS in the
// loop, operands straight from memory in matrix-core order, every weight element dequantised once per row tile, by one lane.  Where
// the tiles do not fill the chip the reduction is shared among workgroups too, as in the tiled kernel (fp32 partial tiles in the
// workspace, a second launch adds them).
//
// Bound by the way of its loads: a wave's operands of X are asked for one to two half steps ahead, its codes a unit, and 48 to 60 % of the waves'
// time is waiting (counters: matrix cores 7 to 16 % busy, VALU 15 to 23 % of a wave's time, two waves a SIMD; a compute unit takes
// in 8 to 13 bytes a clock, its share of the codes and all rows of X along its share of the reduction).  The tiled kernel before it (128 x 128 tiles, 64-deep steps that eight waves pass through together) took 1.1 us a step
// however few of its rows were there.  Graph replay, before / now in us, bf16, int4 | int8 per channel | int8 with one scale:
//     N = K = 4096,          M = 33    15.7 / 15.1 | 19.4 / 13.3 | 29.1 / 12.1        M = 64   17.8 / 15.3 | 22.5 / 16.1 | 32.2 / 14.6
//     N = 11008, K = 4096,   M = 33    27.7 / 20.5 | 42.9 / 23.4 | 86.8 / 20.6        M = 100  (tiled)     | 45.3 / 39.4 | 98.3 / 37.3
//     N = K = 1024,          M = 200   12.7 / 8.1  | 14.1 / 10.1 | 27.4 / 9.1         M = 1024 16.8 / 10.8 | 18.0 / 12.5 | 31.5 / 11.1
//
//   * Lane (j, q) = (lane % 16, lane / 16) supplies reduction elements 32 h + 8 q .. + 7 of half step h of row j (X) or column j (W)
//     of a 16 x 16 tile: an instruction reads 64 contiguous bytes of sixteen rows of X.
//   * Operands of X are loaded a step ahead, each into registers whose operand has just been used; the weight operands of one half
//     step are formed while the other's products run.
//   * The operand is the reference's: code * scale in fp32, rounded once to the compute type.
#include "caifx_gemm_few_plan.hpp"
#include "caifx_internal.hpp"

#include <atomic>
#include <type_traits>

namespace caifx {
namespace {

constexpr int kCols = kFewCols, kWaves = kFewWaves;
constexpr int kScaleBytes = 64 * 1024;      // of a scale vector in LDS

struct FewArgs {
  int64_t M, N, K;
  const void *a;
  const void *wq;
  const void *scales;
  int group_shift;          // int4
  uint32_t period;          // int8: entries of the scale vector; 1 for one scale, 0 for none
  uint32_t row_len;         // the vector in LDS is cut into rows of gcd(K mod P, P) entries, 4 more apart: the runs of neighbouring
  uint32_t row_magic;       //   weight rows start whole rows apart; ceil(2^32 / row_len)
  void *d;                  // Y, or the partial tiles [parts][M][N] in fp32
  int d_dtype;
  const void *addend;       // optional [M, N] of d_dtype: d = T(float(T(acc)) + float(addend))
  FewPlan plan;
};

// Eight int4 codes (element j in nibble j) times one scale, rounded to CT: fma(code + 8, s, -8 s) rounds the exact product once.  The
// odd elements stay in the high nibbles of their bytes (16 (code + 8)) and meet s / 16 instead of a shift.
template <typename CT> __device__ __forceinline__ u32x4_t int4_operand(uint32_t p, float s)
{
  const float s16 = s * 0.0625f, m8 = s * -8.0f;
  p ^= 0x88888888u;
  const uint32_t lo = p & 0x0F0F0F0Fu, hi = p & 0xF0F0F0F0u;
  u32x4_t v;
  v[0] = pack2<CT>(__builtin_fmaf(ubyte0_f32(lo), s, m8), __builtin_fmaf(ubyte0_f32(hi), s16, m8));
  v[1] = pack2<CT>(__builtin_fmaf(ubyte1_f32(lo), s, m8), __builtin_fmaf(ubyte1_f32(hi), s16, m8));
  v[2] = pack2<CT>(__builtin_fmaf(ubyte2_f32(lo), s, m8), __builtin_fmaf(ubyte2_f32(hi), s16, m8));
  v[3] = pack2<CT>(__builtin_fmaf(ubyte3_f32(lo), s, m8), __builtin_fmaf(ubyte3_f32(hi), s16, m8));
  return v;
}

// A lane loads 16 neighbouring bytes of its weight row: the four lanes of a row (q) cover 64 of them, a unit of two steps of int4 or
// one of int8.  What it multiplies are the codes of reduction elements 32 h + 8 q .. + 7 for every half step h: of int4, dword q
// of lane h (a 4 x 4 transposition among the lanes of a row); of int8, the 8 bytes q % 2 of lane 2 h + q / 2.  Exchanging bits of
// the lane number with bits of the register number: v_permlane32_swap swaps the lanes' upper half of one register with the lower
// of the other, v_permlane16_swap the odd sixteens with the even ones.
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b)
{
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b)
{
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
template <int kKind> __device__ __forceinline__ void spread_codes(u32x4_t &v)
{
  uint32_t d[4] = {v[0], v[1], v[2], v[3]};
  if constexpr (kKind == FK_INT4) {
    swap32(d[0], d[2]);
    swap32(d[1], d[3]);
    swap16(d[0], d[1]);
    swap16(d[2], d[3]);
  } else {
    swap16(d[0], d[2]);
    swap16(d[1], d[3]);
    swap32(d[0], d[2]);
    swap32(d[1], d[3]);
  }
  v = u32x4_t{d[0], d[1], d[2], d[3]};
}

template <typename CT, int kKind, int NB>
__global__ __launch_bounds__(64 * kWaves, 2) void few_rows_gemm_kernel(FewArgs g)
{
  typedef typename Mfma32<CT>::vec_t vec_t;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, q = lane >> 4;
  // XCD x (workgroup id mod 8) takes the x-th contiguous eighth of the tiles, the row tiles of one piece of the weight side by side
  const int per_xcd = static_cast<int>(gridDim.x >> 3);
  const int pos = static_cast<int>(blockIdx.x & 7) * per_xcd + static_cast<int>(blockIdx.x >> 3);
  if (pos >= g.plan.row_tiles * g.plan.col_tiles * g.plan.parts) return;
  const int row_tile = pos % g.plan.row_tiles, part = pos / g.plan.row_tiles % g.plan.parts, col_tile = pos / g.plan.row_tiles / g.plan.parts;
  // the last row tile begins early enough to be a whole one; rows in front of `skip` are its predecessor's and not stored
  int64_t row0 = static_cast<int64_t>(row_tile) * g.plan.tile_rows;
  int skip = 0;
  if (row0 + g.plan.tile_rows > g.M && row_tile > 0) {
    skip = static_cast<int>(row0 + g.plan.tile_rows - g.M);
    row0 -= skip;
  }
  const int rows = static_cast<int>(g.M - row0 < g.plan.tile_rows ? g.M - row0 : g.plan.tile_rows);      // more than 16 (NB - 1)
  const int64_t col0 = static_cast<int64_t>(col_tile) * kCols;
  constexpr int kHalves = kKind == FK_INT4 ? 4 : 2, kUnit = 32 * kHalves;      // reduction elements of a unit
  const int units = static_cast<int>(g.K / kUnit);
  const int first = part * g.plan.part_units, end = first + g.plan.part_units < units ? first + g.plan.part_units : units;
  const int mine = first + wave < end ? (end - first - wave + kWaves - 1) / kWaves : 0;      // units first + wave + 8 t

  // rows and columns past the end are loaded from the last one and never stored
  uint32_t w_off[4], s_off[4], s_idx[4];
  const int last_row = 16 * (NB - 1) + j < rows ? 16 * (NB - 1) + j : rows - 1;
  const uint32_t a_off = static_cast<uint32_t>((row0 + (j < rows ? j : rows - 1)) * g.K * 2) + 16 * q;       // M K < 2^31 (host)
  const uint32_t a_last = static_cast<uint32_t>((row0 + last_row) * g.K * 2) + 16 * q;
  const uint32_t block_bytes = static_cast<uint32_t>(32 * g.K);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    int64_t n = col0 + 16 * c + j;
    if (n >= g.N) n = g.N - 1;
    w_off[c] = (static_cast<uint32_t>(n * g.K) >> (kKind == FK_INT4 ? 1 : 0)) + 16 * q;       // N K < 2^32 (host)
    s_off[c] = kKind == FK_INT4 ? (static_cast<uint32_t>(n * g.K) >> g.group_shift) * 2 : 0;
    s_idx[c] = kKind == FK_INT8 ? static_cast<uint32_t>((static_cast<uint64_t>(n * g.K) + 8 * q + static_cast<uint64_t>(first + wave) * kUnit) % g.period) : 0;
  }
  const char *a = static_cast<const char *>(g.a);
  const char *w = static_cast<const char *>(g.wq);
  const char *sc = static_cast<const char *>(g.scales);
  float one = 1.0f;
  if constexpr (kKind == FK_INT8_ONE) {
    if (g.period == 1) one = static_cast<const float *>(g.scales)[0];
  }
  const uint32_t advance = kKind == FK_INT8 ? kWaves * kUnit % g.period : 0;
  // entry i of the scale vector in LDS (i < 2^14, row_len >= 64: the product's upper half is the quotient)
  const auto scale_at = [&](uint32_t i) __attribute__((always_inline)) { return (i + 4 * __umulhi(i, g.row_magic)) * 4; };
  if constexpr (kKind == FK_INT8) {
    for (uint32_t i = 4 * threadIdx.x; i < g.period; i += 4 * 64 * kWaves)
      *reinterpret_cast<floatx4_t *>(smem + scale_at(i)) = *reinterpret_cast<const floatx4_t *>(static_cast<const float *>(g.scales) + i);
  }

  floatx4_t acc[NB][4];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[i][c] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};

  if constexpr (kKind == FK_INT8) __syncthreads();
  {
    // Loads of a unit that the wave does not have are dropped by the buffer's size, which is nothing then: the loop needs no last
    // round of its own, and no load sits behind a branch.
    const auto buffer = [&](const char *p, int64_t unit_bytes, int t) __attribute__((always_inline)) {
      const uint64_t at = uniform64(reinterpret_cast<uint64_t>(p) + static_cast<uint64_t>((first + wave + static_cast<int64_t>(kWaves) * t) * unit_bytes));
      return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(at), 0, __builtin_amdgcn_readfirstlane(t < mine ? -1 : 0), 0x00020000);
    };
    const auto load_a = [&](__amdgpu_buffer_rsrc_t from, int h, int i) __attribute__((always_inline)) {
      const uint32_t at = (i < NB - 1 ? a_off : a_last) + 64 * h;
      return __builtin_bit_cast(vec_t, __builtin_amdgcn_raw_buffer_load_b128(from, at, i < NB - 1 ? i * block_bytes : 0, 0));
    };
    struct Raw {
      u32x4_t p;
      f16_t s;               // int4: a unit lies inside a group
    };
    const auto load_w = [&](__amdgpu_buffer_rsrc_t from, int t, int c) __attribute__((always_inline)) {
      Raw r;
      r.p = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(from, w_off[c], 0, 0));
      if constexpr (kKind == FK_INT4) {
        const auto scales = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(sc), 0, __builtin_amdgcn_readfirstlane(t < mine ? -1 : 0), 0x00020000);
        const uint32_t group = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(((first + wave + kWaves * t) * kUnit) >> g.group_shift) * 2);
        r.s = __builtin_bit_cast(f16_t, static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(scales, s_off[c], group, 0)));
      }
      return r;
    };
    // the operand of half h of the unit that s_idx stands on
    const auto operand = [&](const Raw &r, int h, int c) __attribute__((always_inline)) {
      if constexpr (kKind == FK_INT4) {
        return int4_operand<CT>(r.p[h], to_f32(r.s));
      } else {
        floatx4_t s0 = {one, one, one, one}, s1 = s0;
        if constexpr (kKind == FK_INT8) {
          uint32_t i = s_idx[c] + 32 * h;
          if (i >= g.period) i -= g.period;
          const unsigned char *at = smem + scale_at(i);
          s0 = *reinterpret_cast<const floatx4_t *>(at);
          s1 = *reinterpret_cast<const floatx4_t *>(at + 16);
        }
        float lo[4], hi[4];
        int8x4_to_f32(r.p[2 * h], lo);
        int8x4_to_f32(r.p[2 * h + 1], hi);
        u32x4_t v;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          v[e] = pack2<CT>(lo[2 * e] * s0[2 * e], lo[2 * e + 1] * s0[2 * e + 1]);
          v[2 + e] = pack2<CT>(hi[2 * e] * s1[2 * e], hi[2 * e + 1] * s1[2 * e + 1]);
        }
        return v;
      }
    };
    const auto move_on = [&](int c) __attribute__((always_inline)) {
      if constexpr (kKind == FK_INT8) {
        s_idx[c] += advance;
        if (s_idx[c] >= g.period) s_idx[c] -= g.period;
      }
    };
    // what the registers hold: the operands of X of a step, codes a whole unit ahead or from the time on when the last operand of a
    // unit has been formed
    constexpr bool kAhead = NB < 5;
    vec_t af[NB][2];
    Raw cur[4], nxt[kAhead ? 4 : 1];
    u32x4_t b[2][4];
    auto a_now = buffer(a, kUnit * 2, 0), w_now = buffer(w, 64, 0);
#pragma unroll
    for (int c = 0; c < 4; ++c) cur[c] = load_w(w_now, 0, c);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) af[i][h] = load_a(a_now, h, i);
    if constexpr (kAhead) {
      w_now = buffer(w, 64, 1);
#pragma unroll
      for (int c = 0; c < 4; ++c) nxt[c] = load_w(w_now, 1, c);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      spread_codes<kKind>(cur[c].p);
      b[0][c] = operand(cur[c], 0, c);
    }
    // unit t: on entry its codes are spread, the weight operands of its first half formed, and the codes of unit t + 1 (kAhead) there
    // or on their way; beside the products of a half the operands of the next one are formed
    for (int t = 0; t < mine; ++t) {
      a_now = buffer(a, kUnit * 2, t);
      const auto a_next = buffer(a, kUnit * 2, t + 1);
      w_now = buffer(w, 64, t + (kAhead ? 2 : 1));
#pragma unroll
      for (int h = 0; h < kHalves; ++h) {
        asm volatile("s_nop 1");           // a matrix instruction reads what the VALU wrote two wait states ago at the earliest
#pragma unroll
        for (int i = 0; i < NB; ++i) {
#pragma unroll
          for (int c = 0; c < 4; ++c) mfma16<CT>(acc[i][c], af[i][h & 1], __builtin_bit_cast(vec_t, b[h & 1][c]));
          // both halves of a row's next 128 bytes, together
          if (h & 1) {
#pragma unroll
            for (int x = 1; x <= 2; ++x) af[i][(h + x) & 1] = h + x < kHalves ? load_a(a_now, h + x, i) : load_a(a_next, h + x - kHalves, i);
          }
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (c * NB / 4 == i) {
              if (h + 1 < kHalves) {
                b[(h + 1) & 1][c] = operand(cur[c], h + 1, c);
                if (!kAhead && h + 2 == kHalves) cur[c] = load_w(w_now, t + 1, c);
              } else {
                move_on(c);
                if (kAhead) cur[c] = nxt[kAhead ? c : 0];
                spread_codes<kKind>(cur[c].p);
                b[0][c] = operand(cur[c], 0, c);
                if (kAhead) nxt[kAhead ? c : 0] = load_w(w_now, t + 2, c);
              }
            }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    // the last products have to leave the pipe before their registers are read (the compiler does not see the asm's latency)
    asm volatile("s_nop 15\n\ts_nop 15");
  }

  // the waves' partial tiles: 4 .. 7 onto 0 .. 3, then the four, in a fixed order
  if constexpr (kKind == FK_INT8) __syncthreads();           // the scales have been read
  floatx4_t *red = reinterpret_cast<floatx4_t *>(smem);      // [4][NB * 4][64]
  if (wave >= 4) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) red[((wave - 4) * NB * 4 + i * 4 + c) * 64 + lane] = acc[i][c];
  }
  __syncthreads();
  if (wave < 4) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        floatx4_t &slot = red[(wave * NB * 4 + i * 4 + c) * 64 + lane];
        slot = acc[i][c] + slot;
      }
  }
  __syncthreads();
  constexpr int kPieces = (NB * 256 + 511) / 512;
  floatx4_t sum[kPieces];
#pragma unroll
  for (int x = 0; x < kPieces; ++x) {
    const int at = static_cast<int>(threadIdx.x) + 512 * x;
    if (at >= NB * 256) continue;
    sum[x] = red[at] + red[NB * 256 + at];
    sum[x] += red[2 * NB * 256 + at];
    sum[x] += red[3 * NB * 256 + at];
  }
  __syncthreads();
  constexpr int kPitch = kCols * 4 + 16;                     // a row of the tile in fp32
#pragma unroll
  for (int x = 0; x < kPieces; ++x) {
    const int at = static_cast<int>(threadIdx.x) + 512 * x;
    if (at >= NB * 256) continue;
    const int tile = at >> 6, l = at & 63;                   // tile = 4 i + c
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<float *>(smem + (16 * (tile >> 2) + 4 * (l >> 4) + r) * kPitch + (16 * (tile & 3) + (l & 15)) * 4) = sum[x][r];
  }
  __syncthreads();
  const auto store = [&](auto type_) __attribute__((always_inline)) {
    typedef decltype(type_) T;
    constexpr int kPer = 16 / sizeof(T), kLanes = kCols / kPer;
    T *d = static_cast<T *>(g.d);
    if constexpr (sizeof(T) == 4) d += static_cast<int64_t>(part) * g.M * g.N;      // (parts are in fp32)
    const T *ap = static_cast<const T *>(g.addend);
    const int64_t col = col0 + (threadIdx.x % kLanes) * kPer;
    if (col >= g.N) return;                                  // N is a multiple of 8
    for (int r = threadIdx.x / kLanes; r < rows; r += 64 * kWaves / kLanes) {
      const float *src = reinterpret_cast<const float *>(smem + r * kPitch + (threadIdx.x % kLanes) * kPer * 4);
      const int64_t o = (row0 + r) * g.N + col;
      u32x4_t v;
      T *vp = reinterpret_cast<T *>(&v);
#pragma unroll
      for (int e = 0; e < kPer; ++e) vp[e] = from_f32<T>(src[e]);
      if (r < skip) continue;
      if (ap) {
        const u32x4_t av = *reinterpret_cast<const u32x4_t *>(ap + o);
        const T *aq = reinterpret_cast<const T *>(&av);
#pragma unroll
        for (int e = 0; e < kPer; ++e) vp[e] = from_f32<T>(to_f32<T>(vp[e]) + to_f32<T>(aq[e]));
      }
      *reinterpret_cast<u32x4_t *>(d + o) = v;
    }
  };
  if (g.d_dtype == CAIFX_F32) store(float{});
  else if (g.d_dtype == CAIFX_BF16) store(bf16_t{});
  else store(f16_t{});
}

template <typename CT, int kKind, int NB> int launch(const FewArgs &g, hipStream_t s)
{
  // partial tiles, or the scale vector (the tile in fp32 rows is smaller)
  constexpr int kLds = kKind == FK_INT8 && 4 * NB * 4096 < kScaleBytes ? kScaleBytes : 4 * NB * 4096;
  auto kern = few_rows_gemm_kernel<CT, kKind, NB>;
  static std::atomic<bool> raised{false};
  if (!raised.load(std::memory_order_relaxed)) {
    // the attribute is per kernel and sticky; two threads racing here both set it, which is harmless
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return CAIFX_ERR_LAUNCH_FAILED;
    raised.store(true, std::memory_order_relaxed);
  }
  const unsigned tiles = static_cast<unsigned>(g.plan.row_tiles * g.plan.col_tiles * g.plan.parts);
  hipLaunchKernelGGL(kern, dim3((tiles + 7) / 8 * 8), dim3(64 * kWaves), kLds, s, g);
  return launch_status();
}
template <typename CT, int kKind> int pick_rows(const FewArgs &g, hipStream_t s)
{
  switch ((g.plan.tile_rows + 15) / 16) {
    case 2: return launch<CT, kKind, 2>(g, s);
    case 3: return launch<CT, kKind, 3>(g, s);
    case 4: return launch<CT, kKind, 4>(g, s);
    case 5: return launch<CT, kKind, 5>(g, s);
    case 6: return launch<CT, kKind, 6>(g, s);
    default: return launch<CT, kKind, 7>(g, s);
  }
}
template <typename CT> int pick_kind(const FewArgs &g, int kind, hipStream_t s)
{
  if (kind == FK_INT4) return pick_rows<CT, FK_INT4>(g, s);
  return kind == FK_INT8 ? pick_rows<CT, FK_INT8>(g, s) : pick_rows<CT, FK_INT8_ONE>(g, s);
}

}  // namespace

int mfma_few_forward(const GemmArgs &a, hipStream_t s)
{
  if (a.offsets || a.epilogue != 0 || a.compute_dtype == CAIFX_F32 || a.x_dtype != a.compute_dtype) return CAIFX_ERR_UNSUPPORTED;
  FewArgs g{};
  if (!aligned_to(a.x, 16) || !aligned_to(a.y, 16) || !aligned_to(a.w.q, 16) || (a.addend && !aligned_to(a.addend, 16))) return CAIFX_ERR_UNSUPPORTED;
  int kind;
  if (a.w.kind == CAIFX_W_INT4_GROUP) {
    const int gs = a.w.group_size;
    if (gs < 128 || (gs & (gs - 1)) != 0 || a.K % gs != 0) return CAIFX_ERR_UNSUPPORTED;
    g.group_shift = __builtin_ctz(static_cast<unsigned>(gs));
    kind = FK_INT4;
  } else if (a.w.kind == CAIFX_W_INT8) {
    const int64_t P = a.w.scales ? a.w.scale_period : 0;
    kind = P <= 1 ? FK_INT8_ONE : FK_INT8;
    if (kind == FK_INT8) {
      if (P % 64 != 0 || P > 15872 || !aligned_to(a.w.scales, 16)) return CAIFX_ERR_UNSUPPORTED;
      int64_t len = P;                                       // a multiple of 64, as K and P are: at most 248 skips of 16 bytes
      for (int64_t r = a.K % P; r != 0;) {
        const int64_t t2 = len % r;
        len = r;
        r = t2;
      }
      if ((P + 4 * (P / len)) * 4 > kScaleBytes) return CAIFX_ERR_UNSUPPORTED;
      g.row_len = static_cast<uint32_t>(len);
      g.row_magic = static_cast<uint32_t>(((uint64_t{1} << 32) + len - 1) / len);
    }
    g.period = static_cast<uint32_t>(P);
  } else {
    return CAIFX_ERR_UNSUPPORTED;
  }
  g.plan = plan_few(a.M, a.N, a.K, kind);
  if (g.plan.parts == 0) return CAIFX_ERR_UNSUPPORTED;
  g.M = a.M;
  g.N = a.N;
  g.K = a.K;
  g.a = a.x;
  g.wq = a.w.q;
  g.scales = a.w.scales;
  g.d = a.y;
  g.d_dtype = a.y_dtype;
  g.addend = a.addend;
  const bool split = g.plan.parts > 1;
  if (split) {
    // no more than the tiled kernel's parts ask for: its tiles are as high or higher and twice as wide
    if (!a.workspace || a.workspace_bytes < static_cast<size_t>(g.plan.parts) * static_cast<size_t>(a.M) * static_cast<size_t>(a.N) * 4 || !aligned_to(a.workspace, 16))
      return CAIFX_ERR_UNSUPPORTED;
    g.d = a.workspace;
    g.d_dtype = CAIFX_F32;
    g.addend = nullptr;
  }
  const int st = a.compute_dtype == CAIFX_BF16 ? pick_kind<bf16_t>(g, kind, s) : pick_kind<f16_t>(g, kind, s);
  if (!split || st != CAIFX_OK) return st;
  return splitk_reduce(static_cast<const float *>(a.workspace), g.plan.parts, a.M * a.N, a.y, a.y_dtype, a.addend, s);
}

}  // namespace caifx
