// Grouped dequant-GEMM over token-sorted expert segments, forward and input gradient, int8 codes with a scale vector, and the forward
// with one weight where its tiles are one round: tall tiles whose weight columns never meet in LDS as operands.
//
// A workgroup of eight waves owns up to 256 rows x 256 columns of an expert's result; wave w owns columns [32 w, 32 w + 32) for
// all of the rows and walks the reduction in steps of 64.
//
// Why these tiles: dequantising inside the product costs 160 VALU instructions of four clocks per step and SIMD for 256 columns,
// whatever the rows, besides a round of LDS traffic and two meetings of the waves: 0.5 us a step.  In 128-row tiles (eight waves x
// 32 columns, caifx_gemm_regw8.hip; caifx_gemm_tile.hpp for the gradient) a segment of 384 rows pays it three to four times, here
// twice.  Timed with parts left out (192 rows, 2048-deep, us a step): matrix instructions and meetings 0.70, the requests 0.2 to
// 0.3 more, operand reads 0.1, dequantisation 0.2 to 0.35: 1.2 in all, issue of the two waves of a SIMD being what most of it
// has in common (a wave alone issues a VALU instruction every eight clocks: four waves of 64 columns are no faster).
// 64 experts, 24576 rows, 1408 x 2048 and 2048 x 1408, bf16, us, before (those two kernels) / now: forward 263 / 189 and 226 / 169,
// gradient 290 / 166 and 242 / 155, 0.75 to 0.91 PFLOP/s.
//   * Row tiles: a segment is cut into tiles of equal height (a multiple of 32), so 384 rows make two of 192 and not one of
//     256 and one of 128 that costs as much dequantisation.  The reduction loop is instantiated for 64, 96, .. 256 rows.
//   * The weight: every wave dequantises the 64 x 32 piece of its own columns for the next step in registers, float(code) *
//     scale in fp32, one rounding to the compute type (the reference's dequantise-then-cast weight, bit for bit), spread
//     over the step's matrix instructions.
//   * Lane (j, q) = (lane % 16, lane / 16) supplies the operands of reduction elements 16 q + 8 kk .. + 7 of a step (kk = 0, 1),
//     a permutation of the step's 64 that both operands follow, so a lane's codes of one column are 16 neighbours.
//   * Forward: lane j's column of column tile c is weight row 16 c + j of the wave's 32.  Codes arrive by requests of 8 rows x
//     128 bytes (two steps) into a ring of eight 1 KiB slots that only this wave reads.  Scales: the reference addresses a
//     vector of P entries by the flat index (n K + k) mod P; weight rows equal modulo V = P / gcd(K mod P, P) see the same
//     scales along k, so a step needs V runs of 64 of them: they travel by requests too, into a ring of three steps.
//   * Input gradient: the columns are k, the reduction runs down the weight rows, and lane j's column of column tile c is
//     2 j + c of the wave's 32, so the codes of its two columns in a row are one 16-bit read and their scales one of 8 bytes.
//     No transposition anywhere.  Codes: 64 rows x 256 bytes per step into a ring of three.  Scales: V + 15 rows of 256
//     (16 neighbouring weight rows from any class on, without wrapping), fetched once per tile.
//   * Activations: four half tiles (half of the rows, one step) in LDS, three of them on their way; the waves meet twice per
//     step, when a half has been read by all.  Requests complete in issue order, so every wait is an exact count.
// Tiles are numbered expert by expert, row tile by row tile, column tile last, a contiguous eighth of the list per XCD.
#pragma once

#include "caifx_gemm_regw.hpp"
#include "caifx_gemm_tall_plan.hpp"

#include <atomic>
#include <type_traits>
#include <utility>

namespace caifx {
namespace tall {

typedef __attribute__((__vector_size__(2 * sizeof(float)))) float floatx2_t;

constexpr int BM = kTallRows, BN = kTallCols;
constexpr int kWaves = 8, kCols = 32;         // columns of a wave: two column tiles of 16
constexpr int kHalf = 16 * 1024;             // LDS of half an activation tile: 128 rows of 128 bytes
constexpr int kCodes = 4 * kHalf;            // codes: forward 8 waves x 8 KiB, gradient 3 steps x 16 KiB
constexpr int kScalesFwd = kCodes + 64 * 1024;
constexpr int kScalesBwd = kCodes + 48 * 1024;
constexpr int kMaxClasses = 32;              // V
constexpr int kLdsMax = 160 * 1024;

struct TallArgs {
  int64_t M, N, K;           // rows of the buffer (an upper bound of the segments'), weight [N, K]
  const void *a;             // [M, R] in the compute type
  void *d;                   // [M, C]
  int d_dtype;
  const void *addend;        // optional [M, C] of d_dtype: d = T(float(T(acc)) + float(addend))
  int epilogue;              // gated experts, see EPI_* in caifx_gemm_tile.hpp: 1 forward (e1 = gate), 2 backward (and e2 = up)
  const void *e1, *e2;
  void *d2;
  const int32_t *offsets;    // null: one weight (wq, scales) for all M rows
  const void *wq, *scales;
  const void *const *wq_ptrs;
  const void *const *scales_ptrs;
  int num_experts;
  int height;                // of a row tile at most, a multiple of 32 up to 256
  bool zero_rest;            // rows that no segment covers are to be zero
  uint32_t period;           // entries of a scale vector
  int classes;               // V
  unsigned long long *stamps;      // measurement only, see mfma_grouped_tile_stamps
  long long stamps_capacity;
};

template <int... I, typename F> __device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F f)
{
  (f(std::integral_constant<int, I>{}), ...);
}
template <int kN, typename F> __device__ __forceinline__ void repeat(F f) { each_of(std::make_integer_sequence<int, kN>{}, f); }

// signed byte kByte of a dword as fp32, in one instruction (from the C expression the compiler makes two for some of the bytes)
template <int kByte> __device__ __forceinline__ float code_f32(uint32_t p)
{
  float r;
  if constexpr (kByte == 0) asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(r) : "v"(p));
  if constexpr (kByte == 1) asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(r) : "v"(p));
  if constexpr (kByte == 2) asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(r) : "v"(p));
  if constexpr (kByte == 3) asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(r) : "v"(p));
  return r;
}

__device__ __forceinline__ void request16(uint32_t dst, uint32_t voff, uint64_t src)
{
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(voff), "s"(src) : "memory");
}

// the same by the first kLanes lanes only (every lane of the wave has to be active)
template <int kLanes> __device__ __forceinline__ void request16_by(uint32_t dst, uint32_t voff, uint64_t src)
{
  if constexpr (kLanes == 64)
    request16(dst, voff, src);
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_bfm_b64 exec, %3, 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1" ::"s"(dst), "v"(voff), "s"(src), "n"(kLanes) : "memory");
}

// The tile of a product with one weight: row tiles of equal height, those of a column tile side by side, so that a piece of the weight
// comes into one L2.
__device__ __forceinline__ bool plain_tile(const TallArgs &g, int64_t col_tiles, GroupedTile &out)
{
  const int64_t row_tiles = (g.M + g.height - 1) / g.height, total = row_tiles * col_tiles, per_xcd = (total + 7) >> 3;
  const int64_t slot = blockIdx.x >> 3, pos = static_cast<int64_t>(blockIdx.x & 7) * per_xcd + slot;
  if (slot >= per_xcd || pos >= total) return false;
  out.e = 0;
  out.pos = pos;
  out.col_tile = pos / row_tiles;
  grouped_rows<BM, true>(0, static_cast<int>(g.M), static_cast<int>(row_tiles), static_cast<int>(pos - out.col_tile * row_tiles), out);
  out.wq = g.wq;
  out.scales = g.scales;
  return out.row0 < out.row_end;
}

template <typename CT, bool kBackward>
__global__ __launch_bounds__(64 * kWaves, 2) void tall_gemm_kernel(TallArgs g)
{
  typedef typename Mfma32<CT>::vec_t vec_t;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, q = lane >> 4;
  const int64_t C = kBackward ? g.K : g.N, R = kBackward ? g.N : g.K;

  GroupedTile gt;
  const bool has_tile = !kBackward && !g.offsets ? plain_tile(g, (C + BN - 1) / BN, gt) : grouped_tile<BM, true>(g.offsets, g.num_experts, g.M, (C + BN - 1) / BN, g.wq_ptrs, g.scales_ptrs, lane, gt, g.height);
  if (g.zero_rest) zero_uncovered(g.offsets, g.num_experts, g.M, gt.first, gt.end, gt.ordered, g.d, C * (g.d_dtype == CAIFX_F32 ? 4 : 2));
  if (!has_tile) return;
  // the search's results are the same in every lane: into scalar registers with them
  const int64_t row0 = uniform64(static_cast<uint64_t>(gt.row0)), row_end = uniform64(static_cast<uint64_t>(gt.row_end));
  const int64_t col0 = uniform64(static_cast<uint64_t>(gt.col_tile * BN));
  const int rows = static_cast<int>(row_end - row0);
  const uint64_t wq = uniform64(reinterpret_cast<uint64_t>(gt.wq)), scales = uniform64(reinterpret_cast<uint64_t>(gt.scales));
  int64_t stamp_pos = -1;
  if (g.stamps && threadIdx.x == 0 && gt.pos < g.stamps_capacity) {
    stamp_pos = gt.pos;
    g.stamps[4 * stamp_pos] = static_cast<unsigned long long>(gt.e);
    g.stamps[4 * stamp_pos + 1] = static_cast<unsigned long long>(rows) | (1ull << 32);      // one workgroup per compute unit
    g.stamps[4 * stamp_pos + 2] = wall_clock64();
  }

  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  const uint64_t a_base = uniform64(reinterpret_cast<uint64_t>(g.a) + static_cast<uint64_t>(row0 * R * 2));
  const int steps = static_cast<int>(R / 64), last = steps - 1;
  const uint32_t period = g.period;
  const uint32_t V = static_cast<uint32_t>(g.classes);

  // ---- requests for codes.  Positions of 16-byte pieces are permuted so that the reads below spread over the banks
  uint64_t w_base;
  uint32_t w_voff[2];
  if constexpr (!kBackward) {
    // request rg of a block of 128 k: rows 8 rg .. + 7 of the wave's 32 (N is a multiple of 32; a wave beyond N asks for nothing)
    int64_t n0 = col0 + kCols * wave;
    if (n0 > g.N - kCols) n0 = g.N - kCols;
    w_base = wq + static_cast<uint64_t>(n0 * g.K);
    w_voff[0] = static_cast<uint32_t>((lane >> 3) * g.K) + 16 * ((lane & 7) ^ (lane >> 3));
  } else {
    // request i of a step: rows 32 i + 4 wave .. + 3, 256 columns
    w_base = wq;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      int64_t col = col0 + 16 * ((lane & 15) ^ (4 * (2 * i + (wave >> 2))));
      if (col > g.K - 16) col = g.K - 16;              // columns past the end: loaded, never stored
      w_voff[i] = static_cast<uint32_t>((4 * wave + (lane >> 4)) * g.K + col);
    }
  }
  const uint32_t row_bytes = static_cast<uint32_t>(g.K);

  // ---- scales
  // Forward, a step's table: 32 rows, row m the scales of class m mod V.  Up to 17 classes a lane reads row (first of its column
  // tile) + j, so the sixteen rows of one pass of the LDS are neighbours; it is laid out [q][row][16-byte piece e ^ row / 4],
  // which puts sixteen neighbours into sixteen different bank groups whatever their q (a pass mixes lanes of two q).
  uint32_t s_idx = 0;                    // flat index modulo P of what the lane asks for next
  int s_off[2][4];                       // LDS offset of scales 4 e .. + 3 of the lane's 16, column tile c
  if constexpr (!kBackward) {
    const uint32_t m = 16 * (wave & 1) + (lane >> 2);
    const uint32_t k = 16 * (wave >> 1) + 4 * ((lane ^ (m >> 2)) & 3);
    s_idx = ((m % V) * static_cast<uint32_t>(g.K) + k) % period;
    const uint32_t n0 = static_cast<uint32_t>(col0 + kCols * wave);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int row = V <= 17 ? static_cast<int>((n0 + 16 * c) % V) + j : static_cast<int>((n0 + 16 * c + j) % V);
#pragma unroll
      for (int e = 0; e < 4; ++e) s_off[c][e] = kScalesFwd + q * 2048 + row * 64 + ((e ^ (row >> 2)) & 3) * 16;
    }
  }

  constexpr int kPitch = BN * 2 + 32;      // LDS rows of the staged store (16-bit results): row + 32 bytes
  // the reduction over NB row tiles of 16; kIdle: the wave's columns lie beyond C, it only moves its share and meets the others
  auto run = [&](auto nb_, auto idle_) __attribute__((always_inline)) {
    constexpr int NB = decltype(nb_)::value;
    constexpr bool kIdle = decltype(idle_)::value;
    constexpr int kFull = NB / 8, kRest = NB % 8;      // activation requests of a wave per half: kFull of 8 rows, one of kRest
    constexpr int kReq = kFull + (kRest ? 1 : 0);
    constexpr int T = 4 * NB;                          // matrix instructions of a step: [half][kk][row tile][column tile]
    constexpr int kOwn = !kBackward && !kIdle ? 1 : 0; // forward: code requests per meeting, the wave's own
    constexpr int kFirst = kBackward ? 2 : 1;          // requests for all behind the first meeting: codes (gradient) or scales
    constexpr int kWait = 2 * kReq + 2 * kOwn + kFirst;

    uint32_t a_voff[2][kReq];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int x = 0; x < kReq; ++x) {
        const int lrow = 64 * x + (x < kFull ? 8 : kRest) * wave + (lane >> 3);
        int m = h * 8 * NB + lrow;
        if (m >= rows) m = rows - 1;                   // rows past the end are loaded from the last row and never stored
        a_voff[h][x] = static_cast<uint32_t>(m) * static_cast<uint32_t>(R * 2) + (((lane & 7) ^ ((lrow ^ (lrow >> 3)) & 7)) << 4);
      }
    auto request_a = [&](int s, int h, auto x_) __attribute__((always_inline)) {
      constexpr int x = decltype(x_)::value;
      const uint32_t k0 = static_cast<uint32_t>(s < last ? s : last) * 128;          // past the end: the last step again
      const uint32_t dst = lds0 + (2 * (s & 1) + h) * kHalf + (64 * x + (x < kFull ? 8 : kRest) * wave) * 128;
      request16_by<x < kFull ? 64 : 8 * kRest>(dst, a_voff[h][x], a_base + k0);
    };
    // forward: request rg (0 .. 3) of block b; gradient: request i (0, 1) of step b into slot
    auto request_codes = [&](int b, int slot, int i) __attribute__((always_inline)) {
      if constexpr (!kBackward) {
        const uint32_t blk = static_cast<uint32_t>(b < (last >> 1) ? b : (last >> 1));
        request16(lds0 + kCodes + wave * 8192 + (b & 1) * 4096 + i * 1024, w_voff[0], w_base + 128 * blk + static_cast<uint64_t>(8 * i) * row_bytes);
      } else {
        const uint32_t n0 = static_cast<uint32_t>(b < last ? b : last) * 64 + 32 * i;
        request16(lds0 + kCodes + slot * 16384 + (wave + 8 * i) * 1024, w_voff[i], w_base + static_cast<uint64_t>(n0) * row_bytes);
      }
    };
    auto request_scales = [&](int slot) __attribute__((always_inline)) {
      if constexpr (!kBackward) {
        request16(lds0 + kScalesFwd + slot * 8192 + wave * 1024, s_idx * 4, scales);
        s_idx += 64;
        if (s_idx >= period) s_idx -= period;
      }
    };
    auto request_half = [&](int s, int h) __attribute__((always_inline)) {
      repeat<kReq>([&](auto x_) __attribute__((always_inline)) { request_a(s, h, x_); });
    };

    floatx4_t acc[NB][2];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c) acc[i][c] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // ---- in front of the first step
    if constexpr (kBackward) {
      // the table's rows: row m holds the scales of weight rows n = m mod V, columns col0 ..
      const int per_wave = (static_cast<int>(V) + 15 + kWaves - 1) / kWaves;
      for (int i = 0; i < per_wave; ++i) {
        const uint32_t m = wave + kWaves * i;
        const uint32_t idx = ((m % V) * static_cast<uint32_t>(g.K) + static_cast<uint32_t>(col0) + 4 * lane) % period;
        request16(lds0 + kScalesBwd + m * 1024, idx * 4, scales);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) request_codes(i >> 1, i >> 1, i & 1);
      request_half(0, 0);
      request_half(0, 1);
      request_half(1, 0);
      request_codes(2, 2, 0);
      request_codes(2, 2, 1);
      request_half(1, 1);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * kReq + 2) : "memory");
    } else {
      request_scales(0);
      request_scales(1);
      if constexpr (!kIdle) {
#pragma unroll
        for (int i = 0; i < 4; ++i) request_codes(0, 0, i);
      }
      request_half(0, 0);
      request_half(0, 1);
      if constexpr (!kIdle) {
        request_codes(1, 0, 0);
        request_codes(1, 0, 1);
      }
      request_half(1, 0);
      if constexpr (!kIdle) request_codes(1, 0, 2);
      request_scales(2);
      request_half(1, 1);
      if constexpr (!kIdle) request_codes(1, 0, 3);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * kReq + 4 * kOwn + 1) : "memory");
    }

    // ---- operand reads
    int a_addr[4][2];              // row tile il of a half: a_addr[il % 4] + 2048 il (the swizzle repeats every four)
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) a_addr[x][kk] = j * 128 + (((2 * q + kk) ^ ((j ^ (j >> 3) ^ (2 * x)) & 7)) << 4);
    vec_t fr[8];
    u32x4_t b[2][2][2];            // [parity of the step][column tile][kk]
    // what a lane has read of codes and scales and not yet multiplied: forward a column tile, gradient two weight rows (twice)
    u32x4_t code;
    floatx4_t sc[4];
    uint32_t cw[2][2];
    floatx2_t sr[2][2];
    // of the step that is dequantised next: slot of the rings of three, position in the class rows
    int slot3 = 1, slot3n = 2;
    uint32_t mq = 0, mqn = 0;
    const uint32_t m_step = kBackward ? 64 % V : 0;
    int c_lane = 0;
    if constexpr (kBackward) {
      mq = (16 * q + 64) % V;
      mqn = (16 * q + 128) % V;
      c_lane = kCodes + q * 4096 + (((2 * wave + (j >> 3)) ^ (4 * q)) << 4) + (j & 7) * 2;
    } else {
      c_lane = kCodes + wave * 8192 + (j >> 3) * 1024 + (j & 7) * 128 + ((q ^ (j & 7)) << 4);
    }
    // read x (0 .. 4; gradient 0 .. 3) of unit u of step t: forward unit = column tile, gradient unit = rows 2 u, 2 u + 1 of
    // every 16; `half` = t % 2, slot and m the step's ring slot and class
    constexpr int kUnits = kBackward ? 8 : 2, kReads = kBackward ? 4 : 5;
    auto read_raw = [&](auto half_, auto u_, auto x_, int t, int slot, uint32_t m) __attribute__((always_inline)) {
      constexpr int half = decltype(half_)::value, u = decltype(u_)::value, x = decltype(x_)::value;
      if constexpr (!kBackward) {
        if constexpr (x == 0) {
          const int at = (c_lane ^ (half * 64)) + ((t >> 1) & 1) * 4096;
          code = *reinterpret_cast<const u32x4_t *>(smem + at + u * 2048);
        } else {
          sc[x - 1] = *reinterpret_cast<const floatx4_t *>(smem + s_off[u][x - 1] + slot * 8192);
        }
      } else {
        constexpr int row = 2 * u + (x & 1);
        if constexpr (x < 2)
          cw[u & 1][x] = *reinterpret_cast<const uint16_t *>(smem + c_lane + slot * 16384 + row * 256);
        else
          sr[u & 1][x - 2] = *reinterpret_cast<const floatx2_t *>(smem + kScalesBwd + static_cast<int>(m) * 1024 + wave * 128 + j * 8 + row * 1024);
      }
    };
    auto read_unit = [&](auto half_, auto u_, int t, int slot, uint32_t m) __attribute__((always_inline)) {
      repeat<kReads>([&](auto x_) __attribute__((always_inline)) { read_raw(half_, u_, x_, t, slot, m); });
    };
    // dword d (0 .. 15) of the next operands in three parts: conversions, products, rounding
    float f0 = 0.0f, f1 = 0.0f;
    auto dequant = [&](auto part_, auto d_, u32x4_t(&to)[2][2]) __attribute__((always_inline)) {
      constexpr int part = decltype(part_)::value, d = decltype(d_)::value;
      constexpr int c = kBackward ? d & 1 : d >> 3;
      constexpr int kk = kBackward ? d >> 3 : (d >> 2) & 1;
      constexpr int p = kBackward ? (d >> 1) & 3 : d & 3;
      constexpr int buf = (d >> 1) & 1;                // gradient
      constexpr int e = 2 * kk + (p >> 1), o = 2 * (p & 1);
      if constexpr (part == 0) {
        f0 = kBackward ? code_f32<c>(cw[buf][0]) : code_f32<o>(code[e]);
        f1 = kBackward ? code_f32<c>(cw[buf][1]) : code_f32<o + 1>(code[e]);
      } else if constexpr (part == 1) {
        f0 *= kBackward ? sr[buf][0][c] : sc[e][o];
        f1 *= kBackward ? sr[buf][1][c] : sc[e][o + 1];
      } else {
        to[c][kk][p] = pack2<CT>(f0, f1);
      }
    };
    auto meet = [&]() __attribute__((always_inline)) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kWait) : "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    // fragment f = kk NB / 2 + row tile of half h of a step of parity par; buffer by its place in the order of use
    auto read_frag = [&](auto par_, auto h_, auto f_) __attribute__((always_inline)) {
      constexpr int par = decltype(par_)::value, h = decltype(h_)::value, f = decltype(f_)::value;
      constexpr int il = f % (NB / 2), kk = f / (NB / 2);
      fr[(par * 2 * NB + h * NB + f) & 7] = *reinterpret_cast<const vec_t *>(smem + a_addr[il & 3][kk] + (2 * par + h) * kHalf + il * 2048);
    };
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, 1> I1;

    if constexpr (!kIdle) {
      // step 0's operands; the first unit of step 1 and the first four fragments on their way
      uint32_t m0 = 0;
      if constexpr (kBackward) m0 = (16 * q) % V;
      repeat<kUnits>([&](auto u_) __attribute__((always_inline)) {
        read_unit(I0{}, u_, 0, 0, m0);
        constexpr int u = decltype(u_)::value, per = 16 / kUnits;
        repeat<per>([&](auto i_) __attribute__((always_inline)) {
          typedef std::integral_constant<int, u * per + decltype(i_)::value> D;
          dequant(I0{}, D{}, b[0]);
          dequant(I1{}, D{}, b[0]);
          dequant(std::integral_constant<int, 2>{}, D{}, b[0]);
        });
      });
      read_unit(I1{}, I0{}, 1, slot3, mq);
      repeat<4>([&](auto f_) __attribute__((always_inline)) { read_frag(I0{}, I0{}, f_); });
      __builtin_amdgcn_sched_barrier(0);
    }

    // Step s: its matrix instructions in groups of two (one fragment, two column tiles), and beside them the step after it:
    //  - dequantisation of step s + 1.  Gradient: evenly over the step, codes and scales read one unit (two rows) ahead.
    //    Forward: a column tile per half, its codes and scales read behind the meeting in front of it.
    //  - fragments four groups ahead; two groups in front of a meeting none are read, so that waiting for the own reads
    //    costs little there, and behind it two per group make up for that
    //  - behind the meeting in half h: requests for half h of step s + 2 (that half has been read by all), and codes and
    //    scales.  Forward: block b's code requests start behind the first meeting of step 2 b - 4, one per meeting; the
    //    slots they overwrite were read behind the meeting before at the latest.  Codes and scales of a column tile are first
    //    read behind a meeting that waits for them.
    auto step = [&](auto par_, int s) __attribute__((always_inline)) {
      constexpr int par = decltype(par_)::value;
      typedef std::integral_constant<int, par> Par;
      typedef std::integral_constant<int, par ^ 1> Next;
      const int slot3f = 3 - slot3 - slot3n;           // of step s + 3 (and s)
      auto requests = [&](auto h_, auto i_) __attribute__((always_inline)) {
        constexpr int h = decltype(h_)::value, i = decltype(i_)::value;
        if constexpr (i < kReq) {
          request_a(s + 2, h, i_);
        } else if constexpr (kBackward) {
          if constexpr (h == 0 && i < kReq + 2) request_codes(s + 3, slot3f, i - kReq);
        } else if constexpr (i < kReq + kOwn) {
          request_codes((s + 4) >> 1, 0, 2 * par + h);
        } else if constexpr (h == 0 && i == kReq + kOwn) {
          request_scales(slot3f);
        }
      };
      if constexpr (kIdle) {
        meet();
        repeat<4>([&](auto i_) __attribute__((always_inline)) { requests(I0{}, i_); });
        meet();
        repeat<4>([&](auto i_) __attribute__((always_inline)) { requests(I1{}, i_); });
      } else {
        repeat<T>([&](auto t_) __attribute__((always_inline)) {
          constexpr int t = decltype(t_)::value;
          constexpr int h = t / (2 * NB), gg = (t / 2) % NB, c = t & 1;
          constexpr int il = gg % (NB / 2), kk = gg / (NB / 2);
          typedef std::integral_constant<int, h> H;
          if constexpr (gg == NB - 2 && c == 0) meet();
          mfma16<CT>(acc[h * (NB / 2) + il][c], fr[(par * 2 * NB + h * NB + gg) & 7], __builtin_bit_cast(vec_t, b[par][c][kk]));
          constexpr int after = 2 * (gg - (NB - 2)) + c;          // 0 .. 3: slots behind a meeting
          if constexpr (after >= 0) requests(H{}, std::integral_constant<int, after>{});
          // codes and scales
          if constexpr (kBackward) {
            constexpr int unit = t / (NB / 2), in_unit = t % (NB / 2);
            if constexpr (unit < kUnits - 1 && in_unit == 0) read_unit(Next{}, std::integral_constant<int, unit + 1>{}, s + 1, slot3, mq);
            if constexpr (t == (NB / 2 > 4 ? T - 4 : T - NB / 2)) read_unit(Par{}, I0{}, s + 2, slot3n, mqn);
          } else if constexpr (after >= 0 && after < 3) {
            repeat<(after < 2 ? 2 : 1)>([&](auto i_) __attribute__((always_inline)) {
              typedef std::integral_constant<int, 2 * after + decltype(i_)::value> X;
              if constexpr (h == 0) read_raw(Next{}, I1{}, X{}, s + 1, slot3, 0);
              else read_raw(Par{}, I0{}, X{}, s + 2, slot3n, 0);
            });
          }
          // fragments
          if constexpr (after >= 0) {
            if constexpr (h == 0) read_frag(Par{}, I1{}, std::integral_constant<int, after>{});
            else read_frag(Next{}, I0{}, std::integral_constant<int, after>{});
          } else if constexpr (gg + 4 < NB && c == 0) {
            read_frag(Par{}, H{}, std::integral_constant<int, gg + 4>{});
          }
          // forward: from the third slot of a half to the meeting; gradient: throughout
          constexpr int lead = NB >= 6 ? 2 : 0, slots = kBackward ? T : 2 * NB - 4 - lead;
          constexpr int ts = kBackward ? t : t - h * 2 * NB - lead, base = kBackward ? 0 : 24 * h, parts = kBackward ? 48 : 24;
          if constexpr (ts >= 0 && ts < slots) {
            constexpr int first = base + ts * parts / slots, end = base + (ts + 1) * parts / slots;
            repeat<end - first>([&](auto i_) __attribute__((always_inline)) {
              constexpr int u = first + decltype(i_)::value;
              dequant(std::integral_constant<int, u % 3>{}, std::integral_constant<int, u / 3>{}, b[par ^ 1]);
            });
          }
          __builtin_amdgcn_sched_barrier(0);
        });
      }
      slot3 = slot3n;
      slot3n = slot3f;
      if constexpr (kBackward) {
        mq = mqn;
        mqn += m_step;
        if (mqn >= V) mqn -= V;
      }
    };
    for (int s = 0; s < steps; s += 2) {          // an even number of steps
      step(I0{}, s);
      step(I1{}, s + 1);
    }
    // the last products have to leave the pipe before their registers are read (the compiler does not see the asm's
    // latency), requests past the last step may still be writing LDS, and other waves may still be reading
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    if constexpr (!kIdle) {
      // 16-bit results: into LDS as rows of the tile; fp32 ones straight to memory, 64 (forward) or 256 bytes of a row at a time
      auto stage = [&](auto type_) __attribute__((always_inline)) {
        typedef decltype(type_) T;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            unsigned char *row = smem + (16 * i + 4 * q + r) * kPitch;
            if constexpr (kBackward) {
              *reinterpret_cast<uint32_t *>(row + (kCols * wave + 2 * j) * 2) = pack2<T>(acc[i][0][r], acc[i][1][r]);
            } else {
#pragma unroll
              for (int c = 0; c < 2; ++c) *reinterpret_cast<T *>(row + (kCols * wave + 16 * c + j) * 2) = from_f32<T>(acc[i][c][r]);
            }
          }
      };
      if (g.d_dtype == CAIFX_BF16) {
        stage(bf16_t{});
      } else if (g.d_dtype == CAIFX_F16) {
        stage(f16_t{});
      } else {
        int lane_row = 4 * q;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          asm volatile("" : "+v"(lane_row));           // one row tile's addresses at a time: 64 of them at once do not fit
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int lrow = lane_row + 16 * i + r;
            if (lrow >= rows) continue;
            const int64_t o = (row0 + lrow) * C + col0 + kCols * wave + (kBackward ? 2 * j : j);
            float *dp = static_cast<float *>(g.d) + o;
            const float *ap = static_cast<const float *>(g.addend) + o;
            if constexpr (kBackward) {
              floatx2_t v = {acc[i][0][r], acc[i][1][r]};
              if (g.addend) v += *reinterpret_cast<const floatx2_t *>(ap);
              *reinterpret_cast<floatx2_t *>(dp) = v;
            } else {
#pragma unroll
              for (int c = 0; c < 2; ++c) dp[16 * c] = g.addend ? acc[i][c][r] + ap[16 * c] : acc[i][c][r];
            }
          }
        }
      }
    }
  };
  auto run_rows = [&](auto nb_) __attribute__((always_inline)) {
    if (__builtin_amdgcn_readfirstlane(col0 + kCols * wave >= C ? 1 : 0)) run(nb_, std::true_type{});      // scalar: the branches hold barriers
    else run(nb_, std::false_type{});
  };
  switch (__builtin_amdgcn_readfirstlane((rows + 31) >> 5)) {
    case 0:
    case 1:
    case 2: run_rows(std::integral_constant<int, 4>{}); break;
    case 3: run_rows(std::integral_constant<int, 6>{}); break;
    case 4: run_rows(std::integral_constant<int, 8>{}); break;
    case 5: run_rows(std::integral_constant<int, 10>{}); break;
    case 6: run_rows(std::integral_constant<int, 12>{}); break;
    case 7: run_rows(std::integral_constant<int, 14>{}); break;
    default: run_rows(std::integral_constant<int, 16>{}); break;
  }
  // 16-bit results in whole rows, 16 bytes per lane.  mode: 0 the result, 1 with an addend, 2 and 3 the gated experts' second
  // result (forward, backward)
  auto store = [&](auto type_, auto mode_) __attribute__((always_inline)) {
    typedef decltype(type_) T;
    constexpr int mode = decltype(mode_)::value;
    constexpr int kBatch = 4;
    T *dp = static_cast<T *>(g.d);
    const int chunk = lane & 31;
    const int64_t gcol = col0 + chunk * 8;
    if (gcol >= C) return;                               // C is a multiple of 64
    for (int r0 = 2 * wave + (lane >> 5); r0 < rows; r0 += 2 * kWaves * kBatch) {
      u32x4_t e1[kBatch], e2[kBatch];
      if constexpr (mode != 0) {
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
          const int lrow = r0 + 2 * kWaves * b < rows ? r0 + 2 * kWaves * b : rows - 1;
          const int64_t o = (row0 + lrow) * C + gcol;
          e1[b] = *reinterpret_cast<const u32x4_t *>(static_cast<const T *>(mode == 1 ? g.addend : g.e1) + o);
          if constexpr (mode == 3) e2[b] = *reinterpret_cast<const u32x4_t *>(static_cast<const T *>(g.e2) + o);
        }
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const int lrow = r0 + 2 * kWaves * b;
        if (lrow >= rows) break;
        u32x4_t v = *reinterpret_cast<const u32x4_t *>(smem + lrow * kPitch + chunk * 16);
        const int64_t o = (row0 + lrow) * C + gcol;
        if constexpr (mode != 0) {
          u32x4_t w = v, w2 = v;
          const T *vp = reinterpret_cast<const T *>(&v);
          const T *p1 = reinterpret_cast<const T *>(&e1[b]);
          const T *p2 = reinterpret_cast<const T *>(&e2[b]);
          T *wp = reinterpret_cast<T *>(&w);
          T *w2p = reinterpret_cast<T *>(&w2);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            if constexpr (mode == 1) wp[e] = from_f32<T>(to_f32<T>(vp[e]) + to_f32<T>(p1[e]));
            else if constexpr (mode == 2) w2p[e] = swiglu_fwd_one<T>(p1[e], vp[e]);
            else swiglu_bwd_one<T>(p1[e], p2[e], vp[e], wp[e], w2p[e]);
          }
          if constexpr (mode >= 2) *reinterpret_cast<u32x4_t *>(static_cast<T *>(g.d2) + o) = w2;
          v = w;
        }
        *reinterpret_cast<u32x4_t *>(dp + o) = v;
      }
    }
  };
  if (g.d_dtype != CAIFX_F32) {
    __syncthreads();
    auto store_as = [&](auto type_) __attribute__((always_inline)) {
      if (g.epilogue != 0) store(type_, std::integral_constant<int, kBackward ? 3 : 2>{});
      else if (g.addend) store(type_, std::integral_constant<int, 1>{});
      else store(type_, std::integral_constant<int, 0>{});
    };
    if (g.d_dtype == CAIFX_BF16) store_as(bf16_t{});
    else store_as(f16_t{});
  }
  if (stamp_pos >= 0) g.stamps[4 * stamp_pos + 3] = wall_clock64();
}

template <typename CT, bool kBackward> int launch(const TallArgs &t, hipStream_t s)
{
  constexpr int kStore = BM * (BN * 2 + 32);
  constexpr int kRing = kBackward ? kLdsMax : kScalesFwd + 3 * 8192;
  constexpr int kLds = kRing > kStore ? kRing : kStore;
  auto kern = tall_gemm_kernel<CT, kBackward>;
  static std::atomic<bool> raised{false};
  if (!raised.load(std::memory_order_relaxed)) {
    // the attribute is per kernel and sticky; two threads racing here both set it, which is harmless
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return CAIFX_ERR_LAUNCH_FAILED;
    raised.store(true, std::memory_order_relaxed);
  }
  // segment lengths live on the device: the grid is an upper bound, every expert can add one partial tile
  const int64_t C = kBackward ? t.K : t.N;
  const int64_t tiles = ((t.M + t.height - 1) / t.height + t.num_experts) * ((C + BN - 1) / BN);
  if (tiles > (int64_t{1} << 30)) return CAIFX_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((tiles + 7) / 8 * 8)), dim3(64 * kWaves), kLds, s, t);
  return launch_status();
}

// the launches of one compute type, one translation unit each (they take a minute to compile)
int launch_bf16(const TallArgs &t, bool backward, hipStream_t s);
int launch_f16(const TallArgs &t, bool backward, hipStream_t s);

}  // namespace tall
}  // namespace caifx
