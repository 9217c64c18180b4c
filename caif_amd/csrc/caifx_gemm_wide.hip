// Large-M dequant-GEMM, forward and input gradient, in two launches: the weight is dequantised once into the caller's
// workspace as a dense matrix of the compute type, [columns of the result, reduction] row-major (the input gradient's
// transposed on the way), and a dense kernel multiplies it with the activations.  A weight stored in the 16-bit compute
// type needs no first launch in the forward direction.
//
// What bounds it: the power the chip may draw.  On all-zero operands the kernel runs at 2.03 PFLOP/s and a clock of 2.47
// GHz, on N(0,1) activations x N(0,0.02) weights at 1.50 to 1.56 and 1.99 GHz, in the same number of cycles (M = 4096, C =
// 4096, R = 11008: 236 to 247 us), so what counts is work per flop, not only what waits
// for what:
//  - v_mfma_f32_16x16x32 instead of 32x32x16: the same loop without any memory traffic runs at 2.07 instead of 1.80
//    PFLOP/s on those values (a 16 x 16 result is read and written once per 32 reduction elements, a 32 x 32 one once
//    per 16), the whole kernel at 236 instead of 254 us.
//  - four waves with 128 x 128 of the 256 x 256 tile each (one wave per SIMD, 256 accumulators in the accumulation
//    registers): 128 KB of operand reads from LDS per 64-deep step; eight waves of 128 x 64 read 192 KB (262 us).
//  - the weight is dequantised once per call instead of once per row tile.
// Against the kernels that dequantise inside the product (forward 361 us, input gradient 390 us at M = 4096, N = 11008,
// K = 4096, int4, bf16) the two launches take 293 and 251 us in the same run.
#include "caifx_gemm_regw.hpp"

#include <atomic>
#include <type_traits>

namespace caifx {
namespace {

constexpr int kBK = 64;                    // reduction extent of a step: one 128-byte line of every row
constexpr int kBandRows = 1024;            // rows of a band of the tile order

struct WideArgs {
  const void *a;        // [M, R] activations / gradients of the compute type
  const void *b;        // [C, R] dense weight of the compute type
  void *d;              // [M, C]
  const void *addend;
  int64_t M, C, R;
  int d_dtype;
  // grouped form: rows [offsets[e], offsets[e + 1]) times the e-th [C, R] matrix behind b
  const int32_t *offsets;
  const void *const *wq_ptrs;
  int num_experts;
  bool zero_rest;
  unsigned long long *stamps;      // measurement only, see mfma_grouped_tile_stamps
  long long stamps_capacity;
};

// A result tile has 64 WI rows and 64 WJ columns.  Wave (wm, wn) owns rows h 32 WI + wm 16 WI + [0, 16 WI) and columns
// g 32 WJ + wn 16 WJ + [0, 16 WJ) of it for h, g in {0, 1}: four quadrants of WI x WJ products.  LDS holds four half
// tiles per operand: half h of step s in slot 2 (s & 1) + h.  A step runs through the quadrants (h, g) = (0,0) (0,1)
// (1,1) (1,0); the operands of a quadrant are read during the one before it, so half 1 of step s has been read by
// everybody in the middle of quadrant (1,1) and half 0 in the middle of the next step's (0,0).  There, and only there,
// the waves meet; behind the barrier the freed slot is requested for step s + 2, three half tiles (96 KB per compute
// unit for 256 x 256) are on their way at any time, and every request has one and a half steps to arrive.  Requests
// complete in issue order, so the wait for the half tile that is read next is an exact count (a wave issues WI + WJ
// per half).
template <typename CT, int WI, int WJ, bool kGrouped>
__global__ __launch_bounds__(256, WI + WJ <= 4 ? 2 : 1) void wide_gemm_kernel(WideArgs g)
{
  typedef typename Mfma32<CT>::vec_t vec_t;
  constexpr int BM = 64 * WI, BN = 64 * WJ;
  constexpr int kASlot = BM / 2 * 128, kBSlot = BN / 2 * 128;      // LDS bytes of half an operand tile
  constexpr int kBBase = 4 * kASlot;
  constexpr int kBand = kBandRows / BM;
  constexpr int kReq = WI + WJ;            // requests of a wave per half step
  constexpr int Q = 2 * WI * WJ;           // products per quadrant
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int r16 = lane & 15, kq = lane >> 4;

  // XCD x (workgroup id mod 8, each with its own L2) walks the x-th contiguous eighth of a list that runs through bands
  // of 1024 rows column by column: the 256 x 256 tiles it works on at a time share 4 row and 8 column panels
  const int64_t col_tiles = (g.C + BN - 1) / BN, row_tiles = (g.M + BM - 1) / BM;
  int64_t row0, col0, row_end = g.M;
  uint64_t b_ptr = reinterpret_cast<uint64_t>(g.b);
  int64_t stamp_pos = -1;
  if constexpr (kGrouped) {
    GroupedTile gt;
    const bool has_tile = grouped_tile<BM>(g.offsets, g.num_experts, g.M, col_tiles, g.wq_ptrs, nullptr, lane, gt);
    if (g.zero_rest) zero_uncovered(g.offsets, g.num_experts, g.M, gt.first, gt.end, gt.ordered, g.d, g.C * (g.d_dtype == CAIFX_F32 ? 4 : 2));
    if (!has_tile) return;
    // the search's results are the same in every lane: into scalar registers with them
    row0 = uniform64(static_cast<uint64_t>(gt.row0));
    row_end = uniform64(static_cast<uint64_t>(gt.row_end));
    col0 = uniform64(static_cast<uint64_t>(gt.col_tile * BN));
    b_ptr = uniform64(b_ptr + static_cast<uint64_t>(gt.e) * static_cast<uint64_t>(g.C * g.R * 2));
    if (g.stamps && threadIdx.x == 0 && gt.pos < g.stamps_capacity) {
      stamp_pos = gt.pos;
      const int64_t rows = row_end - row0 < BM ? row_end - row0 : BM;
      g.stamps[4 * stamp_pos] = static_cast<unsigned long long>(gt.e);
      g.stamps[4 * stamp_pos + 1] = static_cast<unsigned long long>(rows) | (WI + WJ <= 4 ? 0ull : 1ull << 32);      // one or two workgroups per compute unit
      g.stamps[4 * stamp_pos + 2] = wall_clock64();
    }
  } else {
    const unsigned bid = blockIdx.x;
    const int64_t per_xcd = gridDim.x >> 3;
    const int64_t pos = static_cast<int64_t>(bid & 7) * per_xcd + (bid >> 3);
    if (pos >= row_tiles * col_tiles) return;
    const int64_t band = pos / (kBand * col_tiles);
    const int64_t within = pos - band * kBand * col_tiles;
    const int64_t left = row_tiles - band * kBand;
    const int64_t band_rows = left < kBand ? left : kBand;
    col0 = (within / band_rows) * BN;
    row0 = (band * kBand + within % band_rows) * BM;
  }

  // request i of a wave for half h of an operand: 8 rows x 128 bytes; LDS position p of row r holds 16-byte chunk
  // p ^ (r ^ r >> 3) & 7 of the row (operand reads without bank conflicts), so that is the chunk a lane asks for.  Rows
  // and columns past the end are loaded from the last one and never stored.
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  uint32_t a_voff[2][WI], b_voff[2][WJ];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int lrow = 8 * (wave + 4 * i) + (lane >> 3);
      int64_t m = row0 + h * (BM / 2) + lrow;
      if (m >= row_end) m = row_end - 1;
      a_voff[h][i] = static_cast<uint32_t>((m - row0) * g.R * 2 + (((lane & 7) ^ ((lrow ^ (lrow >> 3)) & 7)) << 4));
    }
#pragma unroll
    for (int i = 0; i < WJ; ++i) {
      const int lrow = 8 * (wave + 4 * i) + (lane >> 3);
      int64_t c = col0 + h * (BN / 2) + lrow;
      if (c >= g.C) c = g.C - 1;
      b_voff[h][i] = static_cast<uint32_t>((c - col0) * g.R * 2 + (((lane & 7) ^ ((lrow ^ (lrow >> 3)) & 7)) << 4));
    }
  }
  const uint64_t a_base = uniform64(reinterpret_cast<uint64_t>(g.a) + static_cast<uint64_t>(row0 * g.R * 2));
  const uint64_t b_base = uniform64(b_ptr + static_cast<uint64_t>(col0 * g.R * 2));
  const int steps = static_cast<int>(g.R / kBK);
  const int last = steps - 1;
  auto request = [&](int s, int h, int slot, int x) __attribute__((always_inline)) {
    const uint32_t k0 = static_cast<uint32_t>(s < last ? s : last) * 128;          // past the end: the last step again
    const bool is_a = x < WI;
    const int i = is_a ? x : x - WI;
    const uint64_t src = (is_a ? a_base : b_base) + k0;
    const uint32_t dst = lds0 + (is_a ? slot * kASlot : kBBase + slot * kBSlot) + (wave + 4 * i) * 1024;
    const uint32_t voff = is_a ? a_voff[h][is_a ? i : 0] : b_voff[h][is_a ? 0 : i];
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(voff), "s"(src) : "memory");
  };

  // operand (row tile i of 16 rows, reduction half kk): tiles i and i + 2 lie 32 rows apart, which flips the
  // swizzle's third bit, the one that kk selects
  uint32_t a_addr[2][2], b_addr[2][2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int ra = wm * 16 * WI + i * 16 + r16;
      a_addr[i][kk] = ra * 128 + (((4 * kk + kq) ^ ((ra ^ (ra >> 3)) & 7)) << 4);
      const int rb = wn * 16 * WJ + i * 16 + r16;
      b_addr[i][kk] = kBBase + rb * 128 + (((4 * kk + kq) ^ ((rb ^ (rb >> 3)) & 7)) << 4);
    }
  auto read_a = [&](int slot, int i, int kk) __attribute__((always_inline)) {
    return *reinterpret_cast<const vec_t *>(smem + slot * kASlot + (i >> 1) * 4096 + a_addr[i & 1][kk ^ (i >> 1)]);
  };
  auto read_b = [&](int slot, int i, int kk) __attribute__((always_inline)) {
    return *reinterpret_cast<const vec_t *>(smem + slot * kBSlot + (i >> 1) * 4096 + b_addr[i & 1][kk ^ (i >> 1)]);
  };

  floatx4_t acc[2][2][WI][WJ];     // [h][g][row tile][column tile]
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int c = 0; c < WJ; ++c) acc[h][q][i][c] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};

#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int x = 0; x < kReq; ++x) request(u >> 1, u & 1, u, x);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * kReq) : "memory");
  vec_t a0[WI][2], a1[WI][2], b0[WJ][2], b1[WJ][2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
    for (int i = 0; i < WJ; ++i) b0[i][kk] = read_b(0, i, kk);
#pragma unroll
    for (int i = 0; i < WI; ++i) a0[i][kk] = read_a(0, i, kk);
  }

  // one quadrant: its products run to and fro over the row tiles so that one operand stays from product to product;
  // `first` runs in front of the second half, `each` behind every product
  auto quadrant = [&](floatx4_t(&d)[WI][WJ], const vec_t(&a)[WI][2], const vec_t(&b)[WJ][2], auto first, auto each) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < Q; ++t) {
      if (t == Q / 2) first();
      const int u = t % (WI * WJ), kk = t / (WI * WJ);
      const int c = u / WI, i = (c & 1) ? WI - 1 - u % WI : u % WI;
      mfma16<CT>(d[i][c], a[i][kk], b[c][kk]);
      each(t);
      if (t & 1) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // the n reads or requests of half a quadrant, spread over its Q / 2 products (t = 0 .. Q / 2 - 1)
  auto spread = [&](int t, int n, auto op) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < n; ++x)
      if (x * (Q / 2) / n == t) op(x);
  };
  auto meet = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * kReq) : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto nothing = []() __attribute__((always_inline)) {};
  auto step = [&](auto par_, int s) __attribute__((always_inline)) {
    constexpr int p = decltype(par_)::value;
    constexpr int S0 = 2 * p, S1 = 2 * p + 1, S0n = 2 * (p ^ 1);
    quadrant(acc[0][0], a0, b0, meet, [&](int t) __attribute__((always_inline)) {
      spread(t - Q / 2, 2 * WJ, [&](int x) __attribute__((always_inline)) { b1[x % WJ][x / WJ] = read_b(S1, x % WJ, x / WJ); });
      spread(t - Q / 2, kReq, [&](int x) __attribute__((always_inline)) { request(s + 2, 0, S0, x); });
    });
    quadrant(acc[0][1], a0, b1, nothing, [&](int t) __attribute__((always_inline)) {
      spread(t, 2 * WI, [&](int x) __attribute__((always_inline)) { a1[x % WI][x / WI] = read_a(S1, x % WI, x / WI); });
    });
    quadrant(acc[1][1], a1, b1, meet, [&](int t) __attribute__((always_inline)) {
      spread(t - Q / 2, 2 * WI, [&](int x) __attribute__((always_inline)) { a0[x % WI][x / WI] = read_a(S0n, x % WI, x / WI); });
      spread(t - Q / 2, kReq, [&](int x) __attribute__((always_inline)) { request(s + 2, 1, S1, x); });
    });
    quadrant(acc[1][0], a1, b0, nothing, [&](int t) __attribute__((always_inline)) {
      if (t % WI == WI - 1) b0[(t / WI) % WJ][t / (WI * WJ)] = read_b(S0n, (t / WI) % WJ, t / (WI * WJ));
    });
  };
  int s = 0;
  for (; s + 2 <= steps; s += 2) {
    step(std::integral_constant<int, 0>{}, s);
    step(std::integral_constant<int, 1>{}, s + 1);
  }
  if (s < steps) step(std::integral_constant<int, 0>{}, s);
  // the last products have to leave the pipe before their registers are read (the compiler does not see the asm's
  // latency), requests past the last step may still be writing LDS, and other waves may still be reading
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // store through LDS: a pass of whole tile rows (16-bit results: all of them, fp32: one half), row pitch = row + 32
  // bytes so that the four row groups of a wave's registers spread over the banks, then whole rows, 16 bytes per lane.
  // The optional addend is read the same way, a batch of rows ahead (the operand registers are free by now): read row
  // by row in front of each store it took 46 us of 322 at M = 4096, C = 11008, R = 4096.
  auto store = [&](auto type_, auto add_) __attribute__((always_inline)) {
    typedef decltype(type_) T;
    constexpr bool kAdd = decltype(add_)::value;
    constexpr int kPitch = BN * sizeof(T) + 32;
    constexpr int kPer16 = 16 / sizeof(T);
    constexpr int kLanesPerRow = BN / kPer16;            // 16, 32 or 64
    constexpr int kPassHalves = sizeof(T) == 2 ? 2 : 1;
    constexpr int kRows = kPassHalves * (BM / 2);
    constexpr int kRowsPerInstr = 64 / kLanesPerRow;
    constexpr int kInstr = kRows / (4 * kRowsPerInstr);  // rows of a wave per pass, in instructions
    constexpr int kBatch = kInstr < 8 ? kInstr : 8;
    T *dp = static_cast<T *>(g.d);
    const T *ap = static_cast<const T *>(g.addend);
    const int chunk = lane % kLanesPerRow;
    const int64_t gcol = col0 + chunk * kPer16;
    const int64_t acol = gcol < g.C ? gcol : 0;          // C is a multiple of 8
    u32x4_t add[2][kBatch];
    auto fetch = [&](u32x4_t(&to)[kBatch], int pass, int batch) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        int64_t grow = row0 + pass * (BM / 2) + ((batch * kBatch + b) * 4 + wave) * kRowsPerInstr + lane / kLanesPerRow;
        if (grow >= row_end) grow = row_end - 1;
        to[b] = *reinterpret_cast<const u32x4_t *>(ap + grow * g.C + acol);
      }
    };
#pragma unroll
    for (int pass = 0; pass < 2 / kPassHalves; ++pass) {
      if (pass > 0) __syncthreads();
      if constexpr (kAdd) fetch(add[0], pass, 0);
#pragma unroll
      for (int hh = 0; hh < kPassHalves; ++hh)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int i = 0; i < WI; ++i)
#pragma unroll
            for (int c = 0; c < WJ; ++c)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const int lrow = hh * (BM / 2) + wm * 16 * WI + i * 16 + 4 * kq + r;
                *reinterpret_cast<T *>(smem + lrow * kPitch + (q * (BN / 2) + wn * 16 * WJ + c * 16 + r16) * sizeof(T)) =
                    from_f32<T>(acc[pass * kPassHalves + hh][q][i][c][r]);
              }
      __syncthreads();
#pragma unroll
      for (int batch = 0; batch < kInstr / kBatch; ++batch) {
        if constexpr (kAdd) {
          if (batch + 1 < kInstr / kBatch) fetch(add[(batch + 1) & 1], pass, batch + 1);
        }
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
          const int lrow = ((batch * kBatch + b) * 4 + wave) * kRowsPerInstr + lane / kLanesPerRow;
          const int64_t grow = row0 + pass * (BM / 2) + lrow;
          u32x4_t v = *reinterpret_cast<const u32x4_t *>(smem + lrow * kPitch + chunk * 16);
          if constexpr (kAdd) {
            const T *vp = reinterpret_cast<const T *>(&v);
            const T *aq = reinterpret_cast<const T *>(&add[batch & 1][b]);
            u32x4_t w;
            T *wp = reinterpret_cast<T *>(&w);
#pragma unroll
            for (int e = 0; e < kPer16; ++e) wp[e] = from_f32<T>(to_f32<T>(vp[e]) + to_f32<T>(aq[e]));
            v = w;
          }
          if (grow < row_end && gcol < g.C) *reinterpret_cast<u32x4_t *>(dp + grow * g.C + gcol) = v;
        }
      }
    }
  };
  auto store_as = [&](auto type_) __attribute__((always_inline)) {
    if (g.addend) store(type_, std::true_type{});
    else store(type_, std::false_type{});
  };
  if (g.d_dtype == CAIFX_BF16) store_as(bf16_t{});
  else if (g.d_dtype == CAIFX_F16) store_as(f16_t{});
  else store_as(float{});
  if constexpr (kGrouped) {
    if (stamp_pos >= 0) g.stamps[4 * stamp_pos + 3] = wall_clock64();
  }
}

// ------------------------------------------------------------------ the weight as a dense matrix of the compute type
struct DenseArgs {
  const void *q;
  const void *scales;
  void *out;
  int64_t N, K;
  int group_shift;         // int4
  uint32_t period;         // int8; 0 = no scales
  // grouped form: expert blockIdx.z, skipped when it has no rows; its copy is the z-th [N, K] behind out
  const int32_t *offsets;
  const void *const *wq_ptrs;
  const void *const *scales_ptrs;
  int64_t M;
};

// the grouped form's weight of this workgroup; false: nothing to do
__device__ __forceinline__ bool dense_expert(DenseArgs &g)
{
  if (!g.offsets) return true;
  const int e = static_cast<int>(blockIdx.z);
  int lo, hi;
  segment_rows(g.offsets, e, g.M, lo, hi);
  if (lo >= hi) return false;
  g.q = g.wq_ptrs[e];
  g.scales = g.scales_ptrs ? g.scales_ptrs[e] : nullptr;
  g.out = static_cast<char *>(g.out) + static_cast<int64_t>(e) * g.N * g.K * 2;
  return true;
}

enum { DK_INT8 = 0, DK_INT4 = 1, DK_16 = 2 };

// eight consecutive weights of flat index f (a multiple of 8) as fp32, the reference's code * scale
template <typename CT, int kKind>
__device__ __forceinline__ void load_weights8(const DenseArgs &g, int64_t f, float (&e)[8])
{
  if constexpr (kKind == DK_INT4) {
    const uint32_t p = *reinterpret_cast<const uint32_t *>(static_cast<const uint8_t *>(g.q) + (f >> 1));
    dequant_int4x8(p, to_f32(static_cast<const f16_t *>(g.scales)[f >> g.group_shift]), e);
  } else if constexpr (kKind == DK_INT8) {
    const u32x2_t p = *reinterpret_cast<const u32x2_t *>(static_cast<const uint8_t *>(g.q) + f);
    float lo[4], hi[4];
    int8x4_to_f32(p[0], lo);
    int8x4_to_f32(p[1], hi);
    const float *sp = static_cast<const float *>(g.scales);
    if (g.period > 1) {          // a multiple of 4: neither quad wraps inside
      const uint32_t i0 = static_cast<uint32_t>(f) % g.period;      // N * K < 2^32 (host)
      const uint32_t i1 = i0 + 4 < g.period ? i0 + 4 : i0 + 4 - g.period;
      const floatx4_t s0 = *reinterpret_cast<const floatx4_t *>(sp + i0), s1 = *reinterpret_cast<const floatx4_t *>(sp + i1);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        e[t] = lo[t] * s0[t];
        e[4 + t] = hi[t] * s1[t];
      }
    } else {
      const float s = g.period == 1 ? sp[0] : 1.0f;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        e[t] = lo[t] * s;
        e[4 + t] = hi[t] * s;
      }
    }
  } else {
    const u32x4_t p = *reinterpret_cast<const u32x4_t *>(static_cast<const CT *>(g.q) + f);
    const CT *v = reinterpret_cast<const CT *>(&p);
#pragma unroll
    for (int t = 0; t < 8; ++t) e[t] = to_f32<CT>(v[t]);
  }
}

// [N, K] as stored: eight values per thread and round, four rounds requested ahead.  Bound by HBM.
template <typename CT, int kKind>
__global__ __launch_bounds__(256) void dense_rows_kernel(DenseArgs g)
{
  constexpr int kRounds = 4;
  if (!dense_expert(g)) return;
  const int64_t pieces = g.N * g.K / 8;
  const int64_t p0 = static_cast<int64_t>(blockIdx.x) * (256 * kRounds) + threadIdx.x;
  float e[kRounds][8];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int64_t p = p0 + r * 256;
    load_weights8<CT, kKind>(g, (p < pieces ? p : pieces - 1) * 8, e[r]);
  }
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int64_t p = p0 + r * 256;
    if (p >= pieces) continue;
    u32x4_t v;
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] = pack2<CT>(e[r][2 * t], e[r][2 * t + 1]);
    *reinterpret_cast<u32x4_t *>(static_cast<CT *>(g.out) + p * 8) = v;
  }
}

// [K, N], transposed: a workgroup takes 64 rows n x 256 columns k.  A thread reads eight columns of eight rows (the
// 32 lanes of a row together 128 bytes of int4 codes), packs them into eight pieces of eight n and lays them out in
// LDS as rows of 64 n; the rows are then written in whole 128-byte lines.  The piece position is rotated by the
// thread's k so that the eight lanes of a group use different banks.
template <typename CT, int kKind>
__global__ __launch_bounds__(256) void dense_transposed_kernel(DenseArgs g)
{
  __shared__ __attribute__((aligned(16))) unsigned char tile[256 * 128];
  if (!dense_expert(g)) return;
  const int kl = threadIdx.x & 31, ng = threadIdx.x >> 5;
  const int64_t n0 = static_cast<int64_t>(blockIdx.y) * 64, k0 = static_cast<int64_t>(blockIdx.x) * 256;
  if (k0 + 8 * kl < g.K) {
    float e[8][8];
#pragma unroll
    for (int r = 0; r < 8; ++r) load_weights8<CT, kKind>(g, (n0 + 8 * ng + r) * g.K + k0 + 8 * kl, e[r]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      u32x4_t v;
#pragma unroll
      for (int t = 0; t < 4; ++t) v[t] = pack2<CT>(e[2 * t][j], e[2 * t + 1][j]);
      *reinterpret_cast<u32x4_t *>(tile + (8 * kl + j) * 128 + (((ng + kl) & 7) << 4)) = v;
    }
  }
  __syncthreads();
  const int piece = threadIdx.x & 7;
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int k = it * 32 + (threadIdx.x >> 3);
    if (k0 + k >= g.K) continue;
    const u32x4_t v = *reinterpret_cast<const u32x4_t *>(tile + k * 128 + (((piece + (k >> 3)) & 7) << 4));
    *reinterpret_cast<u32x4_t *>(static_cast<CT *>(g.out) + (k0 + k) * g.N + n0 + 8 * piece) = v;
  }
}

template <typename CT>
int launch_dense(const DenseArgs &g, int kind, bool transposed, int experts, hipStream_t s)
{
  if (transposed) {
    const dim3 grid(static_cast<unsigned>((g.K + 255) / 256), static_cast<unsigned>(g.N / 64), static_cast<unsigned>(experts));
    if (kind == DK_INT4) hipLaunchKernelGGL((dense_transposed_kernel<CT, DK_INT4>), grid, dim3(256), 0, s, g);
    else if (kind == DK_INT8) hipLaunchKernelGGL((dense_transposed_kernel<CT, DK_INT8>), grid, dim3(256), 0, s, g);
    else hipLaunchKernelGGL((dense_transposed_kernel<CT, DK_16>), grid, dim3(256), 0, s, g);
  } else {
    const dim3 grid(static_cast<unsigned>((g.N * g.K / 8 + 1023) / 1024), 1, static_cast<unsigned>(experts));
    if (kind == DK_INT4) hipLaunchKernelGGL((dense_rows_kernel<CT, DK_INT4>), grid, dim3(256), 0, s, g);
    else hipLaunchKernelGGL((dense_rows_kernel<CT, DK_INT8>), grid, dim3(256), 0, s, g);
  }
  return launch_status();
}

template <typename CT, int WI, int WJ, bool kGrouped>
int launch_wide(const WideArgs &g, hipStream_t s)
{
  constexpr int BM = 64 * WI, BN = 64 * WJ;
  constexpr int kRing = (BM + BN) * 256, kStore16 = BM * (BN * 2 + 32), kStore32 = BM / 2 * (BN * 4 + 32);
  constexpr int kStore = kStore16 > kStore32 ? kStore16 : kStore32;
  constexpr int kLds = kRing > kStore ? kRing : kStore;
  auto kern = wide_gemm_kernel<CT, WI, WJ, kGrouped>;
  static std::atomic<bool> raised{false};
  if (!raised.load(std::memory_order_relaxed)) {
    // the attribute is per kernel and sticky; two threads racing here both set it, which is harmless
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return CAIFX_ERR_LAUNCH_FAILED;
    raised.store(true, std::memory_order_relaxed);
  }
  // grouped: segment lengths live on the device; an upper bound, every expert can add one partial tile
  const int64_t tiles = ((g.M + BM - 1) / BM + (kGrouped ? g.num_experts : 0)) * ((g.C + BN - 1) / BN);
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((tiles + 7) / 8 * 8)), dim3(256), kLds, s, g);
  return launch_status();
}

// What a 64-deep step of the whole launch costs with one of the three tiles, in us: the number of rounds the tiles take
// times the time of one, measured on N(0,1) x N(0,0.02) bf16 values at R = 4096.  256 x 256 (one workgroup per compute
// unit) 1.39 per round of 256, 128 x 256 (one) 0.87, 128 x 128 (two) 0.91 per round of 512 and 0.49 for a last round of
// at most 256.  M = 4096, C = 11008: 265 / 300 / 300 us; M = 2048, C = 11008: 166 / 149 / 162; M = 1024, C = 4096: 72 /
// 44 / 32.
enum { TILE_256 = 0, TILE_128x256 = 1, TILE_128 = 2 };
// row tiles of bm rows; over expert segments of unknown lengths the last tile of each is taken as half full
int64_t row_tiles_of(int64_t M, int experts, int64_t bm)
{
  if (experts == 0) return (M + bm - 1) / bm;
  const int64_t t = (M + bm - 1) / bm + experts / 2, least = M < experts ? M : experts;
  return t > least ? t : least;
}
double step_cost(int tile, int64_t M, int64_t C, int experts)
{
  const auto tiles = [&](int64_t bm, int64_t bn) { return row_tiles_of(M, experts, bm) * ((C + bn - 1) / bn); };
  if (tile == TILE_256) return 1.39 * static_cast<double>((tiles(256, 256) + 255) / 256);
  if (tile == TILE_128x256) return 0.87 * static_cast<double>((tiles(128, 256) + 255) / 256);
  const int64_t t = tiles(128, 128), rest = t % 512;
  return 0.91 * static_cast<double>(t / 512) + (rest == 0 ? 0.0 : rest <= 256 ? 0.49 : 0.91);
}
int best_tile(int64_t M, int64_t C, int experts)
{
  int best = TILE_256;
  for (int t = TILE_128x256; t <= TILE_128; ++t)
    if (step_cost(t, M, C, experts) < step_cost(best, M, C, experts)) best = t;
  return best;
}

// What a call costs on this path and on the kernels that dequantise inside the product, in us, for the choice between them
// (plain form; measured on N(0,1) x N(0,0.02) bf16 values for eleven weights from 2048 x 2048 to 14336 x 4096, 33 to 2048
// rows, both directions).  A partly filled round costs less than a full one: `base` + `per` for each of its tiles.
double rounds_cost(int64_t tiles, int64_t slots, double full, double base, double per)
{
  const int64_t rest = tiles % slots;
  return full * static_cast<double>(tiles / slots) + (rest == 0 ? 0.0 : base + per * static_cast<double>(rest));
}
double wide_us(const GemmArgs &a, bool backward)
{
  const int64_t C = backward ? a.K : a.N, R = backward ? a.N : a.K;
  const auto tiles = [&](int64_t bm, int64_t bn) { return (a.M + bm - 1) / bm * ((C + bn - 1) / bn); };
  double step;
  switch (best_tile(a.M, C, 0)) {
    case TILE_256: step = rounds_cost(tiles(256, 256), 256, 1.42, 0.75, 0.0026); break;
    case TILE_128x256: step = rounds_cost(tiles(128, 256), 256, 0.81, 0.25, 0.0022); break;
    default: {
      const int64_t t = tiles(128, 128);
      step = t % 512 <= 256 ? rounds_cost(t, 512, 0.82, 0.24, 0.0008) : rounds_cost(t, 512, 0.82, 0.30, 0.0010);
    }
  }
  // the dense copy, per million weights; of a 16-bit weight beyond 48 million it no longer stays in the memory-side cache
  const double millions = 1e-6 * static_cast<double>(a.N) * static_cast<double>(a.K);
  const double copy = a.w.kind == CAIFX_W_INT8          ? 10.0 + 0.42 * millions
                      : a.w.kind == CAIFX_W_INT4_GROUP ? 10.0 + 0.34 * millions
                                                       : 6.0 + (millions > 48.0 ? 0.78 : 0.40) * millions;
  return step * static_cast<double>(R / kBK) + copy;
}
// caifx_gemm.hip: 256 x 128 tiles for long reductions with enough of them, else 128 x 128, whose reduction is shared out
// where at most 128 of them leave compute units idle
double tiled_us(const GemmArgs &a, bool backward)
{
  const int64_t C = backward ? a.K : a.N, R = backward ? a.N : a.K;
  const bool int8 = a.w.kind == CAIFX_W_INT8, int4 = a.w.kind == CAIFX_W_INT4_GROUP;
  const int64_t cols = (C + 127) / 128, tall = (a.M + 255) / 256 * cols, tiles = (a.M + 127) / 128 * cols;
  const double steps = static_cast<double>(R / kBK);
  // int8 codes with one scale or none are unpacked more slowly than those with a scale vector; without a call's scales (the
  // workspace query) they are taken to be such
  const double slower = int8 && a.w.scale_period <= 1 ? 2.3 : 1.0;
  if (tall >= 200 && R > 2048) return static_cast<double>((tall + 255) / 256) * ((int8 ? 1.10 * slower : int4 ? 1.07 : 1.04) * steps + 2.0);
  const auto one_each = [&](int64_t t) {       // us per step with up to 256 workgroups
    return int8 ? 1.07 * slower : int4 ? 0.35 + 0.0015 * static_cast<double>(t) : 0.40 + 0.0009 * static_cast<double>(t);
  };
  if (tiles <= 128) {
    int64_t parts = 256 / tiles;
    if (parts > 8) parts = 8;
    if (parts > R / kBK / 8) parts = R / kBK / 8;
    if (parts >= 2) {
      const int64_t per = (R / kBK + parts - 1) / parts;
      return one_each(tiles * parts) * static_cast<double>(per) + 10.0 + 1.6e-6 * static_cast<double>(parts * a.M) * static_cast<double>(C);
    }
  }
  const double two_each = int8 ? 2.14 * slower : int4 ? 1.18 : 1.20;
  const int64_t rest = tiles % 512;
  return 5.0 + steps * (two_each * static_cast<double>(tiles / 512) + (rest == 0 ? 0.0 : rest <= 256 ? one_each(rest) : two_each));
}
// caifx_gemm_regw.hip and caifx_gemm_regw8.hip: 128 x 256 tiles, one workgroup per compute unit
double regw_us(const GemmArgs &a)
{
  const int64_t tiles = (a.M + 127) / 128 * ((a.N + 255) / 256);
  const double steps = static_cast<double>(a.K / kBK);
  if (a.w.kind == CAIFX_W_INT8) return 4.0 + steps * rounds_cost(tiles, 256, 1.10, 0.75, 0.0013);
  return 4.0 * static_cast<double>((tiles + 255) / 256) + steps * rounds_cost(tiles, 256, 0.90, 0.55, 0.0014);
}

template <typename CT, bool kGrouped>
int pick_wide(const WideArgs &g, hipStream_t s)
{
  switch (best_tile(g.M, g.C, g.num_experts)) {
    case TILE_256: return launch_wide<CT, 4, 4, kGrouped>(g, s);
    case TILE_128x256: return launch_wide<CT, 2, 4, kGrouped>(g, s);
    default: return launch_wide<CT, 2, 2, kGrouped>(g, s);
  }
}
template <typename CT>
int pick_form(const WideArgs &g, hipStream_t s)
{
  return g.offsets ? pick_wide<CT, true>(g, s) : pick_wide<CT, false>(g, s);
}

bool dense16(const GemmArgs &a)
{
  return (a.w.kind == CAIFX_W_BF16 && a.compute_dtype == CAIFX_BF16) || (a.w.kind == CAIFX_W_F16 && a.compute_dtype == CAIFX_F16);
}

// The rule on sizes and types (the workspace query knows nothing else: scale_period is 0 there).
bool wide_shape(const GemmArgs &a, bool backward)
{
  if (a.compute_dtype == CAIFX_F32 || a.x_dtype != a.compute_dtype || a.epilogue != 0) return false;
  const bool codes = a.w.kind == CAIFX_W_INT8 || a.w.kind == CAIFX_W_INT4_GROUP;
  if (!codes && !dense16(a)) return false;
  const int64_t C = backward ? a.K : a.N, R = backward ? a.N : a.K;
  if (R % kBK != 0 || C % 8 != 0 || a.K % 8 != 0 || a.M < 1 || R < 2 * kBK) return false;
  // (the transposing pass has R / 64 rows of workgroups, kept below the 65536 of a grid)
  if (a.N * a.K >= (int64_t{1} << 32) || a.M > (int64_t{1} << 30) || R >= (int64_t{1} << 22)) return false;
  const int64_t tiles = ((a.M + 127) / 128) * ((C + 127) / 128);
  if (tiles > (int64_t{1} << 30)) return false;
  if (a.offsets) {
    // Experts with long segments, and copies of all their weights within half of the memory-side cache (128 MB): the
    // dense pass then costs 10 to 20 us and the product gains a quarter.  Forward / input gradient in us, dequantised
    // inside the product against here, with uniformly drawn ids: N = 1408, K = 2048, 8 experts, 24576 rows, int8 198 / 216
    // against 156 / 158, int4 190 / 203 against 156 / 137; 33 experts (190 MB), 24576 rows, int8 218 / 243 against 244 / 235.
    // Over 840 calls (2 to 64 experts, 512 x 512 to 4096 x 4096, 760 to 4096 rows per expert, even and uneven segments, both
    // storages and directions) the 546 that the rule below admits are 1.26 times as fast in the mean; six are slower by more
    // than 2.5 %, by up to 16 %, where one more row tile than estimated starts another round (int8, 2 experts, 4096 x 4096, 4000
    // rows: 148 against 171).  What it leaves out: fewer rows (33 experts, 1024 x 1536, 29700 rows, int8 forward 122 against
    // 149), reductions of 512 (16 experts, 512 x 2048, 14400 rows, int4 gradient 58 against 64), small products (8 experts,
    // 512 x 1024, 16000 rows 27 against 36).  Stored 16-bit weights stay on the tiled kernel (input gradient, 16 experts: 188
    // against 215 us with 24576 rows, 157 against 147 with 16384).
    if (!codes || a.num_experts < 1 || a.num_experts > 65535) return false;
    const int64_t E = a.num_experts;
    const double product = static_cast<double>(a.M) * static_cast<double>(a.N) * static_cast<double>(a.K);
    return a.M >= (a.w.kind == CAIFX_W_INT8 && !backward ? 1250 : 1000) * E && E * a.N * a.K * 2 <= (int64_t{1} << 27) && R >= 768 &&
           product >= (a.M >= 3000 * E ? 5e9 : 1e10);
  }
  // Is it worth it?  `tiles` counts 128 x 128 tiles.  A stored 16-bit weight needs no extra pass in the forward
  // direction: from 100 tiles on (128: 25.8 against 27.4 us, 256: 31.5 against 39.4; 80: 26.1 against 24.2, where the
  // tiled kernel shares each tile's reduction among workgroups; with up to 128 tiles and long reductions that sharing wins:
  // M = 512, N = 4096, K = 14336 67 against 79 us, K = 11008 57 against 63, K = 4096 27.6 against 24.8).
  if (!codes && !backward) return tiles >= 100 && (tiles > 128 || R <= 6400);
  // int4 forward with whole 256-code blocks has a kernel of its own (caifx_gemm_regw.hip).  M = 512, N = 11008, K = 4096: 55
  // there against 65 us here, M = 2048: 180 against 173, M = 1024: 112 against 94.  K < 2048 stays there (M = 1536, N = 8192,
  // K = 1024: 37 against 39), and so do calls of up to one 128 x 128 tile per compute unit, which go on without a workspace
  // and with the same bits from caifx_qlinear_forward_static as from here (M = 1024, N = K = 4096: 51 us where this takes 41).
  if (!backward && a.w.kind == CAIFX_W_INT4_GROUP && a.K % 256 == 0 && (a.M + 127) / 128 * ((C + 255) / 256) >= 128)
    return tiles > 256 && a.K >= 2048 && wide_us(a, backward) < regw_us(a);
  // Everything else runs on the tiled kernel otherwise: int4 and 16-bit input gradients from 190 tiles on (198: 30.4 against
  // 37.4 us at M = 1367, N = 2880, K = 2304; 128: 85 against 76), int8, whose unpacking costs those kernels more, from 90
  // (96 tiles of the input gradient at N = 5952, K = 2048: 43 against 66 us; 64: 61 against 50), where the copy is used often
  // enough to pay: with one or two row tiles of a large weight it is not (N = 14336, K = 4096: int8, M = 64, 47 us there
  // against 52 here, M = 512 75 against 83; int4, M = 256, 44 against 53; K = 2048 25 against 37; the 16-bit gradient to 14336
  // columns, M = 256, 43 against 65).
  return tiles >= (a.w.kind == CAIFX_W_INT8 ? 90 : 190) && wide_us(a, backward) < tiled_us(a, backward);
}

}  // namespace

// int8 forward with a scale vector and one round of tall tiles (caifx_gemm_tall.hpp), which need no copy: by the estimates, which are
// within 10 % for both from reductions of 2048 on (us, f16 into f16, copy / tall, K = 4096: N = 14336, M = 800 119 / 95, M = 999 119 / 110;
// N = 10240, M = 800 101 / 76, M = 1536 120 / 115; N = 8192, M = 1100 98 / 76; into fp32 by 1.00 to 1.29; over eight weights and
// twelve M it is taken where it is 1.02 to 1.5 times as fast.  With a second round, N = 14336, M = 1100, 139 / 148).  From 769 rows on: below,
// with the same tiles, tests pin which calls make the copy (N = 14336, K = 4096, M = 768 106 / 87).
bool mfma_tall_plain(const GemmArgs &a)
{
  if (a.M <= 768) return false;
  const double us = mfma_tall_plain_us(a);
  return us != 0.0 && wide_shape(a, false) && us < wide_us(a, false) && (!mfma_regw8_takes(a) || us < regw_us(a));
}

size_t mfma_wide_workspace_bytes(const GemmArgs &a, bool backward)
{
  if (!wide_shape(a, backward) || (dense16(a) && !backward)) return 0;
  return static_cast<size_t>(a.offsets ? a.num_experts : 1) * static_cast<size_t>(a.N) * static_cast<size_t>(a.K) * 2;
}

int mfma_wide(const GemmArgs &a, bool backward, hipStream_t s)
{
  if (!wide_shape(a, backward)) return CAIFX_ERR_UNSUPPORTED;
  const bool grouped = a.offsets != nullptr;      // (the tuned kernels take expert weights to be aligned to 16 bytes)
  if (!aligned_to(a.x, 16) || (!grouped && !aligned_to(a.w.q, 16)) || !aligned_to(a.y, 16) || (a.addend && !aligned_to(a.addend, 16))) return CAIFX_ERR_UNSUPPORTED;
  // what the workspace query cannot know: int8 forward with one scale, or with a scale vector that fits its LDS table, has a
  // kernel of its own (one scale, N = 14336, K = 4096, M = 320 59 us there against 75 here, K = 2048, M = 512 41 against 46)
  if (!grouped && !backward && a.w.kind == CAIFX_W_INT8 && mfma_regw8_takes(a) && regw_us(a) < wide_us(a, false)) return CAIFX_ERR_UNSUPPORTED;
  if (!grouped && !backward && mfma_tall_plain(a)) return CAIFX_ERR_UNSUPPORTED;
  WideArgs g{};
  g.a = a.x;
  g.d = a.y;
  g.addend = a.addend;
  g.M = a.M;
  g.C = backward ? a.K : a.N;
  g.R = backward ? a.N : a.K;
  g.d_dtype = a.y_dtype;
  g.b = grouped ? nullptr : a.w.q;
  if (grouped) {
    if (!a.wq_ptrs) return CAIFX_ERR_UNSUPPORTED;
    g.offsets = a.offsets;
    g.wq_ptrs = a.wq_ptrs;
    g.num_experts = a.num_experts;
    g.zero_rest = a.zero_rest;
    mfma_grouped_stamp_target(&g.stamps, &g.stamps_capacity);
  }
  const auto product = [&]() { return a.compute_dtype == CAIFX_BF16 ? pick_form<bf16_t>(g, s) : pick_form<f16_t>(g, s); };
  if (dense16(a) && !backward) return product();
  if (!a.workspace || a.workspace_bytes < mfma_wide_workspace_bytes(a, backward) || !aligned_to(a.workspace, 16)) return CAIFX_ERR_UNSUPPORTED;
  DenseArgs d{};
  d.q = a.w.q;
  d.scales = a.w.scales;
  d.out = a.workspace;
  d.N = a.N;
  d.K = a.K;
  d.M = a.M;
  d.offsets = a.offsets;
  d.wq_ptrs = a.wq_ptrs;
  d.scales_ptrs = a.scales_ptrs;
  int kind = DK_16;
  if (a.w.kind == CAIFX_W_INT4_GROUP) {
    const int gs = a.w.group_size;
    if (gs < 8 || (gs & (gs - 1)) != 0) return CAIFX_ERR_UNSUPPORTED;
    d.group_shift = __builtin_ctz(static_cast<unsigned>(gs));
    kind = DK_INT4;
  } else if (a.w.kind == CAIFX_W_INT8) {
    d.period = (grouped ? a.scales_ptrs != nullptr : a.w.scales != nullptr) ? static_cast<uint32_t>(a.w.scale_period) : 0;
    if (d.period > 1 && (a.w.scale_period % 4 != 0 || a.w.scale_period < 8 || a.w.scale_period > a.N * a.K || (!grouped && !aligned_to(a.w.scales, 16))))
      return CAIFX_ERR_UNSUPPORTED;
    kind = DK_INT8;
  }
  const int experts = grouped ? a.num_experts : 1;
  const int st = a.compute_dtype == CAIFX_BF16 ? launch_dense<bf16_t>(d, kind, backward, experts, s) : launch_dense<f16_t>(d, kind, backward, experts, s);
  if (st != CAIFX_OK) return st;
  g.b = a.workspace;
  return product();
}

}  // namespace caifx
