// fp32 compute type over quantised storage on the 16-bit matrix cores: Y[M,N] = X[M,K] * W[N,K]^T and dX[M,K] = dY[M,N] * W[N,K].
//
// An fp32 value is the exact sum of three bf16 pieces (each the rounded remainder of the ones before).  Activations are
// cut into three; a weight, the reference's fp32 code * scale, into three for int8 and into two for int4 (a 4-bit code times
// an 11-bit scale has 15 bits).  The products of pieces are exact in the matrix core and are summed in fp32; left out are those
// below 2^-25 of the largest (middle x last and last x last): six products for int8, five for int4, at 16 times the rate of
// the fp32 instruction.  Error against 64 bits (2-norm, relative; N(0,1) x N(0,0.02)), fp32 instruction -> here: M = 185, N = 3456,
// K = 3712 int4 1.0e-6 -> 1.6e-7, int8 1.1e-6 -> 2.1e-7; M = 256, 8192 x 4096 1.1e-6 -> 3.3e-7 and 4.0e-7; M = 40, N = 1024, K = 512, gradient
// 2.7e-7 -> 7.6e-8 and 2.9e-7 -> 8.9e-8.  us, forward / gradient (int8 in brackets): M = 200, N = 3456, K = 3712 118 / 121 -> 55 / 60
// (124 / 129 -> 65 / 67); M = 66, 6720 x 3584 81 / 231 -> 52 / 51 (88 / 244 -> 54 / 58); M = 256, 8192 x 4096 189 / 277 -> 130 / 132 (199 / 296 ->
// 152 / 146); M = 2048, 4096 x 4096 540 / 563 -> 402 / 404 (561 / 579 -> 440 / 438).
//
// What bounds it with up to a few hundred rows is not the products but cutting the operands (6 to 8 VALU instructions a value, a
// tile of 64 x 64 x 64 as long as its 48 products per wave) and the latency of a step: at M = 200 the VALU is busy 0.40 to 0.44 of the time,
// the matrix pipes 0.17 to 0.19, waves wait 0.3 of theirs (M = 2048: 0.50, 0.33 to 0.37, 0.23 to 0.31).  So two to four workgroups share a
// compute unit and take turns, and the reduction is shared out until they do: `parts` workgroups write fp32 sums to the
// caller's workspace, a second launch adds them in order.
//
// Tiles of BM x 64, 64 deep; 256 threads.  Wave (wm, wn) multiplies the 16-row blocks 2 i + wm with columns 32 wn .. + 31; blocks
// without rows are left out.  The operands lie in LDS as rows of 64 reduction elements per piece, 16-byte chunks swizzled
// with (row ^ row >> 3) & 7.  The loads of the next step are in flight beside the products of this one.
#include "caifx_internal.hpp"
#include "caifx_gemm_pieces_plan.hpp"

#include <type_traits>

namespace caifx {
namespace {

struct PiecesArgs {
  const void *a;         // activations [M, R]
  void *d;               // result [M, C], or fp32 sums [parts][M][C]
  const uint8_t *wq;
  const void *scales;
  int64_t M, N, K;
  int64_t period;        // int8: 0 = no scales, 1 = one scale, otherwise the length of the scale vector (>= 64, % 4 == 0)
  int d_dtype;
  int group_shift;       // int4: log2(group_size), group_size >= 16
  uint32_t step;         // int8 scale vector: how far the scale index moves per step, modulo period
  int parts, part_steps; // blockIdx.z is the part
  int bm;                // rows of a tile (launch only)
};

__device__ __forceinline__ void store_result(void *p, int dt, int64_t i, float v)
{
  if (dt == CAIFX_BF16) static_cast<bf16_t *>(p)[i] = from_f32<bf16_t>(v);
  else if (dt == CAIFX_F16) static_cast<f16_t *>(p)[i] = from_f32<f16_t>(v);
  else static_cast<float *>(p)[i] = v;
}

__device__ __forceinline__ float low_bf16(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float high_bf16(uint32_t p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

// Pieces are the value where it is zero or its magnitude lies in these ranges.  Below, a piece or a product of first and last pieces
// would be a subnormal number (2^-64 * 2^-38 = 2^-102, its last bits 2^-125); above, sums of fewer than 2^22 products could pass the
// largest number in acc and its negative in rest.  Weights are held to theirs by their scales (int8 codes: zero, or 2^-38 to 2^43; every
// finite fp16 scale does).  A step of a tile that meets another value (an infinity, a NaN, one too large or too small) runs on the fp32
// instruction, with the results that one gives.  What the looking costs: 1 % (int4 628 calls, geometric mean; int8 M = 200 to 2048),
// up to 3 more where zero activations make every step look twice (half of them zero) and 6 where zero scales do (M = 2048, 4096 x 4096,
// gradient 462 us with a zero scale, 438 without; held to be too small they took 1147).  M = 200, N = 3456, K = 3712 takes 62 (int4) and
// 67 us (int8) with ordinary values, the same with one tiny value in a million, and 157 and 163 where all are tiny.
constexpr float kLeastX = 0x1p-64f, kMostX = 0x1p50f;
constexpr float kLeastS = 0x1p-38f, kMostS = 0x1p43f;

// the smallest and the largest magnitude of what a thread has seen of a step (NaN from a NaN on): half an instruction a value each
struct Seen {
  float least, most;
};
__device__ __forceinline__ void see(Seen &o, float v)
{
  o.least = __builtin_elementwise_minimum(o.least, fabsf(v));
  o.most = __builtin_elementwise_maximum(o.most, fabsf(v));
}

// Two values as P pieces each, packed (the first value in the low half)
template <int P> __device__ __forceinline__ void cut2(float x0, float x1, uint32_t (&p)[P])
{
  p[0] = pack2<bf16_t>(x0, x1);
  const float r0 = x0 - low_bf16(p[0]), r1 = x1 - high_bf16(p[0]);
  p[1] = pack2<bf16_t>(r0, r1);
  if constexpr (P > 2) p[2] = pack2<bf16_t>(r0 - low_bf16(p[1]), r1 - high_bf16(p[1]));
}
// n values (a multiple of 2) as pieces: out[piece][i] holds values 2 i and 2 i + 1
template <int P, int n> __device__ __forceinline__ void cut(const float (&x)[n], uint32_t (&out)[P][n / 2])
{
#pragma unroll
  for (int i = 0; i < n / 2; ++i) {
    uint32_t p[P];
    cut2<P>(x[2 * i], x[2 * i + 1], p);
#pragma unroll
    for (int k = 0; k < P; ++k) out[k][i] = p[k];
  }
}

__device__ __forceinline__ int swizzled(int row, int chunk) { return row * 128 + ((chunk ^ ((row ^ (row >> 3)) & 7)) << 4); }
// the same for rows of 64 fp32 values (a step on the fp32 instruction)
__device__ __forceinline__ int swizzled32(int row, int chunk) { return row * 256 + ((chunk ^ (row & 15)) << 4); }

// kVec: int8 with a scale vector
template <typename XT, bool kInt4, bool kVec, bool kBackward, int BM>
__global__ __launch_bounds__(256, BM == 128 ? 2 : 3) void pieces_gemm_kernel(PiecesArgs g)
{
  constexpr int PW = kInt4 ? 2 : 3;        // pieces of a weight
  constexpr int kAV = 16 / sizeof(XT);     // activations per 16-byte load (4 or 8)
  constexpr int kARows = 256 * kAV / kPK;  // rows that one load of the workgroup covers (16 or 32)
  constexpr int kALoads = BM / kARows;
  constexpr int TM = BM / 32;              // 16-row blocks of a wave
  __shared__ __attribute__((aligned(16))) unsigned char As[3][BM * 128];
  __shared__ __attribute__((aligned(16))) unsigned char Bs[PW][kPN * 128];
  __shared__ int fp32_step;                // the last step (from 1 on) in which a wave met a value that the pieces do not hold

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int r16 = lane & 15, kq = lane >> 4;
  const int64_t R = kBackward ? g.N : g.K, C = kBackward ? g.K : g.N;
  const int64_t row0 = static_cast<int64_t>(blockIdx.y) * BM, col0 = static_cast<int64_t>(blockIdx.x) * kPN;
  const int first = static_cast<int>(blockIdx.z) * g.part_steps;
  const int all = static_cast<int>(R / kPK);
  const int steps = all - first < g.part_steps ? all - first : g.part_steps;
  const int rows = static_cast<int>(g.M - row0 < BM ? g.M - row0 : BM);
  const int blocks = (rows + 15) >> 4;
  const int mine = (blocks + 1 - wm) >> 1;                       // 16-row blocks of this wave that hold rows

  // ---- activations: 16 bytes of rows a_row + kARows i, whole lines per instruction
  const int a_row = t / (kPK / kAV), a_col = (t % (kPK / kAV)) * kAV;
  const unsigned char *a_base = static_cast<const unsigned char *>(g.a) + (row0 * R + static_cast<int64_t>(first) * kPK) * sizeof(XT);
  uint32_t a_off[kALoads];                 // (128 rows of less than 2^22 elements: host)
#pragma unroll
  for (int i = 0; i < kALoads; ++i) {
    const int r = a_row + kARows * i;
    a_off[i] = (static_cast<uint32_t>(r < rows ? r : rows - 1) * static_cast<uint32_t>(R) + a_col) * sizeof(XT);
  }
  u32x4_t areg[kALoads];
  auto load_a = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kALoads; ++i)
      areg[i] = *reinterpret_cast<const u32x4_t *>(a_base + static_cast<int64_t>(s) * (kPK * sizeof(XT)) + a_off[i]);
  };
  // A zero is ordinary, another number below kLeastX is not (fp16 holds none).  The bits without the sign, less one: a zero becomes the
  // largest, and a minimum of three is one instruction (two comparisons a value and their masks cost 10 % of a call with zeros).
  auto tiny_a = [&]() __attribute__((always_inline)) {
    uint32_t least = 0xffffffffu;
    if constexpr (!std::is_same<XT, f16_t>::value) {
#pragma unroll
      for (int i = 0; i < kALoads; ++i) {
        const XT *h = reinterpret_cast<const XT *>(&areg[i]);
#pragma unroll
        for (int e = 0; e < kAV; ++e) {
          const uint32_t b = (__builtin_bit_cast(uint32_t, to_f32<XT>(h[e])) << 1) - 1u;
          least = b < least ? b : least;
        }
      }
    }
    return least < (__builtin_bit_cast(uint32_t, kLeastX) << 1) - 1u;
  };
  auto store_a = [&](Seen &seen) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kALoads; ++i) {
      const XT *h = reinterpret_cast<const XT *>(&areg[i]);
      float x[kAV];
#pragma unroll
      for (int e = 0; e < kAV; ++e) {
        x[e] = to_f32<XT>(h[e]);
        see(seen, x[e]);
      }
      uint32_t p[3][kAV / 2];
      cut<3>(x, p);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        unsigned char *to = As[k] + swizzled(a_row + kARows * i, a_col >> 3) + (a_col & 7) * 2;
        if constexpr (kAV == 8) {
          u32x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = p[k][e];
          *reinterpret_cast<u32x4_t *>(to) = v;
        } else {
          u32x2_t v;
          v[0] = p[k][0];
          v[1] = p[k][1];
          *reinterpret_cast<u32x2_t *>(to) = v;
        }
      }
    }
  };
  // ---- weights: four codes along k of four rows per thread and step.
  // forward: rows n = col0 + t / 16 + 16 r, k = 4 (t % 16) ..; gradient: rows n = 4 (t / 16) + r of the step, columns col0 + 4 (t % 16) ..
  const int b_row = kBackward ? 4 * (t >> 4) : t >> 4, b_col = 4 * (t & 15);
  // flat index of the tile's first code at a step (the same in every lane), and of each row's first code from there
  const int64_t flat0 = kBackward ? static_cast<int64_t>(first) * kPK * g.K + col0 : col0 * g.K + static_cast<int64_t>(first) * kPK;
  const int64_t flat_step = kBackward ? kPK * g.K : kPK;
  uint32_t off[4];                         // (64 rows of less than 2^22 codes: host)
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if constexpr (kBackward) {
      const int64_t k = col0 + b_col + 4 <= g.K ? b_col : g.K - 4 - col0;            // columns past the end are never stored
      off[r] = static_cast<uint32_t>((b_row + r) * g.K + k);
    } else {
      const int64_t n = col0 + b_row + 16 * r < g.N ? b_row + 16 * r : g.N - 1 - col0;
      off[r] = static_cast<uint32_t>(n * g.K + b_col);
    }
  }
  const float *s32 = static_cast<const float *>(g.scales);
  const f16_t *s16 = static_cast<const f16_t *>(g.scales);
  const uint32_t period = static_cast<uint32_t>(g.period);
  const float s_one = (!kInt4 && g.period == 1) ? s32[0] : 1.0f;
  uint32_t sidx[4];       // scale index of the first code of each row
  if constexpr (kVec) {
#pragma unroll
    for (int r = 0; r < 4; ++r) sidx[r] = static_cast<uint32_t>((flat0 + off[r]) % g.period);
  }
  uint32_t wreg[4];
  float sc[4][kVec ? 4 : 1];
  auto load_b = [&](int s) __attribute__((always_inline)) {
    const int64_t f0 = flat0 + static_cast<int64_t>(s) * flat_step;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (kInt4) {
        wreg[r] = *reinterpret_cast<const uint16_t *>(g.wq + (f0 >> 1) + (off[r] >> 1));          // both are even
        sc[r][0] = to_f32(s16[(f0 + off[r]) >> g.group_shift]);
      } else {
        wreg[r] = *reinterpret_cast<const uint32_t *>(g.wq + f0 + off[r]);
      }
      if constexpr (kVec) {
        // four scales never straddle the wrap: indices and period are multiples of 4
        const floatx4_t v4 = *reinterpret_cast<const floatx4_t *>(s32 + sidx[r]);
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[r][e] = v4[e];
      }
    }
  };
  auto next_scales = [&]() __attribute__((always_inline)) {
    if constexpr (kVec) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sidx[r] += g.step;
        if (sidx[r] >= period) sidx[r] -= period;
      }
    }
  };
  auto weights = [&](float (&w)[4][4]) __attribute__((always_inline)) {          // [row][along k]
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (kInt4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) w[r][e] = static_cast<float>(static_cast<int>(wreg[r] << (28 - 4 * e)) >> 28) * sc[r][0];
      } else {
        float q[4];
        int8x4_to_f32(wreg[r], q);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[r][e] = q[e] * (kVec ? sc[r][kVec ? e : 0] : s_one);
      }
    }
  };
  // the same question of the scales (those of a channel of zeros may be zero)
  auto tiny_s = [&]() __attribute__((always_inline)) {
    uint32_t least = 0xffffffffu;
    if constexpr (kVec) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t b = (__builtin_bit_cast(uint32_t, sc[r][kVec ? e : 0]) << 1) - 1u;
          least = b < least ? b : least;
        }
    }
    return least < (__builtin_bit_cast(uint32_t, kLeastS) << 1) - 1u;
  };
  // four weights along the reduction, and the row and the reduction element in LDS where they begin
  const int b_at = kBackward ? b_row : b_col;
  auto b_lds_row = [&](int c) __attribute__((always_inline)) { return kBackward ? b_col + c : b_row + 16 * c; };
  auto store_b = [&](Seen &seen) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (kInt4 || kVec) {
#pragma unroll
        for (int e = 0; e < (kVec ? 4 : 1); ++e) see(seen, sc[r][e]);
      }
    }
    float w[4][4];
    weights(w);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float x[4] = {kBackward ? w[0][c] : w[c][0], kBackward ? w[1][c] : w[c][1], kBackward ? w[2][c] : w[c][2], kBackward ? w[3][c] : w[c][3]};
      uint32_t p[PW][2];
      cut<PW>(x, p);
#pragma unroll
      for (int k = 0; k < PW; ++k) {
        u32x2_t v;
        v[0] = p[k][0];
        v[1] = p[k][1];
        *reinterpret_cast<u32x2_t *>(Bs[k] + swizzled(b_lds_row(c), b_at >> 3) + (b_at & 7) * 2) = v;
      }
    }
  };
  // A step's operands as fp32 values in the place of the pieces: read from memory again and in rolled loops, so that this rare
  // path takes no registers from the other.
  auto store_fp32 = [&](int s) __attribute__((always_inline)) {
    const XT *a0 = reinterpret_cast<const XT *>(a_base) + static_cast<int64_t>(s) * kPK + a_col;
#pragma unroll 1
    for (int r = a_row; r < BM; r += kARows) {
      const XT *from = a0 + static_cast<int64_t>(r < rows ? r : rows - 1) * R;
#pragma unroll
      for (int c = 0; c < kAV / 4; ++c) {
        floatx4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = to_f32<XT>(from[4 * c + e]);
        *reinterpret_cast<floatx4_t *>(As[0] + swizzled32(r, (a_col >> 2) + c)) = v;
      }
    }
#pragma unroll 1
    for (int r = 0; r < 4; ++r) {
      int64_t f = flat0 + static_cast<int64_t>(s) * flat_step;
      if constexpr (kBackward) f += (b_row + r) * g.K + (col0 + b_col + 4 <= g.K ? b_col : g.K - 4 - col0);
      else f += (col0 + b_row + 16 * r < g.N ? b_row + 16 * r : g.N - 1 - col0) * g.K + b_col;
      floatx4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (kInt4) v[e] = static_cast<float>(static_cast<int>(static_cast<uint32_t>(g.wq[(f + e) >> 1]) << (28 - 4 * (e & 1))) >> 28) * to_f32(s16[f >> g.group_shift]);
        else v[e] = static_cast<float>(static_cast<const int8_t *>(static_cast<const void *>(g.wq))[f + e]) * (kVec ? s32[f % g.period + e] : s_one);
      }
      if constexpr (kBackward) {
#pragma unroll
        for (int e = 0; e < 4; ++e) *reinterpret_cast<float *>(Bs[0] + swizzled32(b_col + e, b_row >> 2) + 4 * r) = v[e];
      } else {
        *reinterpret_cast<floatx4_t *>(Bs[0] + swizzled32(b_row + 16 * r, b_col >> 2)) = v;
      }
    }
  };

  // the products of first pieces and the rest of them, 2^8 smaller, apart: a sum is rounded once per 32 reduction elements instead
  // of five or six times
  floatx4_t acc[TM][2], rest[TM][2];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = rest[i][j] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // only LDS passes between the waves: __syncthreads() would also wait for the loads in flight
  auto meet = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  // a step past the end reads the last one again; its registers are never stored
  auto load = [&](int s) __attribute__((always_inline)) {
    const int at = s < steps ? s : steps - 1;
    load_a(at);
    load_b(at);
    next_scales();
  };
  // one scale for the weight (or none) is held to its range here
  const unsigned long long one_scale_odd = !kInt4 && !kVec && s_one != 0.0f && !(fabsf(s_one) >= kLeastS && fabsf(s_one) < kMostS);
  load(0);
  if (t == 0) fp32_step = 0;
  meet();
  for (int s = 0; s < steps; ++s) {
    Seen xs{kMostX, 0.0f}, ss{kMostS, kLeastS};
    store_a(xs);
    store_b(ss);
    unsigned long long odd = __ballot(!(xs.most < kMostX)) | one_scale_odd;          // (masks: no lane of the wave leaves the straight line)
    if constexpr (kInt4) odd |= __ballot(!(ss.most <= 65504.0f));
    if constexpr (kVec) odd |= __ballot(!(ss.most < kMostS));
    unsigned long long zero_or_tiny = 0;
    if constexpr (!std::is_same<XT, f16_t>::value) zero_or_tiny = __ballot(!(xs.least >= kLeastX));
    if constexpr (kVec) zero_or_tiny |= __ballot(!(ss.least >= kLeastS));
    if ((odd | zero_or_tiny) != 0) {                    // which of the two is asked only where there is one
      if ((odd | __ballot(tiny_a() | tiny_s())) != 0) fp32_step = s + 1;
    }
    meet();
    const int flagged = fp32_step;          // (written again after this step's last barrier)
    load(s + 1);
    if (__builtin_amdgcn_readfirstlane(flagged) == s + 1) {      // the same for the whole workgroup, rare
      store_fp32(s);
      meet();
#pragma unroll 1
      for (int c = 0; c < 4; ++c) {                              // lane (r16, kq) holds reduction elements 16 c + 4 kq + e in both operands
        floatx4_t b[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) b[j] = *reinterpret_cast<const floatx4_t *>(Bs[0] + swizzled32(32 * wn + 16 * j + r16, 4 * c + kq));
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          if (i >= mine) break;
          const floatx4_t a = *reinterpret_cast<const floatx4_t *>(As[0] + swizzled32(16 * (2 * i + wm) + r16, 4 * c + kq));
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[j][e], acc[i][j], 0, 0, 0);
        }
      }
      meet();
      // the pieces' products then add nothing
      const u32x4_t none = {0, 0, 0, 0};
#pragma unroll 1
      for (int b = 16 * t; b < static_cast<int>(sizeof(As)); b += 16 * 256) *reinterpret_cast<u32x4_t *>(As[0] + b) = none;
#pragma unroll 1
      for (int b = 16 * t; b < static_cast<int>(sizeof(Bs)); b += 16 * 256) *reinterpret_cast<u32x4_t *>(Bs[0] + b) = none;
      meet();
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8_t b[PW][2];
#pragma unroll
      for (int k = 0; k < PW; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j) b[k][j] = *reinterpret_cast<const bf16x8_t *>(Bs[k] + swizzled(32 * wn + 16 * j + r16, 4 * kk + kq));
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (i >= mine) break;                                    // the same for every lane of the wave
        bf16x8_t a[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) a[k] = *reinterpret_cast<const bf16x8_t *>(As[k] + swizzled(16 * (2 * i + wm) + r16, 4 * kk + kq));
#pragma unroll
        for (int sum = 2; sum >= 0; --sum)
#pragma unroll
          for (int k = 0; k < PW; ++k) {
            const int ka = sum - k;
            if (ka < 0) continue;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              floatx4_t &to = sum == 0 ? acc[i][j] : rest[i][j];
              to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ka], b[k][j], to, 0, 0, 0);
            }
          }
      }
    }
    meet();              // the next step overwrites both operands
  }

  // acc[i][j][r]: row 16 (2 i + wm) + 4 kq + r, column 32 wn + 16 j + r16
  const int64_t base = static_cast<int64_t>(blockIdx.z) * g.M * C;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t col = col0 + 32 * wn + 16 * j + r16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * (2 * i + wm) + 4 * kq + r;
        if (row < rows && col < C) store_result(g.d, g.d_dtype, base + (row0 + row) * C + col, acc[i][j][r] + rest[i][j][r]);
      }
    }
}

template <typename XT, bool kInt4, bool kVec, bool kBackward>
int launch_pieces(const PiecesArgs &g, hipStream_t s)
{
  const int64_t C = kBackward ? g.K : g.N;
  const unsigned cols = static_cast<unsigned>((C + kPN - 1) / kPN), parts = static_cast<unsigned>(g.parts);
  const auto grid = [&](int bm) { return dim3(cols, static_cast<unsigned>((g.M + bm - 1) / bm), parts); };
  if (g.bm == 32) hipLaunchKernelGGL((pieces_gemm_kernel<XT, kInt4, kVec, kBackward, 32>), grid(32), dim3(256), 0, s, g);
  else if (g.bm == 64) hipLaunchKernelGGL((pieces_gemm_kernel<XT, kInt4, kVec, kBackward, 64>), grid(64), dim3(256), 0, s, g);
  else hipLaunchKernelGGL((pieces_gemm_kernel<XT, kInt4, kVec, kBackward, 128>), grid(128), dim3(256), 0, s, g);
  return launch_status();
}

template <typename XT> int launch_kind(const PiecesArgs &g, bool int4, bool backward, hipStream_t s)
{
  if (int4) return backward ? launch_pieces<XT, true, false, true>(g, s) : launch_pieces<XT, true, false, false>(g, s);
  if (g.period > 1) return backward ? launch_pieces<XT, false, true, true>(g, s) : launch_pieces<XT, false, true, false>(g, s);
  return backward ? launch_pieces<XT, false, false, true>(g, s) : launch_pieces<XT, false, false, false>(g, s);
}

bool pieces_shape(const GemmArgs &a, bool backward)
{
  if (a.compute_dtype != CAIFX_F32 || a.offsets || a.addend || a.epilogue) return false;
  if (a.w.kind != CAIFX_W_INT8 && a.w.kind != CAIFX_W_INT4_GROUP) return false;
  const int64_t R = backward ? a.N : a.K, C = backward ? a.K : a.N;
  return R >= kPK && R % kPK == 0 && a.K % 16 == 0 && a.M >= 1 && C >= 16 && a.M <= (int64_t{1} << 22) && a.N < (int64_t{1} << 22) && a.K < (int64_t{1} << 22);
}

// the plan of a call; without tiles where the fp32 instruction's kernel takes it, and sooner
PiecesPlan plan_of(const GemmArgs &a, bool backward, size_t room)
{
  const int64_t C = backward ? a.K : a.N, R = backward ? a.N : a.K;
  const bool int4 = a.w.kind == CAIFX_W_INT4_GROUP;
  const PiecesPlan plan = plan_pieces(a.M, C, R, int4, room);
  return a.K % 32 == 0 && split_tile_first(a.M, C, R, int4, room, plan) ? PiecesPlan{} : plan;
}

}  // namespace

size_t pieces_workspace_bytes(const GemmArgs &a, bool backward)
{
  return pieces_shape(a, backward) ? plan_of(a, backward, SIZE_MAX).bytes : 0;
}

int pieces_gemm(const GemmArgs &a, bool backward, hipStream_t s)
{
  if (!pieces_shape(a, backward)) return CAIFX_ERR_UNSUPPORTED;
  const PiecesPlan plan = plan_of(a, backward, a.workspace && aligned_to(a.workspace, 16) ? a.workspace_bytes : 0);
  if (plan.bm == 0) return CAIFX_ERR_UNSUPPORTED;
  if (!aligned_to(a.x, 16) || !aligned_to(a.w.q, 16)) return CAIFX_ERR_UNSUPPORTED;
  PiecesArgs g{};
  g.a = a.x;
  g.d = a.y;
  g.wq = static_cast<const uint8_t *>(a.w.q);
  g.scales = a.w.scales;
  g.M = a.M;
  g.N = a.N;
  g.K = a.K;
  g.d_dtype = a.y_dtype;
  const bool int4 = a.w.kind == CAIFX_W_INT4_GROUP;
  if (int4) {
    const int gs = a.w.group_size;
    if (!a.w.scales || gs < 16 || (gs & (gs - 1)) != 0) return CAIFX_ERR_UNSUPPORTED;     // 16 codes of a thread share a scale
    g.group_shift = __builtin_ctz(static_cast<unsigned>(gs));
  } else if (a.w.scales) {
    g.period = a.w.scale_period;
    if (g.period > 1) {
      if (g.period < kPK || g.period % 4 != 0 || g.period > (int64_t{1} << 30) || !aligned_to(a.w.scales, 16)) return CAIFX_ERR_UNSUPPORTED;
      g.step = static_cast<uint32_t>((backward ? static_cast<int64_t>(kPK) * a.K : kPK) % g.period);
    }
  }
  const bool shared = plan.parts > 1;
  g.bm = plan.bm;
  g.parts = plan.parts;
  g.part_steps = plan.part_steps;
  if (shared) {
    g.d = a.workspace;
    g.d_dtype = CAIFX_F32;
  }
  int st;
  if (a.x_dtype == CAIFX_F32) st = launch_kind<float>(g, int4, backward, s);
  else if (a.x_dtype == CAIFX_BF16) st = launch_kind<bf16_t>(g, int4, backward, s);
  else if (a.x_dtype == CAIFX_F16) st = launch_kind<f16_t>(g, int4, backward, s);
  else return CAIFX_ERR_UNSUPPORTED;
  if (!shared || st != CAIFX_OK) return st;
  return splitk_reduce(static_cast<const float *>(a.workspace), plan.parts, a.M * (backward ? a.K : a.N), a.y, a.y_dtype, nullptr, s);
}

}  // namespace caifx
