// fp32 compute type over quantised storage on the 16-bit matrix cores: Y[M,N] = X[M,K] * W[N,K]^T and dX[M,K] = dY[M,N] * W[N,K].
//
// An fp32 value is the exact sum of three bf16 pieces (each the rounded remainder of the ones before).  Activations are
// cut into three; a weight, the reference's fp32 code * scale, into three for int8 and into two for int4 (a 4-bit code times
// an 11-bit scale has 15 bits).  The products of pieces are exact in the matrix core and are summed in fp32; left out are those
// below 2^-25 of the largest (middle x last and last x last): six products for int8, five for int4, at 16 times the rate of
// the fp32 instruction.  Error against 64 bits (2-norm, relative; N(0,1) x N(0,0.02)), fp32 instruction -> here: M = 185, N = 3456,
// K = 3712 int4 1.0e-6 -> 1.6e-7, int8 1.1e-6 -> 2.1e-7; M = 256, 8192 x 4096 1.1e-6 -> 3.3e-7 and 3.9e-7; M = 40, 1024 x 512 1.9e-7 ->
// 7.4e-8 and 2.1e-7 -> 9.2e-8.  us, forward / gradient: M = 200, N = 3456, K = 3712, int4 120 / 123 -> 60 / 62; M = 66, 6720 x 3584
// 85 / 235 -> 43 / 42; M = 2048, 4096 x 4096 549 / 570 -> 420 / 403 (int8 590 / 594 -> 496 / 456).
//
// What bounds it with up to a few hundred rows is not the products but cutting the operands (6 to 8 VALU instructions a value,
// a tile of 64 x 64 x 64 as long as its 48 products per wave) and the latency of a step, so two to four workgroups share a
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

// Two values as P pieces each, packed (the first value in the low half).
// A value whose first piece is no number (an infinity, a NaN, or a finite value that bf16 would round to an infinity) turns its
// remainder into NaN, which `odd` collects.
template <int P> __device__ __forceinline__ void cut2(float x0, float x1, uint32_t (&p)[P], float &odd)
{
  p[0] = pack2<bf16_t>(x0, x1);
  float r0 = x0 - low_bf16(p[0]), r1 = x1 - high_bf16(p[0]);
  odd = __builtin_fmaf(r0, 0.0f, __builtin_fmaf(r1, 0.0f, odd));
  p[1] = pack2<bf16_t>(r0, r1);
  if constexpr (P > 2) p[2] = pack2<bf16_t>(r0 - low_bf16(p[1]), r1 - high_bf16(p[1]));
}
// the same for such values.  An infinity or a NaN is its last piece: that one meets no piece but the other operand's first, which
// has the value's sign and is zero only with it (an infinity times a middle piece would be NaN or of the wrong sign).  Finite
// values are cut by truncation.
template <int P> __device__ __forceinline__ void cut2_odd(float x0, float x1, uint32_t (&p)[P])
{
  float x[2] = {x0, x1};
#pragma unroll
  for (int i = 0; i < P; ++i) p[i] = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const bool finite = fabsf(x[h]) <= 3.4028235e38f;
    float rest = x[h];
#pragma unroll
    for (int i = 0; i < P; ++i) {
      uint32_t bits = __builtin_bit_cast(uint32_t, rest) >> 16;
      if (!finite) bits = i < P - 1 ? 0u : (x[h] != x[h] ? 0x7fc0u : bits);
      else rest -= __builtin_bit_cast(float, bits << 16);
      p[i] |= bits << (16 * h);
    }
  }
}
// n values (a multiple of 2) as pieces: out[piece][i] holds values 2 i and 2 i + 1
template <int P, bool kOdd, int n> __device__ __forceinline__ void cut(const float (&x)[n], uint32_t (&out)[P][n / 2], float &odd)
{
#pragma unroll
  for (int i = 0; i < n / 2; ++i) {
    uint32_t p[P];
    if constexpr (kOdd) cut2_odd<P>(x[2 * i], x[2 * i + 1], p);
    else cut2<P>(x[2 * i], x[2 * i + 1], p, odd);
#pragma unroll
    for (int k = 0; k < P; ++k) out[k][i] = p[k];
  }
}

__device__ __forceinline__ int swizzled(int row, int chunk) { return row * 128 + ((chunk ^ ((row ^ (row >> 3)) & 7)) << 4); }

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
  auto store_a = [&](auto odd_path_, float &odd) __attribute__((always_inline)) {
    constexpr bool kOdd = decltype(odd_path_)::value;
#pragma unroll
    for (int i = 0; i < kALoads; ++i) {
      const XT *h = reinterpret_cast<const XT *>(&areg[i]);
      float x[kAV];
#pragma unroll
      for (int e = 0; e < kAV; ++e) x[e] = to_f32<XT>(h[e]);
      uint32_t p[3][kAV / 2];
      cut<3, kOdd>(x, p, odd);
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
  auto store_b = [&](auto odd_path_, float &odd) __attribute__((always_inline)) {
    constexpr bool kOdd = decltype(odd_path_)::value;
    float w[4][4];          // [row][along k]
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
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float x[4] = {kBackward ? w[0][c] : w[c][0], kBackward ? w[1][c] : w[c][1], kBackward ? w[2][c] : w[c][2], kBackward ? w[3][c] : w[c][3]};
      uint32_t p[PW][2];
      cut<PW, kOdd>(x, p, odd);
      const int row = kBackward ? b_col + c : b_row + 16 * c, at = kBackward ? b_row : b_col;
#pragma unroll
      for (int k = 0; k < PW; ++k) {
        u32x2_t v;
        v[0] = p[k][0];
        v[1] = p[k][1];
        *reinterpret_cast<u32x2_t *>(Bs[k] + swizzled(row, at >> 3) + (at & 7) * 2) = v;
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
  load(0);
  for (int s = 0; s < steps; ++s) {
    float odd = 0.0f;
    store_a(std::false_type{}, odd);
    store_b(std::false_type{}, odd);
    if (__ballot(!(odd == 0.0f)) != 0) {          // one branch a step for the whole wave, rarely taken: both operands once more
      store_a(std::true_type{}, odd);
      store_b(std::true_type{}, odd);
    }
    meet();
    load(s + 1);
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
  // up to five 128-deep steps of the fp32 instruction's kernel, whose waves share them, are done before the pieces pay (M = 65,
  // R = 512, C = 2176 10.0 us there, 11.6 here; M = 33 and 8 equal; M = 100 12.7 and 12.1; R = 1024 11.6 and 9.4)
  if (a.M <= 80 && R <= 640 && R % 128 == 0) return false;
  return R >= kPK && R % kPK == 0 && a.K % 16 == 0 && a.M >= 1 && C >= 16 && a.M <= (int64_t{1} << 22) && a.N < (int64_t{1} << 22) && a.K < (int64_t{1} << 22);
}

}  // namespace

size_t pieces_workspace_bytes(const GemmArgs &a, bool backward)
{
  if (!pieces_shape(a, backward)) return 0;
  return plan_pieces(a.M, backward ? a.K : a.N, backward ? a.N : a.K, a.w.kind == CAIFX_W_INT4_GROUP, SIZE_MAX).bytes;
}

int pieces_gemm(const GemmArgs &a, bool backward, hipStream_t s)
{
  if (!pieces_shape(a, backward)) return CAIFX_ERR_UNSUPPORTED;
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
  const int64_t C = backward ? a.K : a.N, R = backward ? a.N : a.K;
  const PiecesPlan plan = plan_pieces(a.M, C, R, int4, a.workspace && aligned_to(a.workspace, 16) ? a.workspace_bytes : 0);
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
  return splitk_reduce(static_cast<const float *>(a.workspace), plan.parts, a.M * C, a.y, a.y_dtype, nullptr, s);
}

}  // namespace caifx
