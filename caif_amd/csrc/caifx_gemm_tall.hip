// Host side of caifx_gemm_tall.hpp: which calls it takes; its launches in bf16.
#include "caifx_gemm_tall.hpp"
#include <cmath>

namespace caifx {

int tall::launch_bf16(const TallArgs &t, bool backward, hipStream_t s)
{
  return backward ? launch<bf16_t, true>(t, s) : launch<bf16_t, false>(t, s);
}

// The height a segment's tiles may have.  A launch lasts as many tiles one after the other as its fullest compute unit gets, so
// few tiles are made low and many high: in us, a tile of nb blocks of 16 rows takes 3 + 0.33 nb and 0.47 + 0.06 nb per step (the
// dequantisation, two meetings and the way of the requests; then the products, 16 rows 0.055).  Segment lengths are not known here:
// uniformly drawn ids give them a spread of about the square root of their mean, so a further tile is counted by how likely
// it is.  Over 688 launches (2 to 64 experts, 20 to 1200 rows each, 512 to 2048 columns and reductions, both directions) the height
// chosen of 64, 96, 128, 192 and 256 is 0.4 % off the best in the mean, 19 % at most, and the launch 1.16 times as fast as on the
// kernels this one took the calls from (0.67 to 1.0 with 256 everywhere where there are few tiles); five are slower, by 3 to 12 %.
static int tile_height(int64_t M, int experts, int64_t C, int64_t R, double *estimate = nullptr)
{
  const double mean = static_cast<double>(M) / experts, spread = experts > 1 ? 2.5 * std::sqrt(mean > 1.0 ? mean : 1.0) : 1.0;
  const double cols = static_cast<double>((C + tall::BN - 1) / tall::BN) * experts, steps = static_cast<double>(R) / 64;
  int best = tall::BM;
  double best_us = 0.0;
  for (int h = 64; h <= tall::BM; h += 32) {
    double n = 1.0;                      // tiles of a segment
    if (mean > 8.0 * h) {
      n = mean / h + 0.5;
    } else {
      for (double k = h; k < mean + spread; k += h) {
        const double likely = (mean - k) / spread + 0.5;
        n += likely < 0.0 ? 0.0 : likely > 1.0 ? 1.0 : likely;
      }
    }
    // the highest tile: of a segment that is cut once less than most
    const double whole = mean / std::floor(n + 0.1);
    double nb = 2.0 * std::ceil((whole < h ? whole : h) / 32.0);
    nb = nb < 4.0 ? 4.0 : nb;
    const double rounds = cols * n / 256.0;
    const double us = (rounds < 1.0 ? 1.0 : rounds < 4.0 ? std::ceil(rounds - 0.02) : rounds + 0.5) * (3.0 + 0.33 * nb + steps * (0.47 + 0.06 * nb));
    if (h == 64 || us <= best_us) {      // of equals the highest: a segment longer than expected is no tile more
      best = h;
      best_us = us;
    }
  }
  if (estimate) *estimate = best_us;
  return best;
}

// Classes of weight rows with the same scales along k; 0 where the kernel does not take the sizes.
static int tall_classes(const GemmArgs &a, bool backward)
{
  if (a.K % 128 != 0 || a.K < 256 || a.K > (int64_t{1} << 22) || a.N % (backward ? 128 : 64) != 0 || a.N < 256 || a.N > (int64_t{1} << 22) ||
      a.N * a.K >= (int64_t{1} << 32) || a.M < 1 || a.M > (int64_t{1} << 30))
    return 0;
  const int64_t P = a.w.scale_period;
  if (P % 4 != 0 || P < 64 || P > (int64_t{1} << 24)) return 0;
  int64_t len = P;
  for (int64_t r = a.K % P; r != 0;) {
    const int64_t t2 = len % r;
    len = r;
    r = t2;
  }
  const int64_t V = P / len;
  return V > tall::kMaxClasses ? 0 : static_cast<int>(V);
}

// One round of tiles with one weight (forward): 0 if it would be more, or is not for this kernel.
double mfma_tall_plain_us(const GemmArgs &a)
{
  if (a.offsets || a.epilogue != 0 || a.w.kind != CAIFX_W_INT8 || a.compute_dtype == CAIFX_F32 || a.x_dtype != a.compute_dtype || !a.w.scales) return 0.0;
  if (tall_classes(a, false) == 0 || !aligned_to(a.w.q, 16) || !aligned_to(a.w.scales, 16)) return 0.0;
  double us;
  const int height = tile_height(a.M, 1, a.N, a.K, &us);
  if ((a.M + height - 1) / height * ((a.N + tall::BN - 1) / tall::BN) > 256) return 0.0;
  return us + 8.0;       // the launch's ends
}

int mfma_tall(const GemmArgs &a, bool backward, hipStream_t s)
{
  if (!a.offsets) {
    if (backward || !mfma_tall_plain(a)) return CAIFX_ERR_UNSUPPORTED;
  } else if (a.w.kind != CAIFX_W_INT8 || !a.wq_ptrs || !a.scales_ptrs || a.num_experts < 1) {
    return CAIFX_ERR_UNSUPPORTED;
  }
  if (a.compute_dtype == CAIFX_F32 || a.x_dtype != a.compute_dtype) return CAIFX_ERR_UNSUPPORTED;
  if (!aligned_to(a.x, 16) || !aligned_to(a.y, 16) || (a.addend && !aligned_to(a.addend, 16))) return CAIFX_ERR_UNSUPPORTED;
  if (a.epilogue != 0) {
    if (a.addend || a.y_dtype == CAIFX_F32 || a.epilogue != (backward ? 2 : 1) || !a.e1 || !a.y2 || !aligned_to(a.e1, 16) || !aligned_to(a.y2, 16) ||
        (backward && (!a.e2 || !aligned_to(a.e2, 16))))
      return CAIFX_ERR_UNSUPPORTED;
  }
  const int V = tall_classes(a, backward);
  if (V == 0) return CAIFX_ERR_UNSUPPORTED;

  tall::TallArgs t{};
  t.M = a.M;
  t.N = a.N;
  t.K = a.K;
  t.a = a.x;
  t.d = a.y;
  t.d_dtype = a.y_dtype;
  t.addend = a.addend;
  t.epilogue = a.epilogue;
  t.e1 = a.e1;
  t.e2 = a.e2;
  t.d2 = a.y2;
  t.offsets = a.offsets;
  t.wq_ptrs = a.wq_ptrs;
  t.scales_ptrs = a.scales_ptrs;
  t.num_experts = a.offsets ? a.num_experts : 0;
  t.zero_rest = a.offsets && a.zero_rest;
  if (!a.offsets) {
    t.wq = a.w.q;
    t.scales = a.w.scales;
  }
  t.height = tile_height(a.M, a.offsets ? a.num_experts : 1, backward ? a.K : a.N, backward ? a.N : a.K);
  t.period = static_cast<uint32_t>(a.w.scale_period);
  t.classes = V;
  if (a.offsets) mfma_grouped_stamp_target(&t.stamps, &t.stamps_capacity);
  return a.compute_dtype == CAIFX_BF16 ? tall::launch_bf16(t, backward, s) : tall::launch_f16(t, backward, s);
}

}  // namespace caifx
