// Host side of caifx_gemm_tall.hpp: which calls it takes; its launches in bf16.
#include "caifx_gemm_tall.hpp"

namespace caifx {

int tall::launch_bf16(const TallArgs &t, bool backward, hipStream_t s)
{
  return backward ? launch<bf16_t, true>(t, s) : launch<bf16_t, false>(t, s);
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
  const TallPlan plan = plan_tall(a.M, 1, a.N, a.K);
  if ((a.M + plan.height - 1) / plan.height * ((a.N + tall::BN - 1) / tall::BN) > 256) return 0.0;
  return plan.us + 8.0;       // the launch's ends
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
  t.height = plan_tall(a.M, a.offsets ? a.num_experts : 1, backward ? a.K : a.N, backward ? a.N : a.K).height;
  t.period = static_cast<uint32_t>(a.w.scale_period);
  t.classes = V;
  if (a.offsets) mfma_grouped_stamp_target(&t.stamps, &t.stamps_capacity);
  return a.compute_dtype == CAIFX_BF16 ? tall::launch_bf16(t, backward, s) : tall::launch_f16(t, backward, s);
}

}  // namespace caifx
