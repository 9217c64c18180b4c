// caifx_gemm_tall.hpp: its launches in fp16.
#include "caifx_gemm_tall.hpp"

namespace caifx {

int tall::launch_f16(const TallArgs &t, bool backward, hipStream_t s)
{
  return backward ? launch<f16_t, true>(t, s) : launch<f16_t, false>(t, s);
}

}  // namespace caifx
