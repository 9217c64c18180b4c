// Prints the height of the tall kernel's row tiles for calls read from stdin, one a line: rows experts columns reduction.
#include "caifx_gemm_tall_plan.hpp"

#include <cstdio>

int main()
{
  long long M, E, C, R;
  while (std::scanf("%lld %lld %lld %lld", &M, &E, &C, &R) == 4) {
    const caifx::TallPlan p = caifx::plan_tall(M, static_cast<int>(E), C, R);
    std::printf("%d %.3f\n", p.height, p.us);
  }
  return 0;
}
