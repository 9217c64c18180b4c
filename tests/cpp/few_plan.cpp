// Prints how the few-row forward kernel cuts calls read from stdin, one a line: rows columns reduction kind (0 int4, 1 int8 with a scale
// vector, 2 with one scale or none).
#include "caifx_gemm_few_plan.hpp"

#include <cstdio>

int main()
{
  long long M, N, K;
  int kind;
  while (std::scanf("%lld %lld %lld %d", &M, &N, &K, &kind) == 4) {
    const caifx::FewPlan p = caifx::plan_few(M, N, K, kind);
    std::printf("%d %d %d %d\n", p.row_tiles, p.tile_rows / 16, p.parts, p.part_units);
  }
  return 0;
}
