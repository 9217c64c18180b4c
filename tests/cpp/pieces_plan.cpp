// Prints the plan of the products of bf16 pieces for calls read from stdin, one a line: M C R int4 room; and whether the fp32
// instruction's split tile takes the call instead.
#include "caifx_gemm_pieces_plan.hpp"

#include <cstdio>

int main()
{
  long long M, C, R, int4;
  unsigned long long room;
  while (std::scanf("%lld %lld %lld %lld %llu", &M, &C, &R, &int4, &room) == 5) {
    const caifx::PiecesPlan p = caifx::plan_pieces(M, C, R, int4 != 0, static_cast<size_t>(room));
    std::printf("%d %d %d %zu %d\n", p.bm, p.parts, p.part_steps, p.bytes,
                caifx::split_tile_first(M, C, R, int4 != 0, static_cast<size_t>(room), p) ? 1 : 0);
  }
  return 0;
}
