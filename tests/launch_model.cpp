// For each input line "M N K bits group_size workspace row_identity" (256 CUs):
// "route tile_rows splits unit" of a quantized_matmul call, route 1 for the wide
// kernel (its plan follows) and 0 for the skinny family.
#include <cstdio>

#include "launch.h"

int main() {
  long long M, N, K, bits, gs, ws, rid;
  while (scanf("%lld %lld %lld %lld %lld %lld %lld", &M, &N, &K, &bits, &gs, &ws, &rid) == 7) {
    const bool wide = mq::wide_route(M, N, K, (int)bits, (int)gs, 256, ws != 0, rid != 0);
    const mq::WidePlan p = mq::wide_plan(M, N, K, (int)bits, 256, ws ? 16 : 1);
    printf("%d %d %d %d\n", (int)wide, p.bm, p.splits, mq::wide_unit(K));
  }
  return 0;
}
