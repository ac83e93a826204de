// Host choices of the library, one question a line on stdin:
//   gemm M N K CUS       -> tile shape (nb), K splits, work items
//   attention NQ HEADS NK CUS -> 1 (split over the keys) or 0
#include <cstdio>
#include <cstring>

#include "attn_plan.h"
#include "gemm_launch.h"

int main() {
  char what[16];
  long long a, b, c, cus;
  while (std::scanf("%15s %lld %lld %lld %lld", what, &a, &b, &c, &cus) == 5) {
    if (std::strcmp(what, "gemm") == 0) {
      const w8a8::GemmPlan p = w8a8::gemm_plan(a, b, c, (int)cus);
      std::printf("%d %d %lld\n", p.nb, p.ksplit, (long long)w8a8::plan_tiles(a, b, p) * p.ksplit);
    } else {
      std::printf("%d\n", (int)w8a8::split_wins(a, b, (c + 127) / 128, cus));
    }
  }
}
