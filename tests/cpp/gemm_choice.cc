// Reads products "batch m n k a_column_major b_column_major aligned scratch copies" from standard input and
// prints the kernel each is given: route, copies, tile and k ranges.
#include "f16_gemm_choice.h"

#include <cstdio>

int main() {
  using namespace mi355;
  int b, m, n, k, a_cm, b_cm, aligned;
  unsigned long long scratch, copies;
  while (std::scanf("%d %d %d %d %d %d %d %llu %llu", &b, &m, &n, &k, &a_cm, &b_cm, &aligned, &scratch, &copies) == 9) {
    GemmChoice const c = choose_gemm({b, m, n, k, a_cm != 0, b_cm != 0, aligned != 0, (size_t)scratch, (size_t)copies});
    char const *routes[] = {"tiles", "big", "elements"};
    GemmTile const &t = (a_cm && !c.copy_a ? kGemmTilesColumnMajorA : kGemmTiles)[c.tile];
    std::printf("%s %d %d %d %d %d %d %.2f\n", routes[c.route], c.copy_a, c.copy_b, (int)t.kind, t.bm, t.bn, c.ksplit, c.us);
  }
  return 0;
}
