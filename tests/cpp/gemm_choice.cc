// Reads products "batch m n k a_column_major b_column_major aligned scratch copies" from standard input and
// prints the kernel each is given: route, copies, tile and k ranges.  With an argument: two products of one A, a
// line "... reads_first", and what both of them are given.
#include "f16_gemm_choice.h"

#include <cstdio>

int main(int argc, char **) {
  using namespace mi355;
  int b, m, n, k, a_cm, b_cm, aligned, reads_first;
  unsigned long long scratch, copies;
  while (std::scanf("%d %d %d %d %d %d %d %llu %llu", &b, &m, &n, &k, &a_cm, &b_cm, &aligned, &scratch, &copies) == 9) {
    GemmShape const shape = {b, m, n, k, a_cm != 0, b_cm != 0, aligned != 0, (size_t)scratch, (size_t)copies};
    if (argc > 1) {
      if (std::scanf("%d", &reads_first) != 1) {
        return 1;
      }
      GemmTwoChoice const c = choose_gemm_two(shape, reads_first != 0);
      GemmTile const &t = (a_cm ? kGemmTilesColumnMajorA : kGemmTiles)[c.choice.tile];
      std::printf("%d %d %d %d %d %d %.2f %.2f\n", c.half, c.tiles, (int)t.kind, t.bm, t.bn, c.choice.ksplit, c.us, choose_gemm(shape).us);
      continue;
    }
    GemmChoice const c = choose_gemm(shape);
    char const *routes[] = {"tiles", "big", "elements"};
    GemmTile const &t = (a_cm && !c.copy_a ? kGemmTilesColumnMajorA : kGemmTiles)[c.tile];
    std::printf("%s %d %d %d %d %d %d %.2f\n", routes[c.route], c.copy_a, c.copy_b, (int)t.kind, t.bm, t.bn, c.ksplit, c.us);
  }
  return 0;
}
