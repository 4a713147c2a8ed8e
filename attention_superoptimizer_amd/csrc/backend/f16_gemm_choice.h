// Which kernel a kernel-level fp16 matmul runs on: the tiles there are, what each is expected to take, and
// the choice.  Host code without a device, so that the choice can be looked at where there is none.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>

namespace mi355 {

// f16_gemm_any_kernel, f16_gemm_direct_kernel, f16_gemm_waves_kernel
enum GemmKind { STAGED, DIRECT, WAVES };
struct GemmTile {
  GemmKind kind;
  int bm, bn, wm, wn, kg;
  constexpr int threads() const { return 64 * (bm / wm) * (bn / wn) * kg; }
};
// A row-major: every kernel
constexpr GemmTile kGemmTiles[] = {
    {STAGED, 16, 64, 16, 16, 1}, {STAGED, 16, 64, 16, 16, 2},  {STAGED, 32, 64, 32, 16, 1},  {STAGED, 32, 64, 32, 16, 2},
    {STAGED, 64, 64, 32, 32, 1}, {STAGED, 64, 64, 32, 32, 2},  {STAGED, 64, 128, 32, 64, 1}, {STAGED, 64, 128, 32, 64, 2},
    {STAGED, 128, 128, 64, 64, 1}, {DIRECT, 64, 64, 32, 32, 1}, {DIRECT, 64, 128, 32, 32, 1}, {DIRECT, 128, 64, 64, 32, 1},
    {WAVES, 16, 64, 16, 64, 4},  {WAVES, 32, 64, 32, 64, 4}};
// A column-major (a layout search may ask for one): the middle tiles
constexpr GemmTile kGemmTilesColumnMajorA[] = {{STAGED, 64, 64, 32, 32, 1}, {STAGED, 64, 64, 32, 32, 2}};
constexpr int kWavesRing = 4;  // slots of a wavefront's ring of steps (f16_gemm_waves_kernel)

struct GemmShape {
  int batch, m, n, k;
  bool a_column_major, b_column_major;
  bool aligned;          // A and B on 16-byte boundaries
  size_t scratch_bytes;  // room for the sums of k ranges (0: none)
  size_t copy_bytes;     // room for transposed copies of operands
};
enum GemmRoute { GEMM_TILES, GEMM_BIG /* f16_gemm_nt_kernel */, GEMM_ELEMENTS /* f16_matmul_kernel */ };
struct GemmChoice {
  GemmRoute route;
  bool copy_a, copy_b;  // onto transposed copies of these operands
  int tile, ksplit;     // GEMM_TILES: an index into the list that the storage order of A as multiplied has
  double us;            // expected
};

// Microseconds a tile shape is expected to take: a line fitted to timed launches (m from 1 to 2048, n and
// k from 64 to 5504; on 130 other products of these ranges, each run on all it can run on, the choice made
// with it is 1.9 % above the best on average and 19 % at worst).  A launch, then either the latency of its k stages one after another (0.24 us each) or,
// with the compute units full, what they have to move: 128-byte rows through the vector cache, into
// LDS and from there to the operands, and the matrix instructions.  k ranges need a second launch.
// (The kernels that load LDS directly: 3.2 us, and 35 bytes a cycle per compute unit; a lone workgroup
// waits 1.4 times as long for a stage, but not where wavefronts go their own ways, and 1.25 with eight of them: two on
// a SIMD read operands under each other's products (64 x 128 tiles by four wavefronts and by eight: [300, 2048] .
// [2048, 5504] row-major 14.7 and 13.4 us, column-major 13.8 and 12.7, [300, 5504] . [5504, 2048] in three ranges 20.0
// and 17.2; 64 x 64 there 14.1, 13.9 and 18.8; with 1.0 [256, 4096] . [4096, 4096] went to two ranges, 18.3 -> 19.4).  15 shapes, within 15 %.
// The rings of f16_gemm_waves_kernel leave room for one or two workgroups on a compute unit: those that
// queue there pay their first loads and the adding up again, 1.3 us: [200, 130, 96] . [200, 96, 130] 23.8 us
// on it, 9 on 64 x 64.)
inline double gemm_tile_cost(GemmTile const &t, int batch, int m, int n, int k, int ksplit) {
  if (t.kind != STAGED) {
    double const stages = (k / 32 + 2 * ksplit - 1) / (2 * ksplit), stage = (t.bm + t.bn) * 128.0 / 35.0 / 2400.0;
    double per_cu = (double)((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn) * batch * ksplit / 256.0;
    if (t.kind == WAVES || per_cu < 3.0) {
      per_cu = std::ceil(per_cu);  // (the compute unit with the most workgroups is the last to finish)
    }
    double us = 3.2 + stages * stage * std::max(per_cu, t.kind == WAVES ? 1.0 : t.threads() < 512 ? 1.4 : 1.25) + per_cu * 0.9e-4 * t.bm * t.bn;
    if (t.kind == WAVES) {
      int const resident = 160 * 1024 / (4 * kWavesRing * (t.bm + t.bn) * 64);
      us += 1.3 * (std::ceil(per_cu / resident) - 1.0);
    }
    return us + (ksplit > 1 ? 2.0 + 0.3 * ksplit + 1.4e-6 * batch * (double)m * n * ksplit : 0.0);
  }
  int const stages = (k / 64 + ksplit * t.kg - 1) / (ksplit * t.kg) + (k % 64 != 0 ? 1 : 0);
  double const tiles = (double)((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn) * batch * ksplit;
  double const rows = 3.0 * (t.bm + t.bn) + (t.bm / t.wm) * (t.bn / t.wn) * (t.wm + t.wn);
  double const stage = t.kg * (1.2 * rows + 0.2 * t.bm * t.bn / 32.0) / 2400.0;
  double per_cu = tiles / 256.0;
  if (per_cu <= 2.0) {
    per_cu = per_cu <= 1.0 ? 1.0 : 2.0;
  }
  double us = 2.4 + 0.4 * (t.kg - 1) + std::max(0.24 * stages, per_cu * stages * stage) + per_cu * 0.9e-4 * t.bm * t.bn;
  if (ksplit > 1) {
    us += 2.0 + 0.3 * ksplit + 1.4e-6 * batch * (double)m * n * ksplit;
  }
  return us;
}

// ... and what f16_gemm_nt_kernel is: rounds of 256 tiles of 256 x 256, one to a compute unit; of a round its
// start and its stores (4.9 us, more with every compute unit storing) and its steps of 32 k.  From 980 timed
// products (batches up to 200, m and n from 128 to 8192, k from 32 to 4096, both orders of both operands),
// within 15 % of nine in ten.  It is ahead by up to a quarter where the rounds are full, [32, 2048, 128] .
// [32, 128, 2048] 103 us against 113 on 64 x 128 tiles, [4096, 1024] . [1024, 4096] 38 against 49, and behind
// by as much and more where they are not: [12, 1040, 256] . [12, 256, 1040] 27 against 19.
inline double gemm_big_cost(int batch, int m, int n, int k) {
  double const tiles = (double)((m + 255) / 256) * ((n + 255) / 256) * batch;
  double const rounds = std::ceil(tiles / 256.0), full = tiles / 256.0 / rounds;
  return 2.7 + rounds * (4.9 + 1.6 * full + k / 32 * (0.53 + 0.33 * full));
}
// A transposed copy of an operand (the same products: 6.7 us and 2.3 TB/s)
inline double gemm_copy_cost(size_t bytes) { return 6.7 + 0.44e-6 * bytes; }

// The kernel of least expected time among those that take the product.
inline GemmChoice choose_gemm(GemmShape const &s) {
  GemmChoice best{GEMM_ELEMENTS, false, false, 0, 1, 0.0};
  size_t const a_bytes = s.a_column_major ? (size_t)s.batch * s.m * s.k * 2 : 0, a_room = (a_bytes + 255) & ~(size_t)255;
  size_t const b_bytes = s.b_column_major ? 0 : (size_t)s.batch * s.k * s.n * 2;
  // The tiles, on A as it is stored or on a copy of a column-major one: that has all the tiles, and pays
  // where a product is large and k long: [563, 3520] . [3520, 6177] 64 us as stored, 51 with the copy,
  // [2048, 4096] . [4096, 4096] 114 and 89, [2048, 2048] . [2048, 2048] 32 and 32, [1024, 1024] . [1024, 1024]
  // 7.5 and 13.
  for (bool const copy_a : {false, true}) {
    if (copy_a && (!s.a_column_major || best.route == GEMM_ELEMENTS || a_room > s.copy_bytes)) {
      continue;
    }
    bool const a_kc = !s.a_column_major || copy_a;
    // Byte offsets inside a tile are 31-bit numbers; a contiguous direction shorter than a chunk of
    // eight goes element by element.
    int const a_row = a_kc ? s.k : s.m, b_row = s.b_column_major ? s.k : s.n;
    if (std::min(a_row, b_row) < 8 || std::max(a_row, b_row) >= (1 << 22)) {
      continue;
    }
    bool const chunks = a_kc && (s.b_column_major || s.n % 8 == 0) && s.aligned;
    size_t const range_bytes = (size_t)s.batch * s.m * s.n * sizeof(float);
    GemmTile const *const tiles = a_kc ? kGemmTiles : kGemmTilesColumnMajorA;
    int const count = (int)((a_kc ? sizeof(kGemmTiles) : sizeof(kGemmTilesColumnMajorA)) / sizeof(GemmTile));
    for (int i = 0; i < count; i++) {
      GemmTile const &t = tiles[i];
      if (t.kind != STAGED && (!chunks || s.k % (t.kind == DIRECT ? 64 : 32) != 0)) {
        continue;
      }
      for (int ranges : {1, 2, 3, 4, 6, 8, 12, 16}) {
        // (a range is a stage per group at least, and the ranges' sums fit the scratch memory)
        if (ranges > 1 && (s.k / 64 < ranges * (t.kind == WAVES ? 1 : t.kg) || range_bytes * ranges > s.scratch_bytes)) {
          break;
        }
        // (with A column-major the 64 x 64 tiles take 0.8 of the line, 560 of the products below)
        double const us = gemm_tile_cost(t, s.batch, s.m, s.n, s.k, ranges) * (a_kc ? 1.0 : 0.8) + (copy_a ? gemm_copy_cost(a_bytes) : 0.0);
        if (best.route == GEMM_ELEMENTS || us < best.us) {
          best = {GEMM_TILES, copy_a, false, i, ranges, us};
        }
      }
    }
  }
  // f16_gemm_nt_kernel wants k contiguous in both operands, k in whole steps of 32 and 16-byte aligned rows;
  // an operand stored the other way round is first copied transposed.  (Its consumer stays a launch of its
  // own: applied in the store, exp on [32, 2048, 2048] made the two 210 us instead of 209, a product by a
  // tensor 296 instead of 271.)
  bool const fits = a_room + b_bytes <= s.copy_bytes;
  if (s.k >= 32 && s.k % 32 == 0 && s.aligned && fits && (size_t)std::max(s.m, s.n) * (size_t)s.k < ((size_t)1 << 30)) {
    double const us = gemm_big_cost(s.batch, s.m, s.n, s.k) + (s.a_column_major ? gemm_copy_cost(a_bytes) : 0.0) +
                      (s.b_column_major ? 0.0 : gemm_copy_cost(b_bytes));
    double const tiles = (double)((s.m + 255) / 256) * ((s.n + 255) / 256) * s.batch;
    if (best.route == GEMM_ELEMENTS ? tiles >= 192 : us < best.us) {
      best = {GEMM_BIG, s.a_column_major, !s.b_column_major, 0, 1, us};
    }
  }
  return best;
}

// Two products of the same A and shape (a batch of one), both of them and what consumes them.
struct GemmTwoChoice {
  int half;    // columns of each that a workgroup of both has; 0: no such workgroups
  bool tiles;  // each product's tiles as workgroups of one launch
  GemmChoice choice;
  double us;
};
// A workgroup of both (f16_gemm_direct_kernel, 64 rows), from timed launches: [300, 2048] . [2048, 5504] 26.1 us with 128
// columns of each and 29.1 with 64, [700, 1024] . [1024, 2752] 15.4 and 16.1, [60, 1024] . [1024, 3000] 15.0 and 10.5.
inline double gemm_two_cost(int half, int m, int n, int k) {
  double const tiles = (double)((m + 63) / 64) * ((n + half - 1) / half), per_cu = std::ceil(tiles / 256.0);
  double const stage = half == 128 ? 0.67 * per_cu : 0.38 * per_cu;
  return 4.5 + k / 64 * stage + 1.5 * (per_cu - 1.0);
}
// Without either (half 0, no tiles) one after the other is expected to be faster.  reads_first: the second's consumer
// takes what the first leaves, which whole products of different workgroups could not tell it.  With these
// constants 218 un-fused gated MLPs of 1 - 1000 rows took 0.61 - 1.02 of their time one by one, 0.84 on average; the gain
// is the second launch, the second fold and a chip that one product does not fill (us, one by one / two at a time, the
// whole MLP: 6 x 1419 x 2111 34.6 / 22.7, 28 x 1169 x 1092 26.0 / 17.6, 512 x 2048 x 2048 35.4 / 27.6, 300 x 2048 x
// 5504 56.7 / 47.1).  Not where tiles of one product fill the chip and none of both takes its sizes.
inline GemmTwoChoice choose_gemm_two(GemmShape const &s, bool reads_first) {
  GemmChoice const one = choose_gemm(s);
  GemmTwoChoice best{0, false, one, one.route == GEMM_ELEMENTS ? 1e30 : 2.0 * one.us};
  bool const a_kc = !s.a_column_major;
  int const a_row = a_kc ? s.k : s.m, b_row = s.b_column_major ? s.k : s.n;
  if (std::min(a_row, b_row) < 8 || std::max(a_row, b_row) >= (1 << 22)) {
    return best;
  }
  bool const chunks = a_kc && (s.b_column_major || s.n % 8 == 0) && s.aligned;
  for (int half : {64, 128}) {
    if (chunks && s.k % 64 == 0) {
      double const us = gemm_two_cost(half, s.m, s.n, s.k);
      if (us < best.us) {
        best = {half, false, one, us};
      }
    }
  }
  size_t const range_bytes = 2 * (size_t)s.m * s.n * sizeof(float);
  GemmTile const *const tiles = a_kc ? kGemmTiles : kGemmTilesColumnMajorA;
  int const count = (int)((a_kc ? sizeof(kGemmTiles) : sizeof(kGemmTilesColumnMajorA)) / sizeof(GemmTile));
  for (int i = 0; i < count; i++) {
    GemmTile const &t = tiles[i];
    if (t.kind != STAGED && (!chunks || s.k % (t.kind == DIRECT ? 64 : 32) != 0)) {
      continue;
    }
    for (int ranges : {1, 2, 3, 4, 6, 8, 12, 16}) {
      if (ranges > 1 && (s.k / 64 < ranges * (t.kind == WAVES ? 1 : t.kg) || range_bytes * ranges > s.scratch_bytes)) {
        break;
      }
      if (ranges == 1 && reads_first) {
        continue;
      }
      double const us = gemm_tile_cost(t, 2, s.m, s.n, s.k, ranges) * (a_kc ? 1.0 : 0.8) + 1.5;
      if (us < best.us) {
        best = {0, true, {GEMM_TILES, false, false, i, ranges, us}, us};
      }
    }
  }
  return best;
}

}  // namespace mi355
