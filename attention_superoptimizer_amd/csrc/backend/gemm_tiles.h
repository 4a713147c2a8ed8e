// Between gemm_fused.hip (recognises the skinny-GEMM plans) and gemm_tiles.hip (the kernel for
// tiles of any size).
#pragma once

#include <string>

#include "mi355_kernels/gemm_tiles.h"

namespace mi355 {

struct TileGemmPlan {
  int grid[3];
  int pro, nb, rank;  // rank 0: no lora
  int cols;           // columns of the weight tile
  bool wcm;           // weight-side tensors column-major
};
// 1 = launched, 0 = not a shape of this kernel, negative = error.  `A` holds the tile addresses,
// rows, k extent and for-loop range.
int launch_gemm_tiles(GemmParams const &A, TileGemmPlan const &p);
// The parameter block as C++ source (programs that Graph::generate_hip_program writes).
std::string gemm_params_literal(GemmParams const &A, char const *var);

}  // namespace mi355
