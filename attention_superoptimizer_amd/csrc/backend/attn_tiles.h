// Between attn_fused.hip (recognises attention plans) and attn_tiles.hip (the kernel for tiles of
// any size).
#pragma once

#include <hip/hip_runtime.h>
#include <string>

#include "mi355_kernels/attention.h"

namespace mi355 {

struct TilesShape {
  int rpw = 1, pairs = 0, ip = 1, split = 1, lds = 0;
};
// Whether attn_tiles_kernel takes query tiles of `m` rows against key tiles of NK keys, and in
// which shape; `blocks` = logical thread blocks, F = for-loop range.
bool choose_attn_tiles(int D, int DV, int NK, int m, bool has_div, bool cm, long long blocks, int F, int max_lds,
                       TilesShape &t);
int launch_attn_tiles(AttnParams const &A, dim3 grid, int D, bool has_div, bool cm, TilesShape const &t);
// The parameter block as C++ source (programs that Graph::generate_hip_program writes).
std::string attn_params_literal(AttnParams const &A);

}  // namespace mi355
