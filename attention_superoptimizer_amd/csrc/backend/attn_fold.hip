// The attention kernels that go on with the next operator (include/mi355_kernels/attention_fold.h): instantiations
// and launches.  Which plans take them, and in which shape, is attn_fused.hip's.
#include "attn_launch.h"

namespace mi355 {

int launch_direct_fold(AttnFoldParams const &A, bool cm, dim3 grid, DirectShape const &d, int lds) {
  return cm ? launch_direct<false, true>(A, grid, d, lds) : launch_direct<false, false>(A, grid, d, lds);
}
int launch_stream_fold(AttnFoldParams const &A, dim3 grid, AttnShape const &s) { return launch_stream_shape<false>(A, grid, s); }
int launch_fused_fold(AttnFoldParams const &A, dim3 grid, AttnShape const &s) { return launch_fused_shape<false>(A, grid, s); }

}  // namespace mi355
