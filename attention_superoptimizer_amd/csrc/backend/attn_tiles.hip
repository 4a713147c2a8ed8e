// Launches of attn_tiles_kernel (include/mi355_kernels/attention_tiles.h): which instantiation an
// attention plan of any tile size gets.  Recognition and the parameter block are attn_fused.hip's.
#include "common.h"
#include "tb_program.h"
#include "attn_tiles.h"
#include <algorithm>
#include <string>

#include "mi355_kernels/attention_tiles.h"

namespace mi355 {

namespace {

template <int D, bool HAS_DIV, bool CM, int RPW, int PAIRS, class Params>
int launch_tiles_one(Params const &A, dim3 grid, int ip, int lds) {
  if constexpr (std::is_same_v<Params, AttnParams>) {
    if (EmitSink *sink = emit_sink()) {
      sink->headers |= 8u;
      emit_launch(*sink, "attn_tiles_kernel",
                  emit_fmt("%d, %s, %s, %d, %d", D, HAS_DIV ? "true" : "false", CM ? "true" : "false", RPW, PAIRS), grid, 64 * ip, lds,
                  attn_params_literal(A));
      return 1;
    }
  }
  auto *fn = attn_tiles_kernel<D, HAS_DIV, CM, RPW, PAIRS, Params>;
  MI355_GRANT_LDS(fn, lds);
  MI355_HIP(launch_kernel(fn, grid, 64 * ip, lds, state().stream(), A));
  return 1;
}

template <int D, bool HAS_DIV, bool CM, class Params>
int launch_tiles_shape(Params const &A, dim3 grid, int rpw, int pairs, int ip, int lds) {
  if constexpr (!HAS_DIV) {
    return rpw == 1 ? launch_tiles_one<D, false, CM, 1, 0>(A, grid, ip, lds) : launch_tiles_one<D, false, CM, 2, 0>(A, grid, ip, lds);
  } else {
    switch (rpw * 10 + pairs) {
      case 11: return launch_tiles_one<D, true, CM, 1, 1>(A, grid, ip, lds);
      case 12: return launch_tiles_one<D, true, CM, 1, 2>(A, grid, ip, lds);
      case 21: return launch_tiles_one<D, true, CM, 2, 1>(A, grid, ip, lds);
      case 22: return launch_tiles_one<D, true, CM, 2, 2>(A, grid, ip, lds);
      default: break;
    }
    if constexpr (D == 64) {
      switch (rpw * 10 + pairs) {
        case 13: return launch_tiles_one<D, true, CM, 1, 3>(A, grid, ip, lds);
        case 14: return launch_tiles_one<D, true, CM, 1, 4>(A, grid, ip, lds);
        case 23: return launch_tiles_one<D, true, CM, 2, 3>(A, grid, ip, lds);
        case 24: return launch_tiles_one<D, true, CM, 2, 4>(A, grid, ip, lds);
        default: break;
      }
    }
    return 0;
  }
}

}  // namespace

bool choose_attn_tiles(int D, int DV, int NK, int m, bool has_div, bool cm, long long blocks, int F, int max_lds,
                       TilesShape &t) {
  if (D != DV || (D != 64 && D != 128) || NK % 16 != 0 || NK < 16 || m < 1) {
    return false;
  }
  // The division needs the row sum of the whole tile before P.V: its exponentials stay in registers.
  t.pairs = has_div ? (NK / 16 + 1) / 2 : 0;
  if (t.pairs > (D == 64 ? 4 : 2)) {
    return false;
  }
  // Two row groups per wavefront (each K / V operand then feeds two matrix instructions) where that
  // leaves a workgroup for almost every compute unit, unless rounding the row groups up to whole
  // wavefronts would add more than a third of work.
  int const groups = (m + 15) / 16, halves = (groups + 1) / 2;
  t.rpw = groups >= 2 && 6 * halves <= 4 * groups && blocks * halves >= 192 ? 2 : 1;
  t.split = (groups + t.rpw - 1) / t.rpw;
  // Iteration lanes: one wavefront per iteration up to what the instantiation allows, evened out
  // over the rounds.
  int const most = attn_tiles_lanes(D, t.pairs);
  for (int cap = most; cap >= 1; cap--) {
    int const rounds = (F + cap - 1) / cap;
    t.ip = (F + rounds - 1) / rounds;
    t.lds = attn_tiles_lds(D, t.rpw, t.ip, rounds);
    if (t.lds <= max_lds) {
      return true;
    }
  }
  return false;
}

int launch_attn_tiles(AttnParams const &A, dim3 grid, int D, bool has_div, bool cm, TilesShape const &t) {
  if (D == 64) {
    if (has_div) {
      return cm ? launch_tiles_shape<64, true, true>(A, grid, t.rpw, t.pairs, t.ip, t.lds)
                : launch_tiles_shape<64, true, false>(A, grid, t.rpw, t.pairs, t.ip, t.lds);
    }
    return cm ? launch_tiles_shape<64, false, true>(A, grid, t.rpw, t.pairs, t.ip, t.lds)
              : launch_tiles_shape<64, false, false>(A, grid, t.rpw, t.pairs, t.ip, t.lds);
  }
  if (has_div) {
    return cm ? launch_tiles_shape<128, true, true>(A, grid, t.rpw, t.pairs, t.ip, t.lds)
              : launch_tiles_shape<128, true, false>(A, grid, t.rpw, t.pairs, t.ip, t.lds);
  }
  return cm ? launch_tiles_shape<128, false, true>(A, grid, t.rpw, t.pairs, t.ip, t.lds)
            : launch_tiles_shape<128, false, false>(A, grid, t.rpw, t.pairs, t.ip, t.lds);
}

int launch_attn_tiles_fold(AttnFoldParams const &A, dim3 grid, int D, bool cm, TilesShape const &t) {
  if (D == 64) {
    return cm ? launch_tiles_shape<64, false, true>(A, grid, t.rpw, t.pairs, t.ip, t.lds)
              : launch_tiles_shape<64, false, false>(A, grid, t.rpw, t.pairs, t.ip, t.lds);
  }
  return cm ? launch_tiles_shape<128, false, true>(A, grid, t.rpw, t.pairs, t.ip, t.lds)
            : launch_tiles_shape<128, false, false>(A, grid, t.rpw, t.pairs, t.ip, t.lds);
}

}  // namespace mi355
