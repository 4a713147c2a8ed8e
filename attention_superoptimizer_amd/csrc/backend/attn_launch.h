// Launches of the whole-tile attention kernels, by the form of their parameters: AttnParams (attn_fused.hip, which
// also chooses the shapes) or AttnFoldParams, the kernels that go on with the next operator (attn_fold.hip).
#pragma once

#include "common.h"
#include "tb_program.h"
#include "attn_tiles.h"
#include <string>
#include <type_traits>

#include "mi355_kernels/attention.h"

namespace mi355 {

// The shape of a direct-staging launch: `ip` wavefronts of `rpw` row groups each, `nbuf` tile
// pairs per wavefront, up to `nit` units of work per wavefront, `spi` strips per iteration or
// `ips` iterations per strip.
struct DirectShape {
  int ip = 0, rpw = 1, nbuf = 1, nit = 1, spi = 1, ips = 1;
  int code() const { return ((((ip * 10 + rpw) * 10 + nbuf) * 10 + nit) * 10 + spi) * 10 + ips; }
};

// The key loop's storage order and shape of the other two: `rg` row groups (slabs) of a workgroup.
struct AttnShape {
  int D, NK;
  bool cm;
  int rg, ip = 1, lds = 0, spi = 1;
  bool wide = false;
};
// The folding kernels (attn_fold.hip): 1 launched, 0 no instantiation, < 0 an error.
int launch_direct_fold(AttnFoldParams const &A, bool cm, dim3 grid, DirectShape const &d, int lds);
int launch_stream_fold(AttnFoldParams const &A, dim3 grid, AttnShape const &s);
int launch_fused_fold(AttnFoldParams const &A, dim3 grid, AttnShape const &s);
int launch_attn_tiles_fold(AttnFoldParams const &A, dim3 grid, int D, bool cm, TilesShape const &t);

namespace {

inline char const *tf(bool b) { return b ? "true" : "false"; }

template <bool HAS_DIV, bool CM, int IP, int RPW, int NBUF, int NIT, int SPI, int IPS, class Params>
int launch_direct_one(Params const &A, dim3 grid, int lds, bool dry) {
  if (dry) {
    return 1;  // the question was only whether this shape is built
  }
  constexpr bool plain = std::is_same_v<Params, AttnParams>;
  if constexpr (plain) {
    if (EmitSink *sink = emit_sink()) {
      sink->headers |= 1u;
      emit_launch(*sink, "attn_direct_kernel",
                  emit_fmt("64, 64, 64, %s, %d, %d, %d, %d, %d, %d, false, %s", tf(HAS_DIV), IP, RPW, NBUF, NIT, SPI, IPS,
                           tf(CM)),
                  grid, 64 * IP, lds, attn_params_literal(A));
      return 1;
    }
  }
  auto go = [&](auto *fn) -> int {
    MI355_GRANT_LDS(fn, lds);
    MI355_HIP(launch_kernel(fn, grid, 64 * IP, lds, state().stream(), A));
    return 1;
  };
  if constexpr (plain && SPI == 1 && IPS == 1) {
    if (A.trace != nullptr) {
      return go(attn_direct_kernel<64, 64, 64, HAS_DIV, IP, RPW, NBUF, NIT, SPI, IPS, true, CM>);
    }
  }
  return go(attn_direct_kernel<64, 64, 64, HAS_DIV, IP, RPW, NBUF, NIT, SPI, IPS, false, CM, Params>);
}

// 0: no instantiation for this shape
template <bool HAS_DIV, bool CM, class Params>
int launch_direct(Params const &A, dim3 grid, DirectShape const &d, int lds, bool dry = false) {
#define MI355_DIRECT(IPV, RPWV, NBUFV, NITV, SPIV, IPSV) \
  case ((((IPV * 10 + RPWV) * 10 + NBUFV) * 10 + NITV) * 10 + SPIV) * 10 + IPSV: \
    return launch_direct_one<HAS_DIV, CM, IPV, RPWV, NBUFV, NITV, SPIV, IPSV>(A, grid, lds, dry);
  switch (d.code()) {
    // one 64-key tile per iteration
    MI355_DIRECT(2, 1, 1, 1, 1, 1)
    MI355_DIRECT(4, 1, 1, 1, 1, 1)
    MI355_DIRECT(8, 1, 1, 1, 1, 1)
    MI355_DIRECT(4, 2, 1, 1, 1, 1)
    MI355_DIRECT(4, 1, 2, 2, 1, 1)
    MI355_DIRECT(4, 1, 2, 4, 1, 1)
    MI355_DIRECT(4, 1, 2, 8, 1, 1)
    MI355_DIRECT(4, 1, 1, 2, 1, 1)
    MI355_DIRECT(4, 1, 1, 4, 1, 1)
    MI355_DIRECT(4, 1, 1, 8, 1, 1)
    MI355_DIRECT(8, 1, 1, 2, 1, 1)
    MI355_DIRECT(8, 1, 1, 4, 1, 1)
    // key tiles of 32 and 16: two / four iterations per strip
    MI355_DIRECT(4, 1, 1, 1, 1, 2)
    MI355_DIRECT(4, 2, 1, 1, 1, 2)
    MI355_DIRECT(8, 1, 1, 1, 1, 2)
    MI355_DIRECT(8, 1, 1, 2, 1, 2)
    MI355_DIRECT(4, 1, 1, 1, 1, 4)
    MI355_DIRECT(4, 2, 1, 1, 1, 4)
    MI355_DIRECT(8, 1, 1, 1, 1, 4)
    default: break;
  }
  if constexpr (!HAS_DIV) {
    switch (d.code()) {
      // key tiles of 128 and 256: two / four strips per iteration (no division inside)
      MI355_DIRECT(4, 1, 1, 1, 2, 1)
      MI355_DIRECT(8, 1, 1, 1, 2, 1)
      MI355_DIRECT(8, 1, 1, 2, 2, 1)
      MI355_DIRECT(8, 1, 1, 4, 2, 1)
      MI355_DIRECT(4, 1, 1, 1, 4, 1)
      MI355_DIRECT(8, 1, 1, 1, 4, 1)
      MI355_DIRECT(8, 1, 1, 2, 4, 1)
      MI355_DIRECT(8, 1, 1, 4, 4, 1)
      default: break;
    }
  }
#undef MI355_DIRECT
  return 0;
}

template <int D, int NK, int DV, bool HAS_DIV, int RG, int IP, bool CM, class Params>
int launch_one(Params const &A, dim3 grid, int lds) {
  if constexpr (std::is_same_v<Params, AttnParams>) {
    if (EmitSink *sink = emit_sink()) {
      sink->headers |= 1u;
      emit_launch(*sink, "attn_fused_kernel", emit_fmt("%d, %d, %d, %s, %d, %d, %s", D, NK, DV, tf(HAS_DIV), RG, IP, tf(CM)),
                  grid, 64 * RG * IP, lds, attn_params_literal(A));
      return 1;
    }
  }
  auto *fn = attn_fused_kernel<D, NK, DV, HAS_DIV, RG, IP, CM, Params>;
  MI355_GRANT_LDS(fn, lds);
  MI355_HIP(launch_kernel(fn, grid, 64 * RG * IP, lds, state().stream(), A));
  return 1;
}

template <int D, int NK, int DV, bool HAS_DIV, bool CM, class Params>
int launch_waves(Params const &A, dim3 grid, int rg, int ip, int lds) {
  switch (rg * 16 + ip) {
    case 1 * 16 + 1: return launch_one<D, NK, DV, HAS_DIV, 1, 1, CM>(A, grid, lds);
    case 1 * 16 + 2: return launch_one<D, NK, DV, HAS_DIV, 1, 2, CM>(A, grid, lds);
    case 1 * 16 + 4: return launch_one<D, NK, DV, HAS_DIV, 1, 4, CM>(A, grid, lds);
    case 1 * 16 + 8: return launch_one<D, NK, DV, HAS_DIV, 1, 8, CM>(A, grid, lds);
    case 2 * 16 + 1: return launch_one<D, NK, DV, HAS_DIV, 2, 1, CM>(A, grid, lds);
    case 2 * 16 + 2: return launch_one<D, NK, DV, HAS_DIV, 2, 2, CM>(A, grid, lds);
    case 2 * 16 + 4: return launch_one<D, NK, DV, HAS_DIV, 2, 4, CM>(A, grid, lds);
    case 4 * 16 + 1: return launch_one<D, NK, DV, HAS_DIV, 4, 1, CM>(A, grid, lds);
    case 4 * 16 + 2: return launch_one<D, NK, DV, HAS_DIV, 4, 2, CM>(A, grid, lds);
    default: return 0;
  }
}

template <int D, int NK, int DV, bool HAS_DIV, int RG, int RPW, bool CM, int SPI = 1, class Params>
int launch_stream_one(Params const &A, dim3 grid, int lds) {
  if constexpr (std::is_same_v<Params, AttnParams>) {
    if (EmitSink *sink = emit_sink()) {
      sink->headers |= 1u;
      emit_launch(*sink, "attn_stream_kernel",
                  emit_fmt("%d, %d, %d, %s, %d, %d, %s, %d", D, NK, DV, tf(HAS_DIV), RG, RPW, tf(CM), SPI), grid, 64 * RG,
                  lds, attn_params_literal(A));
      return 1;
    }
  }
  auto *fn = attn_stream_kernel<D, NK, DV, HAS_DIV, RG, RPW, CM, SPI, Params>;
  MI355_GRANT_LDS(fn, lds);
  MI355_HIP(launch_kernel(fn, grid, 64 * RG, lds, state().stream(), A));
  return 1;
}

template <int D, int NK, int DV, bool CM, bool HAS_DIV, class Params>
int launch_stream(Params const &A, dim3 grid, int rg, int lds, bool wide, int spi) {
  if (spi > 1) {  // wider key tiles: four wavefronts of 32 rows, the form without the division
    if constexpr (!HAS_DIV) {
      if (rg == 4 && !wide) {
        switch (spi) {
          case 2: return launch_stream_one<D, NK, DV, false, 4, 2, CM, 2>(A, grid, lds);
          case 4: return launch_stream_one<D, NK, DV, false, 4, 2, CM, 4>(A, grid, lds);
          case 8: return launch_stream_one<D, NK, DV, false, 4, 2, CM, 8>(A, grid, lds);
          default: break;
        }
      }
    }
    return 0;
  }
  if constexpr (D == 64) {
    if (wide) {  // four wavefronts of 64 rows
      return launch_stream_one<D, NK, DV, HAS_DIV, 4, 4, CM>(A, grid, lds);
    }
  }
  return rg == 4 ? launch_stream_one<D, NK, DV, HAS_DIV, 4, 2, CM>(A, grid, lds)
                 : launch_stream_one<D, NK, DV, HAS_DIV, 2, 2, CM>(A, grid, lds);
}

template <bool HAS_DIV, class Params>
int launch_stream_shape(Params const &A, dim3 grid, AttnShape const &s) {
  if (s.cm) {
    return s.D == 64 ? launch_stream<64, 64, 64, true, HAS_DIV>(A, grid, s.rg, s.lds, s.wide, s.spi)
                     : launch_stream<128, 64, 128, true, HAS_DIV>(A, grid, s.rg, s.lds, false, s.spi);
  }
  return s.D == 64 ? launch_stream<64, 64, 64, false, HAS_DIV>(A, grid, s.rg, s.lds, s.wide, s.spi)
                   : launch_stream<128, 64, 128, false, HAS_DIV>(A, grid, s.rg, s.lds, false, s.spi);
}

template <bool HAS_DIV, bool CM, class Params>
int launch_fused_order(Params const &A, dim3 grid, AttnShape const &s) {
  if (s.D == 128) {
    return launch_waves<128, 64, 128, HAS_DIV, CM>(A, grid, s.rg, s.ip, s.lds);
  }
  return s.NK == 64    ? launch_waves<64, 64, 64, HAS_DIV, CM>(A, grid, s.rg, s.ip, s.lds)
         : s.NK == 128 ? launch_waves<64, 128, 64, HAS_DIV, CM>(A, grid, s.rg, s.ip, s.lds)
                       : launch_waves<64, 256, 64, HAS_DIV, CM>(A, grid, s.rg, s.ip, s.lds);
}
template <bool HAS_DIV, class Params>
int launch_fused_shape(Params const &A, dim3 grid, AttnShape const &s) {
  return s.cm ? launch_fused_order<HAS_DIV, true>(A, grid, s) : launch_fused_order<HAS_DIV, false>(A, grid, s);
}

}  // namespace
}  // namespace mi355
