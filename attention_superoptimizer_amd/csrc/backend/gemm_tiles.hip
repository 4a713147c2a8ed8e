// Launches of gemm_tiles_kernel (include/mi355_kernels/gemm_tiles.h): which instantiation and launch
// shape a skinny-GEMM plan of any tile size gets.  Recognition and the tile addresses are
// gemm_fused.hip's.
#include "common.h"
#include "gemm_tiles.h"
#include "tb_program.h"
#include <algorithm>
#include <string>

namespace mi355 {

namespace {

char const *tf(bool b) { return b ? "true" : "false"; }

std::string literal(TileGemmParams const &L) {
  std::string t = gemm_params_literal(L.g, "G") + "    mi355::TileGemmParams P{};\n    P.g = G;\n";
  t += emit_fmt("    P.strips = %d;\n    P.slabs = %d;\n    P.round = %d;\n    P.rank = %d;\n    P.cols = %d;\n", L.strips, L.slabs,
                L.round, L.rank, L.cols);
  t += emit_fmt("    P.m_strips = %uu;\n    P.m_slabs = %uu;\n", L.m_strips, L.m_slabs);
  return t;
}

template <int MT, int CT, int NB, int PRO, bool LORA, bool WCM>
int launch_one(TileGemmParams const &L, dim3 grid, int threads, int lds) {
  if (EmitSink *sink = emit_sink()) {
    sink->headers |= 16u;
    emit_launch(*sink, "gemm_tiles_kernel", emit_fmt("%d, %d, %d, %d, %s, %s", MT, CT, NB, PRO, tf(LORA), tf(WCM)), grid, threads,
                lds, literal(L));
    return 1;
  }
  auto *fn = gemm_tiles_kernel<MT, CT, NB, PRO, LORA, WCM>;
  MI355_GRANT_LDS(fn, lds);
  MI355_HIP(launch_kernel(fn, grid, threads, lds, state().stream(), L));
  return 1;
}

template <int MT, int CT, int NB, int PRO, bool LORA>
int launch_order(TileGemmParams const &L, bool wcm, dim3 grid, int threads, int lds) {
  return wcm ? launch_one<MT, CT, NB, PRO, LORA, true>(L, grid, threads, lds)
             : launch_one<MT, CT, NB, PRO, LORA, false>(L, grid, threads, lds);
}

}  // namespace

int launch_gemm_tiles(GemmParams const &A, TileGemmPlan const &p) {
  State &s = state();
  if (p.cols % 16 != 0 || A.KT % 32 != 0 || A.M < 1 || (p.rank != 0 && p.rank != 8 && p.rank != 16 && p.rank != 32)) {
    return 0;
  }
  bool const lora = p.rank != 0, plain = p.nb == 1 && p.pro == PRO_NONE && !lora;
  int const F = A.forloop_range;
  long long const blocks = (long long)p.grid[0] * p.grid[1] * p.grid[2];
  int const groups = (A.M + 15) / 16;
  // Rows: as many as one slab can hold (64; 32 for the members with a prologue or a second product),
  // so that the weights stream once, while that leaves a workgroup for every compute unit; fewer
  // otherwise: the slabs then re-read weights of a few MB from the L2, which costs less than an idle
  // chip (38 rows x 48 columns x 12 blocks, for-loop 24: 9.9 us in 36 workgroups, 6.7 in 108).  A
  // lora slab also repeats X.A, so it is cut later.
  int mt = groups <= 1 ? 1 : (groups == 2 || !plain ? 2 : 4);
  while (mt > 1 && blocks * ((groups + mt - 1) / mt) * (p.cols / 16) < (lora ? 128 : 256)) {
    mt /= 2;
  }
  int const slabs = (groups + mt - 1) / mt;
  // Columns: 32 per workgroup where that still leaves two workgroups for every compute unit (half
  // the activation traffic, and 64-byte rows of a row-major weight strip), else 16.
  int const ct = plain && p.cols % 32 == 0 && blocks * slabs * (p.cols / 32) >= 512 ? 2 : 1;
  TileGemmParams L{};
  L.g = A;
  L.strips = p.cols / (16 * ct);
  L.slabs = slabs;
  L.rank = p.rank;
  L.cols = p.cols;
  L.m_strips = fast_div_magic(L.strips);
  L.m_slabs = fast_div_magic(L.slabs);
  unsigned long long const gx = (unsigned long long)p.grid[0] * L.strips * L.slabs;
  if (gx * (unsigned)std::max(L.strips, L.slabs) >= (1ull << 32) || gx > 2147483647ull) {
    return 0;  // (the magics are exact below 2^32)
  }
  // Lanes: a wavefront per iteration up to what the instantiation allows, sixteen only while there
  // are fewer than two workgroups for every compute unit (16 rows x 128 columns x 119 blocks: 13.6 us
  // with eight lanes, 15.8 with sixteen).  A round is the whole for-loop while its slots
  // take at most 64 KB (two workgroups per compute unit), else as many whole sets of lanes as fit
  // half of that, double buffered.
  int const slot = p.nb * 16 * mt * (16 * ct + 4) * 2;
  int const most = gx * p.grid[1] * p.grid[2] < 512 ? gemm_tiles_lanes(mt, ct, p.nb, p.pro, lora) : 8;
  int const sets = (F + most - 1) / most, ip = (F + sets - 1) / sets;
  L.round = (long long)F * slot <= 65536 ? F : std::max(1, 32768 / (ip * slot)) * ip;
  if (L.round > F) {
    L.round = F;
  }
  int const lds = (L.round < F ? 2 : 1) * L.round * slot + (p.wcm ? 0 : ip * (32 * (16 * ct + 8) + (lora ? 32 * 40 : 0)) * 2);
  if (lds > s.max_lds) {
    return 0;
  }
  dim3 const grid((unsigned)gx, p.grid[1], p.grid[2]);
  int const threads = 64 * ip;
  int rc = 0;
#define MI355_TILES(MTV, CTV, NBV, PROV, LORAV)                                                          \
  if (mt == MTV && ct == CTV && p.nb == NBV && p.pro == PROV && lora == LORAV) {                         \
    rc = launch_order<MTV, CTV, NBV, PROV, LORAV>(L, p.wcm, grid, threads, lds);                         \
  }
  MI355_TILES(1, 1, 1, PRO_NONE, false)
  MI355_TILES(2, 1, 1, PRO_NONE, false)
  MI355_TILES(4, 1, 1, PRO_NONE, false)
  MI355_TILES(1, 2, 1, PRO_NONE, false)
  MI355_TILES(2, 2, 1, PRO_NONE, false)
  MI355_TILES(4, 2, 1, PRO_NONE, false)
  MI355_TILES(1, 1, 1, PRO_EXP, false)
  MI355_TILES(2, 1, 1, PRO_EXP, false)
  MI355_TILES(1, 1, 1, PRO_SILU, false)
  MI355_TILES(2, 1, 1, PRO_SILU, false)
  MI355_TILES(1, 1, 2, PRO_NONE, false)
  MI355_TILES(2, 1, 2, PRO_NONE, false)
  MI355_TILES(1, 1, 1, PRO_SILU_MUL, false)
  MI355_TILES(2, 1, 1, PRO_SILU_MUL, false)
  MI355_TILES(1, 1, 1, PRO_NONE, true)
  MI355_TILES(2, 1, 1, PRO_NONE, true)
#undef MI355_TILES
  if (rc == 1) {
    s.last().kernel_id = MI355_KERNEL_F16_GEMM;
    s.last().workgroups = (int)(grid.x * grid.y * grid.z);
    s.last().threads = threads;
    s.last().lds_bytes = lds;
    s.last().row_split = L.strips * L.slabs;
  }
  return rc;
}

}  // namespace mi355
