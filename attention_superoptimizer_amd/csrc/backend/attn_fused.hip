// Fused, register-resident kernel for the attention family of thread-block graphs:
//
//   form A   S = Q.K ; E = exp(S) ; r = rowsum(E) ; P = E / r ; O = P.V        -> accumulate O
//   form B   S = Q.K ; E = exp(S) ; O = E.V ; r = rowsum(E)                     -> accumulate O and r
//
// (the single-op GQA decode plan and the reference's two-output split-KV plans,
// e.g. cpp_examples/group_query_attn_inc_decode.cc:47-74).  Same arithmetic and the
// same fp16 rounding points as the generic interpreter, but no intermediate tile
// ever touches LDS:
//
//  * one wavefront owns 16 query rows for one for-loop iteration at a time.  A
//    workgroup is RG row groups x IP iteration lanes: the IP wavefronts of a row
//    group work on IP consecutive iterations at once and hand their fp16 results to
//    the group's first wavefront, which adds them in iteration order (the order the
//    sequential loop would use).  A logical thread block's rows are split over as
//    many workgroups as it takes to fill the chip: the plan's grid is a lower bound
//    on parallelism, not the launch shape;
//  * S is produced TRANSPOSED (S^T = K^T.Q^T) with 16x16x32 fp16 MFMA, so that each
//    lane ends up holding four consecutive keys of one query row — exactly the
//    A-operand layout of the next MFMA.  exp, the row sum (two cross-lane adds) and
//    the normalisation happen on those accumulator registers; P.V consumes them
//    directly;
//  * K tiles arrive [head_dim][keys] and V tiles [keys][dv], both with the MFMA's
//    reduction index strided in memory, so they are transposed once while being
//    staged into LDS (four 16-byte global reads -> eight 8-byte LDS writes per 4x8
//    patch) and every operand fetch is one contiguous LDS read.  LDS rows are
//    unpadded; 16-byte chunks are XOR-swizzled with (row ^ row>>3) & 7, which makes
//    both the transposing writes and the operand reads spread over all banks;
//  * as many for-loop iterations as fit are staged per barrier, and every load of
//    a staging step is issued before the first one is waited for;
//  * the for-loop accumulators live in VGPRs (fp16-rounded each iteration, as the
//    reference's generated programs do) and are written once, through LDS, as full
//    16-byte row segments.
//
// This file is the host side: it recognises the family in a lowered program, chooses kernel
// and launch shape and either launches or, for Graph::generate_hip_program, prints the launch
// as source.  The kernels are in include/mi355_kernels/attention.h, which generated
// programs include as well.
#include "common.h"
#include "tb_program.h"
#include "attn_launch.h"
#include "attn_tiles.h"
#include <algorithm>
#include <cstdlib>
#include <string>

#include "mi355_kernels/attention.h"

namespace mi355 {

// ---------------------------------------------------------------------------------------
// host: recognise the family in a lowered program and launch
// ---------------------------------------------------------------------------------------
namespace {

// (a column-major tensor -- DevOp::sub == 1 on its loader -- holds element (r, c) at
// c * d_rows + r: a step along the rows is one element, a step along the columns d_rows, and
// `d_cols` of the result is that leading dimension)
// `fits` is cleared when a tile origin could leave 31 bits (the kernels multiply and add the
// strides in 32 bits); `extents` = the plan's grid and its for-loop range.
TileAddr tile_addr(DevOp const &op, void const *ptr, int const (&extents)[4], bool &fits) {
  TileAddr t;
  t.ptr = ptr;
  bool const cm = op.kind == DOP_LOAD && op.sub == 1;
  long long const rstep = cm ? 1 : op.d_cols, cstep = cm ? op.d_rows : 1;
  long long lin[4];
  for (int i = 0; i < 3; i++) {
    lin[i] = op.g_bs[i] + op.row_bs[i] * rstep + op.col_bs[i] * cstep;
  }
  lin[3] = op.g_fs + op.row_fs * rstep + op.col_fs * cstep;
  long long reach = 0;
  for (int i = 0; i < 4; i++) {
    long long const a = lin[i] < 0 ? -lin[i] : lin[i];
    if (a >= (1LL << 31)) {
      fits = false;
    }
    reach += a * (extents[i] > 0 ? extents[i] - 1 : 0);
    t.lin[i] = (int)lin[i];
  }
  if (reach >= (1LL << 31)) {
    fits = false;
  }
  t.d_cols = cm ? op.d_rows : op.d_cols;
  return t;
}

// The parameter block as C++ source (for programs that Graph::generate_hip_program writes).
std::string literal(TileAddr const &t) {
  return emit_fmt("mi355::TileAddr{%s, {%d, %d, %d, %d}, %d}", emit_pointer(t.ptr).c_str(), t.lin[0], t.lin[1],
                  t.lin[2], t.lin[3], t.d_cols);
}
std::string literal(AttnParams const &A) {
  std::string t = "    mi355::AttnParams P{};\n";
  t += "    P.q = " + literal(A.q) + ";\n    P.k = " + literal(A.k) + ";\n    P.v = " + literal(A.v) + ";\n";
  t += "    P.o = " + literal(A.o) + ";\n    P.r = " + literal(A.r) + ";\n";
  t += emit_fmt("    P.forloop_range = %d;\n    P.split = %d;\n    P.stages = %d;\n    P.lds_stage_bytes = %d;\n",
                A.forloop_range, A.split, A.stages, A.lds_stage_bytes);
  for (int i = 0; i < 3; i++) {
    t += emit_fmt("    P.perm[%d] = %d;\n    P.perm_ext[%d] = %uu;\n    P.perm_magic[%d] = %uu;\n", i, A.perm[i], i,
                  A.perm_ext[i], i, A.perm_magic[i]);
  }
  t += emit_fmt("    P.split_magic = %uu;\n    P.rows = %d;\n    P.trace = nullptr;\n    P.r_copies = %d;\n"
                "    P.r_copy_stride = %d;\n    P.in_order = %d;\n", A.split_magic, A.rows, A.r_copies, A.r_copy_stride, A.in_order);
  return t;
}

struct Match {
  int q, k, v;        // load op indices
  int out_o, out_r;   // output op indices (out_r < 0 in form A)
  bool has_div;
  int m, D, NK, DV;
  // K and V are both DmemColumnMajor (the layout every attention plan of the reference declares,
  // e.g. cpp_examples/group_query_attn_inc_decode.cc:41-44): K [D][keys] is then stored key by key
  // with the head dim contiguous, V [keys][DV] column by column with the keys contiguous, so both
  // tiles arrive with the MFMA's reduction index contiguous and no read transposes anything
  bool kv_colmajor;
};

// `pieces`: the value tile may be narrower than 16 bytes (checked by merge_column_pieces)
bool match(DevProgram const &P, Match &M, bool pieces = false) {
  if (has_column_major_saver(P) || P.num_ops < 9 || P.ops[0].kind != DOP_LOAD || P.ops[1].kind != DOP_LOAD ||
      P.ops[2].kind != DOP_LOAD || P.ops[3].kind != DOP_MATMUL) {
    return false;
  }
  auto loader_of = [&](int tensor) {
    for (int i = 0; i < 3; i++) {
      if (P.ops[i].dst == tensor) {
        return i;
      }
    }
    return -1;
  };
  DevOp const &mm1 = P.ops[3];
  DevOp const &ex = P.ops[4];
  M.q = loader_of(mm1.src0);
  M.k = loader_of(mm1.src1);
  if (M.q < 0 || M.k < 0 || M.q == M.k || ex.kind != DOP_UNARY || ex.sub != TB_EXP_OP ||
      ex.dst != mm1.dst) {
    return false;
  }
  int const E = mm1.dst;
  auto is_rowsum = [&](DevOp const &op) {
    return op.kind == DOP_REDUCE && op.src0 == E && P.t[op.dst].cols == 1 &&
           P.t[op.dst].rows == P.t[E].rows && op.red_inner == 1 && op.red_deg == P.t[E].cols;
  };
  int mm2 = -1, red = -1;
  if (P.num_ops == 9 && is_rowsum(P.ops[5]) && P.ops[6].kind == DOP_BINARY &&
      P.ops[6].sub == TB_DIV_OP && P.ops[6].src0 == E && P.ops[6].src1 == P.ops[5].dst &&
      P.ops[7].kind == DOP_MATMUL && P.ops[7].src0 == P.ops[6].dst &&
      P.ops[8].kind == DOP_OUTPUT && P.ops[8].src0 == P.ops[7].dst) {
    M.has_div = true;
    mm2 = 7;
    M.out_o = 8;
    M.out_r = -1;
  } else if (P.num_ops == 9 && P.ops[7].kind == DOP_OUTPUT && P.ops[8].kind == DOP_OUTPUT) {
    if (P.ops[5].kind == DOP_MATMUL && is_rowsum(P.ops[6])) {
      mm2 = 5;
      red = 6;
    } else if (is_rowsum(P.ops[5]) && P.ops[6].kind == DOP_MATMUL) {
      mm2 = 6;
      red = 5;
    } else {
      return false;
    }
    if (P.ops[mm2].src0 != E) {
      return false;
    }
    M.has_div = false;
    M.out_o = M.out_r = -1;
    for (int o = 7; o <= 8; o++) {
      if (P.ops[o].src0 == P.ops[mm2].dst) {
        M.out_o = o;
      } else if (P.ops[o].src0 == P.ops[red].dst) {
        M.out_r = o;
      }
    }
    if (M.out_o < 0 || M.out_r < 0) {
      return false;
    }
  } else {
    return false;
  }
  M.v = loader_of(P.ops[mm2].src1);
  if (M.v < 0 || M.v == M.q || M.v == M.k) {
    return false;
  }
  DevTensor const &tq = P.t[P.ops[M.q].dst], &tk = P.t[P.ops[M.k].dst], &tv = P.t[P.ops[M.v].dst];
  M.m = tq.rows;
  M.D = tq.cols;
  M.NK = tk.cols;
  M.DV = tv.cols;
  if (tk.rows != M.D || tv.rows != M.NK) {
    return false;
  }
  // Q must be loop invariant; all tiles reachable with 16-byte accesses
  DevOp const &lq = P.ops[M.q];
  if (lq.row_fs != 0 || lq.col_fs != 0 || lq.g_fs != 0) {
    return false;
  }
  // Q row-major; K and V in one storage order (a mixed pair takes the interpreter)
  if (lq.sub == 1 || P.ops[M.k].sub != P.ops[M.v].sub) {
    return false;
  }
  M.kv_colmajor = P.ops[M.k].sub == 1;
  if (!lq.galign || !P.ops[M.k].galign ||
      (!pieces && (!P.ops[M.v].galign || !P.ops[M.out_o].galign))) {
    return false;
  }
  for (void const *p : {P.in[lq.io], P.in[P.ops[M.k].io], P.in[P.ops[M.v].io],
                        (void const *)P.out[P.ops[M.out_o].io]}) {
    if ((reinterpret_cast<uintptr_t>(p) & 15) != 0) {
      return false;
    }
  }
  return true;
}

// A plan that cuts the value columns into pieces along one grid dimension -- every block of
// that dimension loads the same Q and K tiles, takes DV / G columns of V, stores its columns of
// the result and, in the row-sum form, its own copy of the same row sums -- computes the scores
// G times.  Column j of the result depends on column j of V only, so the G blocks are one block
// with the whole value tile: Q gets that program (grid dimension `g` of extent 1, V and the
// result 64 columns wide, the row sums stored G times).  False when P is not of this shape.
bool merge_column_pieces(DevProgram const &P, Match &M, DevProgram &Q, int &copies, int &copy_stride) {
  if (!match(P, M, true) || M.DV >= 64 || 64 % M.DV != 0) {
    return false;
  }
  int const G = 64 / M.DV;
  DevOp const &lq = P.ops[M.q], &lk = P.ops[M.k], &lv = P.ops[M.v], &oo = P.ops[M.out_o];
  for (int g = 0; g < 3; g++) {
    if (P.grid[g] != G) {
      continue;
    }
    auto free_of = [&](DevOp const &op) { return !op.row_bs[g] && !op.col_bs[g] && !op.g_bs[g]; };
    auto pieced = [&](DevOp const &op) { return !op.row_bs[g] && !op.g_bs[g] && op.col_bs[g] == M.DV; };
    if (!free_of(lq) || !free_of(lk) || !pieced(lv) || !pieced(oo)) {
      continue;
    }
    copies = 1;
    copy_stride = 0;
    if (M.out_r >= 0) {
      DevOp const &orr = P.ops[M.out_r];
      if (orr.row_bs[g] || orr.g_bs[g]) {
        continue;
      }
      copies = G;
      copy_stride = orr.col_bs[g];
    }
    Q = P;
    Q.grid[g] = 1;
    Q.ops[M.v].col_bs[g] = 0;
    Q.ops[M.out_o].col_bs[g] = 0;
    if (M.out_r >= 0) {
      Q.ops[M.out_r].col_bs[g] = 0;
    }
    // 16-byte reachability of the widened tiles
    for (int o : {M.v, M.out_o}) {
      DevOp &d = Q.ops[o];
      if (d.kind == DOP_LOAD && d.sub == 1) {
        // column-major V: a wider tile is more columns, i.e. more rows of V^T, each as
        // reachable with 16-byte accesses as before
        if (!d.galign) {
          return false;
        }
        Q.t[d.dst].cols = 64;
        continue;
      }
      bool al = d.d_cols % 8 == 0 && d.col_fs % 8 == 0 && d.g_fs % 8 == 0;
      for (int e = 0; e < 3; e++) {
        al = al && d.col_bs[e] % 8 == 0 && d.g_bs[e] % 8 == 0;
      }
      if (!al) {
        return false;
      }
      d.galign = d.vec8 = 1;
      Q.t[d.dst].cols = 64;
    }
    void const *vp = P.in[lv.io], *op = P.out[oo.io];
    if (((reinterpret_cast<uintptr_t>(vp) | reinterpret_cast<uintptr_t>(op)) & 15) != 0) {
      return false;
    }
    M.DV = 64;
    return true;
  }
  return false;
}

// A plan that cuts the query rows into tiles along a grid dimension K and V do not move with: row
// r of block i is row i m + r of one tall tile (every row is worked on by itself), so Q becomes
// that program -- grid dimension of extent 1, G m rows -- and no row group is left half empty at
// the end of every tile.  False when P is not of this shape.
bool merge_row_blocks(DevProgram const &P, Match &M, DevProgram &Q) {
  for (int g = 0; g < 3; g++) {
    int const G = P.grid[g];
    if (G < 2 || (long long)G * M.m > (1 << 24)) {
      continue;
    }
    auto still = [&](DevOp const &op) { return !op.row_bs[g] && !op.col_bs[g] && !op.g_bs[g]; };
    auto stacked = [&](DevOp const &op) { return op.row_bs[g] == M.m && !op.col_bs[g] && !op.g_bs[g]; };
    if (!still(P.ops[M.k]) || !still(P.ops[M.v]) || !stacked(P.ops[M.q]) || !stacked(P.ops[M.out_o]) ||
        (M.out_r >= 0 && !stacked(P.ops[M.out_r]))) {
      continue;
    }
    Q = P;
    Q.grid[g] = 1;
    for (int o : {M.q, M.out_o, M.out_r}) {
      if (o >= 0) {
        Q.ops[o].row_bs[g] = 0;
      }
    }
    M.m *= G;
    return true;
  }
  return false;
}

}  // namespace

// Fills the division magics decode_block uses for this launch grid; false when an id times an
// extent could leave 32 bits (the magics are exact only below that).
//
// The order of blocks: an XCD has a run of them that share K and V, also where eight does not divide their number
// (us of an operator again and again / of a pass on changing inputs, launch order and runs: prefill of 11 heads of 9 row
// blocks, head size 128, row-major, 70.7 and 62.5 / 74.3 and 73.9, of 13 of 5 40.6 and 35.9 / 44.3 and 44.3; column-major
// and head size 64 within 2 %; decoding within 0.05 us).  K and V that nobody shares and the last-level cache does not
// keep (`streamed` bytes) go in launch order, neighbours in memory side by side over all XCDs; the next row of DRAM
// is then asked for while the one before is open.  64 groups of 16,384 keys (268 MB) 57.0 us as runs, 50.6 in launch
// order, in blocks of 512 keys 65.8 and 50.6; 134 MB 30.5 and 28.7; 67 MB (two row groups) 16.0 and 18.2.
static bool set_grid_magics(AttnParams &A, dim3 grid, long long streamed) {
  if (streamed >= (128ll << 20) && A.split == 1) {
    std::stable_sort(A.perm, A.perm + 3, [&](int x, int y) {
      return std::llabs((long long)A.k.lin[x]) + std::llabs((long long)A.v.lin[x]) <
             std::llabs((long long)A.k.lin[y]) + std::llabs((long long)A.v.lin[y]);
    });
    A.in_order = 1;
  }
  unsigned const ext[3] = {grid.x, grid.y, grid.z};
  unsigned long long const total = (unsigned long long)grid.x * grid.y * grid.z;
  for (int i = 0; i < 3; i++) {
    unsigned const e = ext[A.perm[i]];
    if (total * e >= (1ull << 32)) {
      return false;
    }
    A.perm_ext[i] = e;
    A.perm_magic[i] = fast_div_magic((int)e);
  }
  if ((unsigned long long)grid.x * (unsigned)A.split >= (1ull << 32)) {
    return false;
  }
  A.split_magic = fast_div_magic(A.split);
  return true;
}

// Shapes the register-transposed and the throughput variants are built for.
static bool shape_supported(Match const &M) {
  return (M.m % 16 == 0 || M.m == 8) &&
         ((M.D == 64 && M.DV == 64 && (M.NK == 64 || M.NK == 128 || M.NK == 256)) ||
          (M.D == 128 && M.DV == 128 && M.NK == 64));
}

// Whether (and in which shape) the direct-staging variant takes the plan: head size 64,
// key tiles of 16 ... 256 on 64-key strips.
static bool choose_direct(DevProgram const &P, Match const &M, DirectShape &d, int &lds) {
  State &s = state();
  if (M.D != 64 || M.DV != 64 || s.attention_mode == 3 || !(M.m % 16 == 0 || M.m == 8)) {
    return false;
  }
  int const F = P.forloop_range;
  d = DirectShape{};
  if (M.NK == 16 || M.NK == 32) {
    // consecutive iterations' tiles must lie side by side: K advances by NK columns, V by NK rows
    DevOp const &lk = P.ops[M.k], &lv = P.ops[M.v];
    d.ips = 64 / M.NK;
    if (lk.col_fs != M.NK || lk.row_fs != 0 || lk.g_fs != 0 || lv.row_fs != M.NK || lv.col_fs != 0 ||
        lv.g_fs != 0 || F % d.ips != 0) {
      return false;
    }
  } else if (M.NK == 128 || M.NK == 256) {
    d.spi = M.NK / 64;
    if (M.has_div) {
      return false;
    }
  } else if (M.NK != 64) {
    return false;
  }
  int const units = F / d.ips;
  int const groups = (M.m + 15) / 16;
  long long const blocks = (long long)P.grid[0] * P.grid[1] * P.grid[2];
  auto round_nit = [](int per) { return per <= 1 ? 1 : (per <= 2 ? 2 : (per <= 4 ? 4 : 8)); };
  if ((groups == 1 && units > 1) || units > 8) {
    // a lone row group (or a loop too long for a wavefront per unit: then every row group is
    // a workgroup of its own): eight lanes with a tile pair each; four when the grid is large
    // enough to put two workgroups on every compute unit; or (DIRECT_LANES = 4, whole-tile
    // iterations only) four lanes with two tile pairs each
    int const per8 = (units + 7) / 8, per4 = (units + 3) / 4;
    if (s.direct_lanes == 4 && d.spi == 1 && d.ips == 1 && per4 <= 8 && units > 4) {
      d.ip = 4;
      d.nbuf = 2;
      d.nit = round_nit(per4) < 2 ? 2 : round_nit(per4);
    } else if (units <= 4 && d.spi == 1) {
      d.ip = units <= 2 ? 2 : 4;
      if (d.ips > 1) {
        d.ip = 4;
      }
    } else if (s.direct_lanes == 0 && blocks >= 512 && units > 4 && per4 <= 8 && d.spi == 1 && d.ips == 1) {
      // enough blocks for two workgroups on every compute unit: four single-buffered lanes (half
      // the LDS), so that one workgroup streams while its neighbour starts up or adds up its
      // results (the HBM-bound decode: 5.75 -> 6.3 TB/s)
      d.ip = 4;
      d.nit = round_nit(per4);
    } else {
      d.ip = 8;
      d.nit = round_nit(per8);
    }
  } else if (units >= 1 && units <= 8 && (groups > 1 || units == 1)) {
    // every unit on a wavefront of its own, one slab of one or two row groups per workgroup
    d.ip = units <= 2 && d.ips == 1 && d.spi == 1 ? 2 : (units <= 4 ? 4 : 8);
    if (d.ip == 4 && d.spi == 1 && groups % 2 == 0 && blocks * (groups / 2) >= 256 && s.direct_lanes != 1) {
      d.rpw = 2;
    }
    if (d.ip == 2 && units == 1) {
      return false;  // a single iteration: nothing to hand over, the other variants serve it
    }
  } else {
    return false;
  }
  int const pair_bytes = (64 * 64 + 64 * 64) * 2;
  lds = d.ip * (d.nbuf * pair_bytes + d.rpw * 16 * M.D * 2);  // + a Q tile per wavefront
  if (lds > s.max_lds || (long long)P.grid[0] * (groups / d.rpw) > 2147483647LL) {
    return false;
  }
  AttnParams none{};
  return (M.has_div ? launch_direct<true, false>(none, dim3(1, 1, 1), d, lds, true)
                    : launch_direct<false, false>(none, dim3(1, 1, 1), d, lds, true)) == 1;
}

// Whether (and in which shape) the throughput variant takes the plan: query tiles of whole
// 64- or 128-row slabs, enough of them to fill the chip twice over, a for-loop long enough to
// pipeline; key tiles of 64 keys, or (the form without the division, 128-row slabs) of 128 / 256 /
// 512 keys walked as strips of 64.
struct StreamShape {
  int rgs = 0, spi = 1;
  bool wide = false;
};
static bool choose_stream(DevProgram const &P, Match const &M, StreamShape &st) {
  State &s = state();
  st = StreamShape{};
  if (s.attention_mode == 1 || s.attention_mode == 3) {
    return false;
  }
  long long const blocks_all = (long long)P.grid[0] * P.grid[1] * P.grid[2];
  int const slabs = M.m / 32;
  st.rgs = (M.m % 128 == 0) ? 4 : ((M.m % 64 == 0) ? 2 : 0);
  bool const heads = (M.D == 64 && M.DV == 64) || (M.D == 128 && M.DV == 128);
  if (st.rgs == 0 || !heads) {
    return false;
  }
  if (M.NK == 128 || M.NK == 256 || M.NK == 512) {
    st.spi = M.NK / 64;
    if (M.has_div || st.rgs != 4) {
      return false;
    }
  } else if (M.NK != 64) {
    return false;
  }
  // (64-key tiles on a small grid are better served by the latency variants; wider key tiles
  // have no other kernel, so they take this one whatever the grid)
  if (s.attention_mode != 2 && st.spi == 1 &&
      !(P.forloop_range >= 2 && blocks_all * (slabs / st.rgs) >= 512)) {
    return false;
  }
  // Head size 64 with 256-row query tiles and enough of them for two wavefronts per SIMD:
  // wavefronts of 64 rows (half the LDS operand reads per MFMA; at head size 64 the registers
  // still fit two wavefronts per SIMD).  Measured on the 32-group x 16,384-key decode plan:
  // 68.8 -> 67.0 us.
  st.wide = st.spi == 1 && M.D == 64 && M.m % 256 == 0 &&
            (s.attention_mode == 2 || blocks_all * (M.m / 64) >= 2048);
  if (st.wide) {
    st.rgs = 8;
  }
  return true;
}

std::string attn_params_literal(AttnParams const &A) { return literal(A); }

static bool choose_tiles(DevProgram const &P, Match const &M, TilesShape &t) {
  State &s = state();
  long long const blocks = (long long)P.grid[0] * P.grid[1] * P.grid[2];
  return choose_attn_tiles(M.D, M.DV, M.NK, M.m, M.has_div, M.kv_colmajor, blocks, P.forloop_range, s.max_lds, t) &&
         (long long)P.grid[0] * t.split <= 2147483647LL;
}

bool attention_applicable(DevProgram const &P) {
  Match M;
  DirectShape d;
  StreamShape st;
  TilesShape tiles;
  int lds = 0;
  if (match(P, M) && (shape_supported(M) || choose_stream(P, M, st) || choose_direct(P, M, d, lds) ||
                      choose_tiles(P, M, tiles))) {
    return true;
  }
  DevProgram merged;
  int copies = 1, stride = 0;
  return merge_column_pieces(P, M, merged, copies, stride) && choose_direct(merged, M, d, lds);
}

// What the next operator's fold of rows is to this launch: a workgroup's rows, and the places of its
// results in them.  False where the operator is no fold of exactly these results, row by row.
//
// With whole rows in a workgroup it always pays: both launches of [12, 1040, 1040] in tiles of 80 18.9 -> 16.7 us, of
// [32, 2048, 2048] at head size 128 80.2 -> 77.6 (both tensors' stores are what is left), 60 prefill plans 0.76 of the
// time on the device in the mean, none above 1.  Where the pieces come from several workgroups the last of them pays three trips to the
// memory that all XCDs share (its stores, its ticket, the pieces), 3 us against the 3.5 - 4.5 of a launch, and all others two while
// they hold their place on a compute unit.  So: blocks that run in one round (64 groups of 16 blocks, two rounds, 50.8
// us either way, folded 52.1), as many columns of threads as there are columns, and sixteen pieces, what a thread loads
// together (7 groups of 16 rows, 20 pieces, one wavefront 8.8 us, folded 12.5).
// Nor where the other launch is short and many workgroups pay for it.  It adds up pieces in batches of four, or of sixteen
// where there are so many (combine.h), and what is left over piece by piece: for four and sixteen, and for two, it has one
// trip to make.  Of one row each there is little but that trip: from 32 workgroups on 46 plans of four or sixteen pieces take
// 1.05 of the time on the device in the mean when folded (16 groups, 4 pieces of 10 tiles of 16 keys 8.23 / 8.73 us, 33
// groups, 16 pieces of a tile of 48 7.85 / 8.96), 14 of two 1.01; other numbers of pieces less.  From eight iterations on the
// host's second launch is hidden by the device's work, and the line is nearer: 24 workgroups (7 groups, 4 pieces of 13 tiles of 32
// keys, passes back to back, 8.50 / 8.93), 48 where the other launch makes two or three trips (18 groups, 5 pieces of 16 tiles of 32 9.40 /
// 9.78, 12 groups, 8 of 11 tiles of 16 8.93 / 9.28; four trips and more, 7 pieces, 21 groups of 12 tiles of 64, 12.73 / 12.08).  Below
// these lines 86 plans of one row take 0.98 of the time of two launches, 0.88 - 1.02.  Of more rows so it is for
// sixteen pieces and more than 128 workgroups, 40 plans 1.08 (20 groups of 16 rows, 7 tiles of 16 keys 9.11 / 11.02; 95 with
// up to 128 0.97); for 4, 8 and 12 pieces and more than 192 workgroups it comes to the same, 0.90 - 1.14 of the time.
// 435 other drawn split-KV plans 0.92 of the time on the device in the mean, 0.60 - 1.08, twenty above 1.01.
// [5, 12, 64] against 12 pieces of 5 tiles of 48 keys 8.4 -> 7.9.
static bool make_fold(AttnParams const &A, Match const &M, DevProgram const &P, int wg_rows, int threads, int lds, FoldRequest &f,
                      AttnFold &out) {
  RowFold const &R = f.rows;
  int const C = R.S * R.X;
  if (M.out_r < 0 || A.r_copies != 1 || state().phase_trace != nullptr || A.o.ptr != R.n || A.r.ptr != R.d || R.X != M.DV || A.o.d_cols != C || A.r.d_cols != R.SD ||
      R.SD != R.S || (R.S > 1 && R.mode != SUM_THEN_DIV) || (long long)C * R.rows >= (1LL << 31)) {
    return false;
  }
  // One grid dimension may cut the columns: piece after piece, row sum after row sum.  The others cut the rows.
  long long stride[3];
  int extent[3], row_dims = 0, pieces = 1;
  for (int i = 0; i < 3; i++) {
    out.lin[i] = out.ticket_lin[i] = 0;
    if (P.grid[i] == 1) {
      continue;
    }
    if (R.S > 1 && pieces == 1 && A.o.lin[i] == R.X && A.r.lin[i] == 1 && P.grid[i] == R.S) {
      pieces = P.grid[i];
      continue;
    }
    if (A.o.lin[i] % C != 0 || A.r.lin[i] % R.SD != 0 || A.o.lin[i] / C != A.r.lin[i] / R.SD || A.o.lin[i] / C % M.m != 0) {
      return false;
    }
    out.lin[i] = A.o.lin[i] / C;
    out.ticket_lin[i] = out.lin[i] / M.m * A.split;
    stride[row_dims] = out.lin[i];
    extent[row_dims++] = P.grid[i];
  }
  long long rows = 0;
  if (pieces != R.S || !covers_rows(M.m, stride, extent, row_dims, rows) || rows != R.rows) {
    return false;
  }
  // (what the fold writes is read by no other workgroup of this launch)
  uintptr_t const o0 = reinterpret_cast<uintptr_t>(R.o), o1 = o0 + ((size_t)(R.rows - 1) * R.o_cols + R.X) * 2;
  for (void const *p : {A.q.ptr, A.k.ptr, A.v.ptr, A.o.ptr, A.r.ptr}) {
    if (reinterpret_cast<uintptr_t>(p) >= o0 && reinterpret_cast<uintptr_t>(p) < o1) {
      return false;
    }
  }
  out.n = static_cast<_Float16 const *>(R.n);
  out.d = static_cast<_Float16 const *>(R.d);
  out.o = static_cast<_Float16 *>(R.o);
  out.arrivals = R.S;
  out.S = R.S;
  out.X = R.X;
  out.o_cols = R.o_cols;
  out.mxv = fast_div_magic(R.X / 4);
  out.after = R.mode == SUM_THEN_DIV ? -0.0f : 0.0f;
  out.tickets = nullptr;
  if (R.S > 1) {
    int const per_cu = std::max(1, std::min(state().max_lds / std::max(lds, 1), 1024 / threads));
    int const trips = (std::min(wg_rows, M.m) * R.X / 4 + threads - 1) / threads;
    long long const workgroups = (long long)P.grid[0] * P.grid[1] * P.grid[2] * A.split;
    if (R.S > kFoldPieces || trips > (R.S <= 8 ? 2 : 1) || wg_rows * R.S * 2 + 16 > lds || workgroups > 256 * per_cu) {
      return false;
    }
    int const other = R.S == 16 ? 1 : R.S / 4 + R.S % 4;  // trips of the other launch
    bool const one_trip = R.S == 2 || other == 1;         // (of two the first is loaded ahead)
    int const most = one_trip ? (P.forloop_range < 8 ? 32 : 24) : other <= 3 && P.forloop_range >= 8 ? 48 : 1 << 30;
    if ((M.m == 1 && workgroups >= most) || (R.S == 16 && workgroups > 128) || (R.S % 4 == 0 && workgroups > 192)) {
      return false;
    }
    out.tickets = f.tickets(R.rows / M.m * A.split);
    if (out.tickets == nullptr) {
      return false;
    }
  }
  return true;
}

int try_launch_attention(DevProgram const &P0, FoldRequest *fold) {
  Match M;
  DevProgram merged;
  DevProgram const *run = &P0;
  int r_copies = 1, r_copy_stride = 0;
  // as the plan states it, or (value tiles narrower than 64 columns) with its column pieces merged
  bool pieces = !match(P0, M);
  TilesShape tiles_shape;
  bool tiles = false;
  if (!pieces) {
    DirectShape probe;
    StreamShape probe_stream;
    int probe_lds = 0;
    pieces = !shape_supported(M) && !choose_stream(P0, M, probe_stream) &&
             !choose_direct(P0, M, probe, probe_lds);
    if (pieces || state().any_size_kernels) {
      // sizes the kernels of whole tiles are not built for: any-size kernel, row tiles joined
      Match T = M;
      DevProgram tall;
      bool const joined = merge_row_blocks(P0, T, tall);
      tiles = choose_tiles(joined ? tall : P0, T, tiles_shape);
      if (tiles) {
        pieces = false;
        M = T;
        if (joined) {
          merged = tall;
          run = &merged;
        }
      }
    }
  }
  if (pieces) {
    if (!merge_column_pieces(P0, M, merged, r_copies, r_copy_stride)) {
      return 0;
    }
    run = &merged;
  }
  DevProgram const &P = *run;
  DirectShape dshape;
  int direct_lds = 0;
  bool const direct = !tiles && choose_direct(P, M, dshape, direct_lds);
  StreamShape stream_probe;
  bool const stream = !tiles && !pieces && choose_stream(P, M, stream_probe);
  if (!tiles && !direct && !stream && (pieces || !shape_supported(M))) {
    return 0;  // (only the direct-staging variant stores copies of the row sums)
  }
  State &s = state();
  AttnParams A;
  A.in_order = 0;
  A.r_copies = r_copies;
  A.r_copy_stride = r_copy_stride;
  int const extents[4] = {P.grid[0], P.grid[1], P.grid[2], P.forloop_range};
  bool fits = true;
  A.q = tile_addr(P.ops[M.q], P.in[P.ops[M.q].io], extents, fits);
  A.k = tile_addr(P.ops[M.k], P.in[P.ops[M.k].io], extents, fits);
  A.v = tile_addr(P.ops[M.v], P.in[P.ops[M.v].io], extents, fits);
  A.o = tile_addr(P.ops[M.out_o], P.out[P.ops[M.out_o].io], extents, fits);
  A.r = M.out_r >= 0 ? tile_addr(P.ops[M.out_r], P.out[P.ops[M.out_r].io], extents, fits) : A.o;
  if (!fits) {
    return 0;  // a tensor of more than 2^31 elements: the generic interpreter takes the plan
  }
  A.forloop_range = P.forloop_range;
  A.rows = M.m < 16 ? M.m : 16;
  A.trace = nullptr;
  long long streamed;  // bytes of K and V if every block has its own
  {
    // grid dims the K / V tiles do not depend on vary fastest in the workgroup id
    int n = 0;
    bool dep[3];
    for (int d = 0; d < 3; d++) {
      DevOp const &lk = P.ops[M.k], &lv = P.ops[M.v];
      dep[d] = lk.row_bs[d] || lk.col_bs[d] || lk.g_bs[d] || lv.row_bs[d] || lv.col_bs[d] || lv.g_bs[d];
    }
    for (int d = 0; d < 3; d++) {
      if (!dep[d]) {
        A.perm[n++] = d;
      }
    }
    for (int d = 0; d < 3; d++) {
      if (dep[d]) {
        A.perm[n++] = d;
      }
    }
    bool const shared = (!dep[0] && P.grid[0] > 1) || (!dep[1] && P.grid[1] > 1) || (!dep[2] && P.grid[2] > 1);
    streamed = shared ? 0 : (long long)P.grid[0] * P.grid[1] * P.grid[2] * P.forloop_range * M.NK * (M.D + M.DV) * 2;
  }
  // ---- any tile size
  if (tiles) {
    A.split = tiles_shape.split;
    A.rows = M.m;
    A.stages = M.NK;
    A.lds_stage_bytes = 0;
    if (A.k.d_cols >= (1 << 24) || A.v.d_cols >= (1 << 24)) {
      return 0;  // (offsets inside a tile are 32-bit: up to 128 rows of the tensor)
    }
    dim3 const grid(P.grid[0] * A.split, P.grid[1], P.grid[2]);
    if (!set_grid_magics(A, grid, streamed)) {
      return 0;
    }
    AttnFoldParams F;
    if (fold != nullptr && !make_fold(A, M, P, 16 * tiles_shape.rpw, 64 * tiles_shape.ip, tiles_shape.lds, *fold, F.fold)) {
      return 0;
    }
    F.attn = A;
    int const rc = fold != nullptr ? launch_attn_tiles_fold(F, grid, M.D, M.kv_colmajor, tiles_shape)
                                   : launch_attn_tiles(A, grid, M.D, M.has_div, M.kv_colmajor, tiles_shape);
    if (rc == 1) {
      s.last().kernel_id = MI355_KERNEL_F16_ATTENTION;
      s.last().workgroups = grid.x * grid.y * grid.z;
      s.last().threads = 64 * tiles_shape.ip;
      s.last().lds_bytes = tiles_shape.lds;
      s.last().row_split = A.split;
    }
    return rc;
  }
  // ---- throughput variant
  {
    StreamShape st;
    if (!pieces && choose_stream(P, M, st)) {
      int const slabs = M.m / 32, rgs = st.rgs;
      A.split = slabs / rgs;
      A.stages = 2;
      A.lds_stage_bytes = (64 * M.D + M.DV * 64) * 2;  // one strip of 64 keys of K and of V
      int const out_bytes = rgs * 32 * (M.DV + 8) * 2;
      int lds = 2 * A.lds_stage_bytes;
      lds = lds > out_bytes ? lds : out_bytes;
      if (lds <= s.max_lds && (long long)P.grid[0] * A.split <= 2147483647LL) {
        dim3 grid(P.grid[0] * A.split, P.grid[1], P.grid[2]);
        if (!set_grid_magics(A, grid, streamed)) {
          return 0;
        }
        AttnShape const shape{M.D, M.NK, M.kv_colmajor, rgs, 1, lds, st.spi, st.wide};
        AttnFoldParams F;
        if (fold != nullptr && !make_fold(A, M, P, 32 * rgs, st.wide ? 256 : 64 * rgs, lds, *fold, F.fold)) {
          return 0;
        }
        F.attn = A;
        int const rc = fold != nullptr ? launch_stream_fold(F, grid, shape)
                       : M.has_div     ? launch_stream_shape<true>(A, grid, shape)
                                       : launch_stream_shape<false>(A, grid, shape);
        if (rc == 1) {
          s.last().kernel_id = MI355_KERNEL_F16_ATTENTION;
          s.last().workgroups = grid.x * grid.y * grid.z;
          s.last().threads = st.wide ? 256 : rgs * 64;
          s.last().lds_bytes = lds;
          s.last().row_split = A.split;
        }
        if (rc != 0) {
          return rc;
        }
      }
    }
  }

  // ---- direct-staging variant (attention mode 3 keeps the register-transposed staging):
  // head size 64, key tiles of 16 ... 256, in two situations.
  // (a) Every unit of work (an iteration, or a 64-key strip of several) has a wavefront of
  //     its own.  A wavefront takes two row groups when that still puts a workgroup on every
  //     compute unit: each K / V operand read from LDS then feeds two MFMAs and half as many
  //     wavefronts stream the tiles (C2: 256 workgroups of 4 wavefronts x 32 rows; the
  //     L2 -> LDS traffic and the LDS reads, both per-CU bandwidth limits at this size, halve).
  // (b) A lone row group (decode: 8 or 16 query rows) with a longer for-loop: eight
  //     wavefronts that each stream every eighth unit through a tile pair of their own, or
  //     (DIRECT_LANES = 4) four wavefronts with two tile pairs each.
  if (direct) {
    int const groups = (M.m + 15) / 16;
    AttnParams B = A;
    B.split = groups / dshape.rpw;
    B.trace = s.phase_trace;
    dim3 const direct_grid(P.grid[0] * B.split, P.grid[1], P.grid[2]);
    if (set_grid_magics(B, direct_grid, streamed)) {
      if (B.trace != nullptr && (size_t)direct_grid.x * direct_grid.y * direct_grid.z * dshape.ip * 6 * 8 >
                                    s.phase_trace_bytes) {
        B.trace = nullptr;
      }
      AttnFoldParams F;
      if (fold != nullptr && !make_fold(B, M, P, 16 * dshape.rpw, 64 * dshape.ip, direct_lds, *fold, F.fold)) {
        return 0;
      }
      F.attn = B;
      int const rc = fold != nullptr ? launch_direct_fold(F, M.kv_colmajor, direct_grid, dshape, direct_lds)
                     : M.kv_colmajor
                         ? (M.has_div ? launch_direct<true, true>(B, direct_grid, dshape, direct_lds)
                                      : launch_direct<false, true>(B, direct_grid, dshape, direct_lds))
                         : (M.has_div ? launch_direct<true, false>(B, direct_grid, dshape, direct_lds)
                                      : launch_direct<false, false>(B, direct_grid, dshape, direct_lds));
      if (rc != 0) {
        if (rc == 1) {
          s.last().kernel_id = MI355_KERNEL_F16_ATTENTION;
          s.last().workgroups = direct_grid.x * direct_grid.y * direct_grid.z;
          s.last().threads = dshape.ip * 64;
          s.last().lds_bytes = direct_lds;
          s.last().row_split = B.split;
        }
        return rc;
      }
    }
    if (pieces || !shape_supported(M)) {
      return 0;
    }
  }

  if (pieces || !shape_supported(M)) {
    return 0;  // (a shape only the throughput variant is built for)
  }
  // Row groups per workgroup: up to 4, fewer when that is what it takes to put a
  // workgroup on every compute unit.  Iteration lanes: whatever is left of 8
  // wavefronts, at most the for-loop range.
  int const groups = (M.m + 15) / 16;
  int rg = groups % 4 == 0 ? 4 : (groups % 2 == 0 ? 2 : 1);
  long long const blocks = (long long)P.grid[0] * P.grid[1] * P.grid[2];
  while (rg > 1 && blocks * (groups / rg) < 256) {
    rg /= 2;
  }
  int ip = 1;
  while (ip * 2 * rg <= 8 && ip * 2 <= P.forloop_range) {
    ip *= 2;
  }
  A.split = groups / rg;
  if ((long long)P.grid[0] * A.split > 2147483647LL) {
    return 0;
  }
  int const stage_bytes = (M.NK * M.D + M.DV * M.NK) * 2;
  int const tail_bytes = rg * 16 * (M.DV + 8) * 2 + rg * (ip - 1) * (M.DV / 8 + 1) * 64 * 4;
  int stages = (96 * 1024 - tail_bytes) / stage_bytes;
  stages = stages < 1 ? 1 : (stages > P.forloop_range ? P.forloop_range : stages);
  if (stages >= ip) {
    stages -= stages % ip;  // whole rounds per staging step
  } else {
    ip = 1;
    while (ip * 2 <= stages) {
      ip *= 2;
    }
    stages = ip;
  }
  A.stages = stages;
  A.lds_stage_bytes = stage_bytes;
  int lds = stages * stage_bytes + tail_bytes;
  if (lds > s.max_lds) {
    return 0;
  }
  dim3 grid(P.grid[0] * A.split, P.grid[1], P.grid[2]);
  int const nw = rg * ip;
  int rc = 0;
  if (!set_grid_magics(A, grid, streamed)) {
    return 0;
  }
  AttnShape const shape{M.D, M.NK, M.kv_colmajor, rg, ip, lds};
  AttnFoldParams F;
  if (fold != nullptr && !make_fold(A, M, P, 16 * rg, 64 * nw, lds, *fold, F.fold)) {
    return 0;
  }
  F.attn = A;
  rc = fold != nullptr ? launch_fused_fold(F, grid, shape)
       : M.has_div     ? launch_fused_shape<true>(A, grid, shape)
                       : launch_fused_shape<false>(A, grid, shape);
  if (rc == 1) {
    s.last().kernel_id = MI355_KERNEL_F16_ATTENTION;
    s.last().workgroups = grid.x * grid.y * grid.z;
    s.last().threads = nw * 64;
    s.last().lds_bytes = lds;
    s.last().row_split = A.split;
  }
  return rc;
}

}  // namespace mi355
