// Fused kernel for the skinny-GEMM family of thread-block graphs: a handful of rows
// of activations against streamed weight tiles, accumulated over the for-loop.
//
//   plain      O  = sum_i pro(A_i) . B_i                         pro in {id, exp, silu}
//   two-weight O1 = sum_i A_i . B1_i ;  O2 = sum_i A_i . B2_i    (gated MLP, first half)
//   gate       O  = sum_i (silu(G_i) * U_i) . B_i                (gated MLP, second half)
//   lora       O  = sum_i [X_i | X_i.A_i] . [W_i ; B]            (concat-then-matmul,
//                                                                 cpp_examples/lora.cc:45-67)
//
// These are HBM-bound: what matters is how many bytes of weights are in flight, not
// the MFMAs.  Three kernels.  gemm_lanes_kernel (further down) runs a plan in ONE launch with
// the output tile cut into 16 x 16 pieces, one workgroup each, whose wavefronts take the
// for-loop's iterations side by side; it serves the launch-bound members.  gemm_stream_kernel
// (gemm_stream.h) takes the ones whose weights' bytes cost: iterations of whole 64 k.
// gemm_fused_kernel takes the rest (iterations of 96 or 160 k, more rows than half of them);
// like the streaming kernel it cuts the for-loop and needs a second launch to add the ranges.
// Its design:
//  * the plan's grid is a lower bound on parallelism.  Each logical block's for-loop
//    is cut into `ksplit` contiguous ranges handled by different workgroups, sized so
//    that a few workgroups sit on every compute unit; a workgroup issues every load
//    of an iteration before it waits for any, so one compute unit keeps several
//    whole tiles in flight;
//  * the reference's generated programs round each iteration's product to fp16 and
//    add it to an fp16 accumulator in iteration order (src/kernel/triton_code_gen.cc:
//    223-232).  A workgroup that owns a whole for-loop does exactly that in registers.
//    When the for-loop is cut into ranges, summing each range by itself would regroup
//    the fp16 additions ((t0+t1)+(t2+t3) instead of ((t0+t1)+t2)+t3), which is a
//    different rounding sequence; so a range's workgroup stores every iteration's fp16
//    product tile to a scratch slab instead (a few percent of the weight bytes) and a
//    second, small launch adds the tiles of each block in ITERATION order, rounding to
//    fp16 after each add: the same sequence of roundings as the unsplit loop;
//  * products are formed transposed (weights as the first MFMA operand), which leaves a
//    lane with four consecutive output columns of one row: 8-byte stores;
//  * weight tiles arrive [k][n] with n contiguous while the MFMA wants k contiguous
//    per lane, so they are transposed once while being staged into LDS (4 x 16 B
//    global reads -> 8 x 8 B LDS writes per 4x8 patch), into unpadded rows with a
//    16-byte-chunk XOR swizzle; activation tiles are staged as they are, with the
//    element-wise prologue applied on the way;
//  * the LoRA inner product is produced transposed ((X.A)^T = A^T.X^T), which leaves
//    each lane holding the A-operand fragment of the following [X.A].B MFMA, so it
//    never leaves registers and the two concats cost nothing.
//
// This file is the host side (recognition, choice of kernel and launch shape, the launch or,
// for Graph::generate_hip_program, its source text); the kernels are in
// include/mi355_kernels/gemm.h, which generated programs include as well.
#include "common.h"
#include "tb_program.h"
#include <algorithm>
#include <string>

#include "gemm_tiles.h"
#include "mi355_kernels/gemm_stream.h"

namespace mi355 {

// ---------------------------------------------------------------------------------------
// host: recognise the family and launch
// ---------------------------------------------------------------------------------------
namespace {

// (a column-major tensor -- DevOp::sub == 1 on its loader -- holds element (r, c) at
// c * d_rows + r: a step along the rows is one element, a step along the columns d_rows, and
// `d_cols` of the result is that leading dimension)
// The tile origin of a loader / saver as one stride per block coordinate and per iteration.
// `fits` is cleared when an origin could leave 31 bits (the kernels multiply and add these
// strides in 32 bits): `extents` = the grid and the for-loop range.
GTile gtile(DevOp const &op, void const *ptr, int const (&extents)[4], bool &fits) {
  GTile t;
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

// The parameter blocks as C++ source (for programs that Graph::generate_hip_program writes).
std::string literal(GTile const &t) {
  return emit_fmt("mi355::GTile{%s, {%d, %d, %d, %d}, %d}", emit_pointer(t.ptr).c_str(), t.lin[0], t.lin[1],
                  t.lin[2], t.lin[3], t.d_cols);
}
std::string literal(GemmParams const &A, char const *var) {
  std::string t = emit_fmt("    mi355::GemmParams %s{};\n", var);
  char const *names[8] = {"a0", "a1", "b0", "b1", "la", "lb", "o0", "o1"};
  GTile const *tiles[8] = {&A.a0, &A.a1, &A.b0, &A.b1, &A.la, &A.lb, &A.o0, &A.o1};
  for (int i = 0; i < 8; i++) {
    t += emit_fmt("    %s.%s = ", var, names[i]) + literal(*tiles[i]) + ";\n";
  }
  t += emit_fmt("    %s.M = %d;\n    %s.KT = %d;\n    %s.forloop_range = %d;\n    %s.ksplit = %d;\n", var, A.M, var,
                A.KT, var, A.forloop_range, var, A.ksplit);
  t += emit_fmt("    %s.scratch = static_cast<_Float16 *>(%s);\n", var, emit_pointer(A.scratch).c_str());
  return t;
}
std::string literal(LaneParams const &L) {
  std::string t = literal(L.g, "G") + "    mi355::LaneParams P{};\n    P.g = G;\n";
  t += emit_fmt("    P.gx = %d;\n    P.gy = %d;\n    P.blocks = %d;\n    P.mtiles = %d;\n    P.slot_base = %d;\n", L.gx,
                L.gy, L.blocks, L.mtiles, L.slot_base);
  t += emit_fmt("    P.pieces = %d;\n    P.rank = %d;\n    P.m_group = %uu;\n    P.m_pieces = %uu;\n    P.m_columns = %uu;\n", L.pieces,
                L.rank, L.m_group, L.m_pieces, L.m_columns);
  t += emit_fmt("    P.m_gx = %uu;\n    P.m_gy = %uu;\n", L.m_gx, L.m_gy);
  return t;
}
std::string literal(StreamParams const &L) {
  return literal(L.g, "G") + "    mi355::StreamParams P{};\n    P.g = G;\n" + emit_fmt("    P.results = %d;\n    P.strips = %d;\n", L.results, L.strips);
}
char const *tf(bool b) { return b ? "true" : "false"; }

struct GMatch {
  int pro, nb;
  bool lora;
  int a0, a1, b0, b1, la, lb;  // load op indices (-1 when absent)
  int o0, o1;                  // output op indices
  int M, KT, NC, rank;         // rows, k extent and columns of the tiles; lora rank (0: no lora)
  // the sizes gemm_fused_kernel is built for (64 columns, k up to 512, up to 64 rows, rank 16);
  // anything else runs on gemm_tiles_kernel
  bool whole;
  // every weight-side operand (b0, b1, la, lb) is a DmemColumnMajor tensor, as the reference's
  // plans declare their weights (cpp_examples/lora.cc:36-41): k is contiguous in memory
  bool wcm;
};

int loader_of(DevProgram const &P, int nloads, int tensor) {
  for (int i = 0; i < nloads; i++) {
    if (P.ops[i].dst == tensor) {
      return i;
    }
  }
  return -1;
}

bool gmatch(DevProgram const &P, GMatch &G) {
  if (has_column_major_saver(P)) {
    return false;
  }
  int nl = 0;
  while (nl < P.num_ops && P.ops[nl].kind == DOP_LOAD) {
    nl++;
  }
  G.a1 = G.b1 = G.la = G.lb = G.o1 = -1;
  G.pro = PRO_NONE;
  G.nb = 1;
  G.lora = false;
  G.rank = 0;
  DevOp const *o = P.ops + nl;
  int const n = P.num_ops - nl;
  auto L = [&](int tensor) { return loader_of(P, nl, tensor); };
  if (nl == 2 && n == 2 && o[0].kind == DOP_MATMUL && o[1].kind == DOP_OUTPUT &&
      o[1].src0 == o[0].dst) {
    G.a0 = L(o[0].src0);
    G.b0 = L(o[0].src1);
    G.o0 = nl + 1;
  } else if (nl == 2 && n == 3 && o[0].kind == DOP_UNARY && o[1].kind == DOP_MATMUL &&
             o[1].src0 == o[0].dst && o[2].kind == DOP_OUTPUT && o[2].src0 == o[1].dst) {
    G.pro = o[0].sub == TB_EXP_OP ? PRO_EXP : PRO_SILU;
    G.a0 = L(o[0].src0);
    G.b0 = L(o[1].src1);
    G.o0 = nl + 2;
  } else if (nl == 3 && n == 4 && o[0].kind == DOP_MATMUL && o[1].kind == DOP_MATMUL &&
             o[0].src0 == o[1].src0 && o[2].kind == DOP_OUTPUT && o[3].kind == DOP_OUTPUT &&
             o[2].src0 == o[0].dst && o[3].src0 == o[1].dst) {
    G.nb = 2;
    G.a0 = L(o[0].src0);
    G.b0 = L(o[0].src1);
    G.b1 = L(o[1].src1);
    G.o0 = nl + 2;
    G.o1 = nl + 3;
  } else if (nl == 3 && n == 4 && o[0].kind == DOP_UNARY && o[0].sub == TB_SILU_OP &&
             o[1].kind == DOP_BINARY && o[1].sub == TB_MUL_OP && o[1].src0 == o[0].dst &&
             o[2].kind == DOP_MATMUL && o[2].src0 == o[1].dst && o[3].kind == DOP_OUTPUT &&
             o[3].src0 == o[2].dst) {
    G.pro = PRO_SILU_MUL;
    G.a0 = L(o[0].src0);
    G.a1 = L(o[1].src1);
    G.b0 = L(o[2].src1);
    G.o0 = nl + 3;
    if (G.a1 < 0 || P.t[P.ops[G.a1].dst].rows != P.t[o[0].dst].rows ||
        P.t[P.ops[G.a1].dst].cols != P.t[o[0].dst].cols) {
      return false;
    }
  } else if (nl == 4 && n == 5 && o[0].kind == DOP_MATMUL && o[1].kind == DOP_CONCAT &&
             o[2].kind == DOP_CONCAT && o[3].kind == DOP_MATMUL && o[4].kind == DOP_OUTPUT &&
             o[1].src0 == o[0].src0 && o[1].src1 == o[0].dst &&   // [X | X.A]
             o[3].src0 == o[1].dst && o[3].src1 == o[2].dst && o[4].src0 == o[3].dst &&
             P.t[o[1].dst].rows == P.t[o[0].src0].rows &&          // concat along columns
             P.t[o[2].dst].cols == P.t[o[2].src0].cols) {          // concat along rows
    G.lora = true;
    G.a0 = L(o[0].src0);
    G.la = L(o[0].src1);
    G.b0 = L(o[2].src0);
    G.lb = L(o[2].src1);
    G.o0 = nl + 4;
    if (G.la < 0 || G.lb < 0) {
      return false;
    }
    DevTensor const &ta = P.t[P.ops[G.la].dst], &tb = P.t[P.ops[G.lb].dst];
    DevOp const &lb = P.ops[G.lb];
    G.rank = ta.cols;
    if (tb.rows != G.rank || (G.rank != 8 && G.rank != 16 && G.rank != 32) || lb.row_fs != 0 || lb.col_fs != 0 ||
        lb.g_fs != 0 || !P.ops[G.la].galign || !lb.galign) {
      return false;
    }
  } else {
    return false;
  }
  if (G.a0 < 0 || G.b0 < 0 || (G.nb == 2 && G.b1 < 0)) {
    return false;
  }
  // activations row-major; the weight-side operands all in one storage order
  G.wcm = P.ops[G.b0].sub == 1;
  for (int i : {G.a0, G.a1}) {
    if (i >= 0 && P.ops[i].sub == 1) {
      return false;
    }
  }
  for (int i : {G.b0, G.b1, G.la, G.lb}) {
    if (i >= 0 && (P.ops[i].sub == 1) != G.wcm) {
      return false;
    }
  }
  DevTensor const &ta = P.t[P.ops[G.a0].dst], &tb = P.t[P.ops[G.b0].dst];
  G.M = ta.rows;
  G.KT = ta.cols;
  G.NC = tb.cols;
  if (tb.rows != G.KT || G.NC % 16 != 0 || G.KT % 32 != 0 || G.M < 1 || G.M > 256) {
    return false;
  }
  G.whole = G.NC == 64 && G.KT >= 64 && G.KT <= 512 && G.M <= (G.pro == PRO_NONE && G.nb == 1 && !G.lora ? 64 : 16) &&
            (!G.lora || G.rank == 16);
  if (G.nb == 2 && (P.t[P.ops[G.b1].dst].rows != G.KT || P.t[P.ops[G.b1].dst].cols != G.NC)) {
    return false;
  }
  if (G.lora && P.t[P.ops[G.lb].dst].cols != G.NC) {
    return false;
  }
  for (int i : {G.a0, G.a1, G.b0, G.b1, G.la, G.lb}) {
    if (i >= 0 && (!P.ops[i].galign || (reinterpret_cast<uintptr_t>(P.in[P.ops[i].io]) & 15) != 0)) {
      return false;
    }
  }
  if (G.lora && (ta.cols != P.t[P.ops[G.la].dst].rows)) {
    return false;
  }
  for (int i : {G.o0, G.o1}) {
    if (i >= 0 && (!P.ops[i].galign || (reinterpret_cast<uintptr_t>(P.out[P.ops[i].io]) & 15) != 0)) {
      return false;
    }
  }
  return true;
}

template <int MT, int NB, int PRO, bool LORA, bool WCM>
int launch_kt(GemmParams const &A, dim3 grid, int lds) {
  if (EmitSink *sink = emit_sink()) {
    sink->headers |= 2u;
    int const ktmax = A.KT <= 64 ? 64 : (A.KT <= 256 ? 256 : 512);
    emit_launch(*sink, "gemm_fused_kernel", emit_fmt("%d, %d, %d, %s, %d, %s", MT, NB, PRO, tf(LORA), ktmax, tf(WCM)), grid,
                256, lds, literal(A, "P"));
    return 1;
  }
  State &s = state();
  auto go = [&](auto *fn) -> int {
    MI355_GRANT_LDS(fn, lds);
    MI355_HIP(launch_kernel(fn, grid, 256, lds, s.stream(), A));
    return 1;
  };
  if (A.KT <= 64) {
    return go(gemm_fused_kernel<MT, NB, PRO, LORA, 64, WCM>);
  }
  if (A.KT <= 256) {
    return go(gemm_fused_kernel<MT, NB, PRO, LORA, 256, WCM>);
  }
  return go(gemm_fused_kernel<MT, NB, PRO, LORA, 512, WCM>);
}

// How gemm_stream_kernel takes a plan (see include/mi355_kernels/gemm_stream.h).
struct StreamPlan {
  int ranges = 0;       // 0: not at all
  bool strips = false;  // 16 columns a workgroup
  bool lone = false;    // of those, in one workgroup a compute unit at most
  bool pairs = false;   // both of two weights
  int mt = 0;           // 16-row groups
  int ring = 0, lds = 0, groups = 0;  // bytes of the slots, of LDS; workgroups of a block
  size_t slab = 0;      // bytes between the two launches of more than one range
};
StreamPlan stream_plan(DevProgram const &P, GMatch const &G) {
  State &s = state();
  StreamPlan plan;
  int const mt = G.M <= 16 ? 1 : (G.M <= 32 ? 2 : 4), F = P.forloop_range;
  // (with more rows than half an iteration's k the product slots rival the weights: the kernel that
  // keeps its sums in registers where a block is not split stays ahead there)
  if (s.any_size_kernels || !G.whole || G.KT % 64 != 0 || 2 * G.M > G.KT) {
    return plan;
  }
  long long const blocks = (long long)P.grid[0] * P.grid[1] * P.grid[2];
  int const ring = 4 * kStreamRing * stream_slot_bytes(G.pro, G.lora, G.M <= 8 ? 0 : mt);
  int const results = F * G.M * 128;  // of one weight
  size_t const slab = (size_t)blocks * G.nb * results;
  int const steps = (F + 3) / 4 * (G.KT / 64);  // of a wavefront that has a whole block of one weight
  bool const fits = ring + results <= s.max_lds;
  // Strips of 16 columns where they fill most of the chip and two workgroups fit on a compute unit (4 rows, us, strips
  // / ranges: 3840 columns x 4096, 240 workgroups, 7.6 / 10.7; 28672 39.9 / 51.6; two weights of 3072 x 8192
  // with a gated MLP's second product 37.9 / 40.1), but not where one weight's whole blocks fill it as well (below:
  // 4 rows x 12416 x 1536 9.7 / 8.0, 16 x 14656 x 1792 13.6 / 11.4, but 16 x 7360 x 1280, 115 blocks, 6.1 / 6.8).
  int const eights = G.M <= 8 ? 1 : 2, strip_ring = 4 * columns_ring(eights, G.lora) * columns_slot_bytes(eights, G.lora);
  int const strip_lds = strip_ring + F * G.M * 32;
  bool const narrow = G.wcm && G.pro == PRO_NONE && G.M <= 16;
  bool strips = narrow && !G.lora && 4 * G.nb * blocks >= 192 && 2 * strip_lds <= s.max_lds && !(G.nb == 1 && fits && blocks >= 192 && steps <= 8);
  // In 256-k iterations a 16-column strip asks for enough at a time that one workgroup a compute unit keeps up with
  // memory, and one launch without a slab is ahead of both other kernels (us, the others / strips: LoRA 4096 columns x
  // 4096 of 8 rows 10.9 / 8.0, x 1024 4.1 / 3.6, 3072 x 4096 8.2 / 7.2; one product of 16 rows 4096 x 8192 14.3 / 11.9,
  // x 14336 26.6 / 24.9, 3072 x 4096 7.0 / 6.3), but not with fewer workgroups (LoRA of 2048 x 2048 4.75 / 4.9, one
  // product of 16 x 2560 x 1536 3.9 / 4.2), where the wavefronts wait for one of them (5 iterations, 16 rows x 3072
  // 3.4 / 3.9), in 64-k iterations, of which the ring holds a quarter (LoRA 4096 x 1024 of 8 rows 3.7 / 4.1), or where
  // half the rows halve the others' slab, short of long loops (8 rows x 4096: 4096 7.5 / 7.8, 44 - 52 iterations 0.97 -
  // 1.08 of the others' time, 53 of 58 and more blocks 1.02 - 1.05 (fewer 1.0), 54 - 63 0.92 - 1.03, 64 - 112 0.88 - 1.02).
  // Iterations of 128 and of 512 k were not timed in these strips: they keep the kernels they had.  Nor does a printed program
  // change: the text of a LoRA's is what programs built around it know (two launches and a workspace that it allocates;
  // tests/test_generated_hip.py pins it), the same bits, 11.2 us for 16 rows x 4096 x 4096 where the strips take 7.9.
  plan.lone = narrow && G.nb == 1 && G.KT == 256 && F >= 3 * ((F + 3) / 4) && 4 * blocks <= 256 && strip_lds <= s.max_lds &&
              (G.lora ? blocks >= 40 && !emit_sink() : blocks >= 48 && (G.M > 8 || F > 52));
  strips = strips || plan.lone;
  // One range per block where the blocks alone occupy the chip and a wavefront has a few steps to
  // make: no slab and no second launch (4 x 8192 x 2048 in 64-k iterations: 8.9 us against 12).
  // Otherwise four iterations, one per wavefront, to a range, as far as that many workgroups are
  // resident at a time: a slot of 10 KB leaves room for two on a compute unit, which then also gain
  // from taking turns; a larger one for one, where a second round would start late (32 x 3840 x 5120:
  // 13.8 us in 240 workgroups, 16.0 in 300).
  bool one = fits && blocks * G.nb >= 96 && steps <= 8;
  // Blocks for more than half of the chip are not cut at all where the slab would be large beside the weights: with
  // SiLU(a) * u (8 rows, us, one range / ranges: 14336 x 3712 in 64-k iterations 20.8 / 29.8, 8768 x 2944 14.5 / 16.8,
  // but 114 blocks, 7296 x 4608, 20.4 either way, and 10240 x 4096 in 256-k ones, 16 steps, 24.2 / 21.7) ...
  if (G.pro == PRO_SILU_MUL && G.M <= 8) {
    one = one || (fits && blocks > 128 && blocks <= 256 && (steps <= 12 || blocks >= 192));
  }
  // ... and with two weights (8 rows, row-major: 4160 x 4096 in 256-k iterations 16.1 / 19.2, 6784 x 6144 30.1 / 35.0,
  // 6400 x 4096 in 64-k ones 23.7 / 31.2, but 16 rows of these 41.5 / 36.8, and 4096 x 8192 39.1 / 34.1).
  if (G.nb == 2 && 2 * blocks >= 128 && 2 * blocks <= 256) {
    one = one || (fits && (steps <= 16 || (blocks >= 100 && steps <= 24)) && (G.M <= 8 || G.KT >= 128));
  }
  // Past that a compute unit has room for one workgroup of one weight: one of both then leaves less of the last
  // round empty and reads the activations once (8 rows, row-major, us, both / one weight a workgroup: 10944 x 704 8.1 / 10.6,
  // 8448 x 768 8.0 / 11.0, 14336 x 832 12.2 / 14.9, 14336 x 4096 49.5 / 53.8, 16 rows x 9216 x 2048 23.9 / 27.6; where two
  // of one weight fit, 16384 x 512 9.1 / 8.2).
  bool pairs = !strips && G.nb == 2 && blocks > 128 && blocks <= 256 && 2 * (ring + results) > s.max_lds && ring + 2 * results <= s.max_lds;
  one = one || pairs;
  // Row-major, also where their ranges are a workgroup for every compute unit: the two weights are read in turn, not
  // side by side at the same offsets of a power-of-two stride (8 rows, us, both / one weight: 2048 x 8192 in 256-k iterations
  // 20.5 / 23.9, in 64-k ones 27.0 / 28.5, 4096 x 4096 in 256-k ones 19.1 / 21.4, but in 64-k ones 24.7 / 22.7).
  int const filling = (int)(256 / blocks);
  bool const even = G.nb == 2 && !G.wcm && blocks >= 32 && blocks <= 64 && filling * blocks == 256 && (blocks < 64 || G.KT == 256) &&
                    (F + 3) / 4 >= filling;
  bool const slab_fits = slab <= (emit_sink() ? kEmitScratchBytes : s.scratch_bytes);
  int ks = 1;
  if (even && slab_fits) {
    pairs = true;
    ks = filling;
  } else if (!one && slab_fits) {
    // (two weights have workgroups of their own: a wavefront of one takes two iterations of 64 k, so that one's loads
    // run under the other's products; 8 rows x 4096 x 3904 20.4 -> 18.8 us, 2944 x 6464 22.1 -> 20.2)
    // (eight rows of SiLU(a) * u leave room for two workgroups of long row-major iterations on a compute unit, but one
    // has more of them in flight: 4096 x 6400 in 256-k iterations, 256 workgroups 17.2 us, 448 18.9, 2560 x 8192 15.4 and
    // 17.4; column-major 4096 x 14336 29.4 and 28.6)
    bool const single = ring > 80 * 1024 || (G.pro == PRO_SILU_MUL && G.KT == 256 && !G.wcm);
    long long const most = (single ? 256 / G.nb : 1024) / blocks;
    int const least = G.nb == 2 && G.KT == 64 ? 8 : 4;
    ks = (int)std::max<long long>(1, std::min<long long>((F + least - 1) / least, most));
    // (one round of long iterations rather than a part of a second: 8 rows x 2560 x 4096 in 256-k iterations 15.8 us in
    // 320 workgroups, 13.3 in 240)
    long long const wanted = blocks * G.nb * ks;
    if (G.nb == 2 && G.KT == 256 && wanted > 256 && wanted < 512) {
      ks = (int)std::max<long long>(1, 256 / (blocks * G.nb));
    }
  }
  if (ks == 1 && !fits && !strips) {
    return plan;
  }
  int const per = (F + ks - 1) / ks;
  plan.strips = strips;
  plan.pairs = pairs;
  plan.mt = mt;
  plan.ranges = strips ? 1 : (F + per - 1) / per;  // (no empty range)
  plan.ring = strips ? strip_ring : ring;
  plan.lds = strips ? strip_lds : ring + (plan.ranges == 1 ? results * (pairs ? 2 : 1) : 0);
  plan.groups = (pairs ? 1 : G.nb) * (strips ? 4 : plan.ranges);
  plan.slab = plan.ranges > 1 ? slab : 0;
  return plan;
}

// gemm_lanes_kernel for this plan, or 0 when it is not the better choice (see the rule in
// try_launch_lanes); k extents 32 / 64 / 96 / 128 / 256.
template <int NB, int PRO, int LORA, bool WCM>
int launch_lanes_kt(LaneParams const &L, int grid, int threads, int lds) {
  if (EmitSink *sink = emit_sink()) {
    sink->headers |= 2u;
    emit_launch(*sink, "gemm_lanes_kernel", emit_fmt("%d, %d, %d, %s, %s", L.g.KT, NB, PRO, LORA == 2 ? "2" : tf(LORA == 1), tf(WCM)),
                dim3(grid, 1, 1), threads, lds, literal(L));
    return 1;
  }
  State &s = state();
  auto go = [&](auto *fn) -> int {
    MI355_GRANT_LDS(fn, lds);
    MI355_HIP(launch_kernel(fn, grid, threads, lds, s.stream(), L));
    return 1;
  };
  switch (L.g.KT) {
    case 32:
      return go(gemm_lanes_kernel<32, NB, PRO, LORA, WCM>);
    case 64:
      return go(gemm_lanes_kernel<64, NB, PRO, LORA, WCM>);
    case 96:
      return go(gemm_lanes_kernel<96, NB, PRO, LORA, WCM>);
    case 128:
      return go(gemm_lanes_kernel<128, NB, PRO, LORA, WCM>);
    case 256:
      return go(gemm_lanes_kernel<256, NB, PRO, LORA, WCM>);
    default:
      return 0;
  }
}

// What the chain of a wavefront's iterations takes in the one-launch kernel, and what the streaming one takes, in ns:
// fitted to the column-major ones of 2160 plans of 2 - 256 blocks, k 256 - 24000 and every prologue, on weights that change
// from pass to pass (rms 14 and 12 %; the chain stands 18 % above its fit, where the choice lost least).  A piece's
// wavefronts walk the whole of k, so its time grows with k however few pieces there are, and past a few hundred iterations
// their results leave LDS for one or two wavefronts (us, here / there: silu of 16 rows x 256 x 19264 in 64-k iterations
// 139 / 24, of 8 x 320 x 20736 in 256-k ones 34.5 / 11.2, 4 rows x 256 x 18176 14.0 / 10.0, two weights of 4 x 1984 x 9536
// 113 / 28, a LoRA of 4 x 448 x 15232 40 / 13; row-major two weights of 4 x 192 x 8832 42 / 13, silu of 8 x 320 x 7424
// 19.0 / 9.1).  Row-major chains are longer still, so there the estimate only finds the clear cases.
double lanes_chain_ns(GMatch const &G, long long units, int F, int ip, int lds, long long pieces) {
  State &s = state();
  // ns for 64 k, and for sixteen wavefronts on the compute unit instead of none
  double const alone = G.nb == 2 ? 230 : G.lora ? 270 : G.pro == PRO_EXP ? 300 : G.pro == PRO_SILU ? 620 : G.pro == PRO_SILU_MUL ? 720 : 250;
  double const more = G.nb == 2 ? 920 : G.lora ? 1030 : G.pro == PRO_EXP ? 740 : G.pro == PRO_SILU ? 1210 : G.pro == PRO_SILU_MUL ? 1390 : 560;
  long long const resident = std::max<long long>(1, std::min<long long>(s.max_lds / lds, 16 / ip)), each = (pieces + 255) / 256;
  int const turns = (F + ip - 1) / ip;
  double waves = (double)ip * std::min(resident, each);
  if (turns > 1) {  // (few wavefronts wait for memory instead of each other)
    waves = std::max(waves, G.wcm && G.pro == PRO_NONE && G.nb == 1 && !G.lora ? 10.0 : 8.0);
  }
  double const chain = (double)turns * (double)units / F;
  return 2000 + (double)((each + resident - 1) / resident) * (chain * (alone + more * waves / 16) + 550);
}
double stream_ns(DevProgram const &P, GMatch const &G, StreamPlan const &plan, long long weight_bytes) {
  State &s = state();
  int const F = P.forloop_range;
  long long const groups = (long long)P.grid[0] * P.grid[1] * P.grid[2] * plan.groups, resident = std::max(1, s.max_lds / plan.lds);
  int const per = (F + plan.ranges - 1) / plan.ranges;
  double const steps = (double)((per + 3) / 4) * (G.KT / 64) * (plan.pairs ? 2 : 1) / (plan.strips ? 4 : 1);
  double const step = 270 + (G.pro == PRO_SILU || G.pro == PRO_SILU_MUL ? (G.M > 8 ? 270 : 120) : 0);
  double ns = 3700 + (double)weight_bytes / (plan.strips ? 6150 : 8400) + (double)((groups + 256 * resident - 1) / (256 * resident)) * steps * step;
  if (plan.ranges > 1) {
    ns += 3000 + (double)plan.slab * 0.45e-3 + F * (21 + 12 * G.M / 16.0);
  }
  return ns;
}

// `gate`: see GateRequest; *gated tells whether a launch was made that takes care of it.  `R`: the program as the choice sees it, G but
// for a row-major second operator of such a pair, which runs where it would run by itself: without its prologue no
// kernel is slower than with it (2 rows x 576 x 6528 14.8 us before and so, 16.8 in the kernel of a plain product).
int try_launch_lanes(DevProgram const &P, GMatch const &G, GMatch const &R, GemmParams const &A, _Float16 *gate, bool *gated) {
  State &s = state();
  // lora A comes in 16-rank pieces, the last one half full where its columns are rows in memory; two weights in
  // tiles of 64 columns and whole 64-k units only (programs printed for others are known to hold the tiles' kernel)
  bool const takes = (G.nb == 1 || (G.NC == 64 && G.KT % 64 == 0)) && (G.KT == 32 || G.KT == 64 || G.KT == 96 || G.KT == 128 || G.KT == 256) && G.M <= 64 &&
                     (!G.lora || G.rank % 16 == 0 || (G.wcm && G.rank == 8));
  if (s.gemm_mode == 1 || s.any_size_kernels || !takes) {
    return 0;
  }
  long long const blocks = (long long)P.grid[0] * P.grid[1] * P.grid[2];
  int const mtiles = (G.M + 15) / 16, pieces = G.NC / 16, S = pieces * mtiles, F = P.forloop_range;
  int const lora = G.lora ? (G.rank + 15) / 16 : 0;
  long long const groups = (blocks + 7) / 8;
  // (the kernel decodes the flat id with multiply-high magics: exact while id x divisor < 2^32)
  long long const widest = std::max<long long>(8 * S, std::max(P.grid[0], P.grid[1]));
  if (groups * 8 * S * widest >= (1LL << 32)) {
    return 0;
  }
  bool const three = G.lora || G.pro == PRO_SILU_MUL;
  int const wave_bytes = lanes_wave_bytes(G.KT, G.nb, lora, G.wcm, G.pro);
  int const slot_bytes = F * G.nb * 512;
  // Workgroups of 16 wavefronts while about one round of them covers the grid; half that where two share a compute
  // unit and one's loads can run under the other's products (64 rows x 6400 x 4096 in 256-k iterations: 25.5 -> 19.7
  // us; 16 rows x 1280, 80 workgroups: 5.2 against 5.7 the other way).  Two weights leave LDS for one workgroup of 13
  // and more: half as many there too, evened out over the rounds (8 rows, column-major: 832 x 14336 14.0 -> 10.6 us,
  // 1024 x 12224 12.1 -> 10.0, 4096 x 3904 in one round 12.3 either way; row-major 832 x 6464 8.8 -> 7.4).  The
  // registers of 16 wavefronts with SiLU(a) * u or a LoRA tile fill the unit either way (13.1 us there, 15.0 here).
  int const waves = G.nb == 2 || (!three && (long long)blocks * S * G.KT > 98304) ? 8 : 16;
  int const most = std::min(waves, lanes_most(G.KT, lora));
  int ip = F < most ? F : most;
  if (G.nb == 2) {
    int const rounds = (F + ip - 1) / ip;
    ip = (F + rounds - 1) / rounds;
  }
  while (ip > 1 && ip * wave_bytes + slot_bytes > s.max_lds) {
    ip = (ip + 1) / 2;
  }
  int const lds = ip * wave_bytes + slot_bytes;
  if (lds > s.max_lds) {
    return 0;
  }
  // One launch, whose pieces of 16 columns each read the activation rows, against whole lines moved once by the
  // range-splitting kernel and a second launch that adds its ranges.
  // Row-major weights: a 16-column strip uses 32 bytes of every line it pulls into a compute unit's vector cache,
  // so only where the launch sets the time (16 rows, in us, here / there: 3840 columns in 128-k iterations, 16 MB,
  // 6.7 / 8.3; 6400, 26 MB, 9.8 / 9.1; 64-column blocks of 256 k fill LDS with fewer wavefronts: 1280 columns,
  // 10 MB, 9.6 / 7.6; few pieces leave the chip idle: two weights of 1088 columns, 14 MB, 68 pieces, 0.5 us behind).
  // Column-major weights: a piece's columns are whole lines of its own, and the line lies far out, where the
  // activation rows that the pieces read outnumber what the second launch costs.  One weight (64 rows x 12800 x 4096
  // 45 / 62, 8 x 28672 x 4096, 235 MB of weights, 39.6 / 53, but 64 x 28672 x 1024, 7168 pieces, 22.2 / 19.6);
  // a LoRA tile or a second activation makes it three operand rows a column (lora 16 x 4096 x 2048 6.5 / 9.4, 21 MB;
  // 16 x 4096 x 4096, 42 MB, 10.1 / 11.1, is still below the crossing, 16 x 8192 x 4096 17.3 / 17.1, but the program
  // printed for it is known to hold the streaming kernel and its workspace, and stays so); two weights in 64-k or
  // 128-k iterations at any size (8 rows: 832 x 14336 10.6 / 13.1, 4096 x 6464 25.4 / 29.9, 4096 x 14336, 235 MB,
  // 49.2 / 53.6), in 256-k ones 4096 x 8192, 134 MB, 28.2 / 25.4.
  // Two row-major weights with almost a workgroup for every compute unit stand between (4096 x 3904 14.0 / 18.8,
  // 1536 x 3904 7.0 / 8.0, but 256 workgroups 10.8 / 9.8, 404 13.6 / 10.8, and 128-k iterations 8.9 / 7.1;
  // with both products of a gated MLP 160 workgroups, 4096 x 2560, 28.4 / 25.0, 176 24.0 / 24.9, 200 25.9 either way).
  long long const weight_bytes = blocks * F * (long long)(G.nb * G.KT * G.NC + (G.lora ? G.KT * G.rank : 0)) * 2;
  long long most_mb = 256;
  if (!G.wcm) {
    most_mb = G.KT == 256 || blocks * S < 128 ? 8 : (G.nb == 2 && G.KT == 64 && blocks * S >= 192 && blocks * S < 256 ? 68 : 17);
  } else if (G.lora || three) {
    most_mb = G.lora ? 32 : 48;
  } else if (G.nb == 2 && G.KT == 256) {
    most_mb = 68;
  }
  // SiLU(a) * u is done again by each of a block's pieces, one piece's iterations take the same time however few
  // pieces there are, and past 104 units of 64 k the result slots leave LDS for half the wavefronts.  The other
  // kernel's time grows with the weights and with the slab between its launches.  Both in ns (8 and 16 rows, us,
  // here / there: 64 k an iteration, column-major 4096 outputs of 3904 11.0 / 14.6, 2048 of 3904 10.2 / 11.3, 832 of
  // 6464 14.9 / 12.2, 640 of 12224 31.5 / 12.2; 128 k 3776 of 4992 12.5 / 14.0, 2048 of 8192 17.1 / 13.0.  Row-major
  // weights that come from memory and not from the last-level cache cost the strips more, so those lines are of both
  // products of a gated MLP in turn: 4096 of 3904 35.2 / 34.3, 3584 of 5440 48.7 / 45.6, 4096 of 2560 28.4 / 30.2.
  // Of 28 such pairs of either order the choice is the faster one or within 1.1 us, but for row-major 2944 of 4032,
  // 23.8 / 24.9 and, 16 rows, 23.8 / 26.4).
  long long const units = (long long)F * G.KT / 64;
  // (In 256-k iterations a piece's loads are waited for together: 8 x 4096 x 4096 column-major 12.0 / 11.4.  One range
  // of the other kernel has neither the slab nor its launch: 8 rows x 10112 x 768 9.3 / 5.8, 14336 x 832 12.7 / 6.2.)
  StreamPlan const plan = G.whole && G.KT % 64 == 0 ? stream_plan(P, R) : StreamPlan{};
  long long const here_ns = (1000 + (!G.wcm ? 225 : G.KT == 256 ? 185 : 142) * units) * ((blocks * S + 255) / 256);
  long long const there_ns = plan.ranges == 1 ? 4000 + blocks * units : 7000 + blocks * units + blocks * F * 7 / 10 + 15 * F;
  // Other tiles run on the any-size kernel or, in 96-k iterations of 64 columns, on the one with a barrier a step:
  // both are behind but for larger row-major plans (us, here / there: 64 rows x 3008 x 5120 in blocks of 32 columns
  // 13.6 / 30.7, a LoRA of rank 32 of 16 x 2304 x 3584 10.1 / 17.2, 64 x 1280 x 768 in 96-k iterations 4.0 / 8.9;
  // row-major 16 x 6144 x 2048 in blocks of 48 12.2 / 19.6, 64 x 12800 x 2048 in 128-k iterations 39.7 / 50.8, but
  // 64 x 3840 x 2048 in 256-k ones 19.4 / 15.7, 64 x 3840 x 1920 in 96-k ones 18.6 / 15.3 and, of 64 columns,
  // 16 x 6400 x 3072 15.1 / 14.4).
  bool there;
  if (G.whole && G.KT % 64 == 0) {
    there = plan.lone || blocks * S > (G.wcm ? 4096 : 1024) || weight_bytes > (most_mb << 20);
    if (R.pro == PRO_SILU_MUL && G.M <= 16) {
      there = units > 104 || here_ns > there_ns;
    }
    if (plan.ranges > 0 && (R.pro != PRO_SILU_MUL || (G.wcm && plan.ranges == 1 && blocks * S > 256))) {
      there = there || lanes_chain_ns(R, units, F, ip, lds, blocks * S) > stream_ns(P, R, plan, weight_bytes);
    }
    // Row-major, the other kernel's whole blocks on more than half of the chip, and a prologue that is not done again
    // for every 16 columns (us, here / there: silu of 4 rows x 12416 x 640 7.6 / 6.5, lora 8576 x 768 7.5 / 6.4,
    // two weights of 8 x 13824 x 256 6.7 / 5.8).
    if (!G.wcm && plan.ranges == 1 && blocks >= 128 && (R.pro != PRO_NONE || G.lora || G.nb == 2)) {
      there = true;
    }
  } else if (G.wcm) {
    there = false;
  } else if (G.whole) {
    there = weight_bytes > (17LL << 20);
  } else {
    there = G.M > 32 && (G.KT == 96 || G.KT == 256) && weight_bytes > (8LL << 20);
  }
  if (s.gemm_mode == 0 && there) {
    return 0;
  }
  LaneParams L{};
  L.g = A;
  L.gx = P.grid[0];
  L.gy = P.grid[1];
  L.blocks = (int)blocks;
  L.mtiles = mtiles;
  L.pieces = pieces;
  L.rank = G.rank;
  L.slot_base = ip * wave_bytes;
  L.g.gate = gate;
  L.m_group = fast_div_magic(8 * S);
  L.m_pieces = fast_div_magic(S);
  L.m_columns = fast_div_magic(pieces);
  L.m_gx = fast_div_magic(P.grid[0]);
  L.m_gy = fast_div_magic(P.grid[1]);
  int const grid = (int)(groups * 8 * S);
  int rc = 0;
#define MI355_LANES_CASE(NBV, PROV, LORAV)                                  \
  if (G.nb == NBV && G.pro == PROV && lora == LORAV) {                      \
    rc = G.wcm ? launch_lanes_kt<NBV, PROV, LORAV, true>(L, grid, ip * 64, lds)   \
               : launch_lanes_kt<NBV, PROV, LORAV, false>(L, grid, ip * 64, lds); \
  }
  MI355_LANES_CASE(1, PRO_NONE, 0)
  MI355_LANES_CASE(1, PRO_EXP, 0)
  MI355_LANES_CASE(1, PRO_SILU, 0)
  MI355_LANES_CASE(2, PRO_NONE, 0)
  MI355_LANES_CASE(1, PRO_SILU_MUL, 0)
  MI355_LANES_CASE(1, PRO_NONE, 1)
  MI355_LANES_CASE(1, PRO_NONE, 2)
#undef MI355_LANES_CASE
  if (rc == 1) {
    *gated = gate != nullptr;
    s.last().kernel_id = MI355_KERNEL_F16_GEMM;
    s.last().workgroups = grid;
    s.last().threads = ip * 64;
    s.last().lds_bytes = lds;
    s.last().row_split = S;
  }
  return rc;
}

// the fold of a split for-loop: the launch, or its source text
int launch_combine(GemmParams const &A, int nb, dim3 blocks) {
  State &s = state();
  int const lds = A.forloop_range * 1024;
  int const sets = A.gate != nullptr ? 2 : 1;  // weights of a workgroup
  dim3 const fold_grid(blocks.x * (nb / sets) * ((A.M + 7) / 8), blocks.y, blocks.z);
  if (EmitSink *sink = emit_sink()) {
    bool const fold = lds <= s.max_lds;
    emit_launch(*sink, fold ? "gemm_fold_kernel" : "gemm_combine_kernel", emit_fmt("%d", nb), fold ? fold_grid : blocks, 256,
                fold ? lds : 0, literal(A, "P"));
    return 1;
  }
  if (lds > s.max_lds) {
    MI355_HIP(launch_kernel(nb == 1 ? gemm_combine_kernel<1> : gemm_combine_kernel<2>, blocks, 256, 0, s.stream(), A));
    return 1;
  }
  auto *fn = nb == 1 ? gemm_fold_kernel<1> : gemm_fold_kernel<2>;
  MI355_GRANT_LDS(fn, lds * sets);
  MI355_HIP(launch_kernel(fn, fold_grid, 256 * sets, lds * sets, s.stream(), A));
  return 1;
}

template <int NB, int PRO, bool LORA, bool WCM, int MT>
int launch_stream_one(StreamParams const &L, dim3 grid, int lds) {
  if (EmitSink *sink = emit_sink()) {
    sink->headers |= 32u;
    emit_launch(*sink, "gemm_stream_kernel", emit_fmt("%d, %d, %s, %s, %d", NB, PRO, tf(LORA), tf(WCM), MT), grid, 256, lds, literal(L));
    return 1;
  }
  auto *fn = gemm_stream_kernel<NB, PRO, LORA, WCM, MT>;
  MI355_GRANT_LDS(fn, lds);
  MI355_HIP(launch_kernel(fn, grid, 256, lds, state().stream(), L));
  return 1;
}

template <bool WCM, int GROUPS>
int launch_stream_pairs(StreamParams const &L, dim3 grid, int lds) {
  if (EmitSink *sink = emit_sink()) {
    sink->headers |= 32u;
    emit_launch(*sink, "gemm_stream_pairs_kernel", emit_fmt("%s, %d", tf(WCM), GROUPS), grid, 256, lds, literal(L));
    return 1;
  }
  auto *fn = gemm_stream_pairs_kernel<WCM, GROUPS>;
  MI355_GRANT_LDS(fn, lds);
  MI355_HIP(launch_kernel(fn, grid, 256, lds, state().stream(), L));
  return 1;
}

// gemm_stream_kernel for this plan, or 0.
int try_launch_stream(DevProgram const &P, GMatch const &G, GemmParams const &A, _Float16 *gate, bool *gated) {
  State &s = state();
  StreamPlan const plan = stream_plan(P, G);
  if (plan.ranges == 0 || (long long)P.grid[0] * plan.groups > 2147483647LL) {
    return 0;
  }
  int const ks = plan.ranges, lds = plan.lds, mt = plan.mt;
  EmitSink *const sink = emit_sink();
  StreamParams L{};
  L.g = A;
  L.g.ksplit = ks;
  L.g.scratch = ks > 1 ? static_cast<_Float16 *>(s.scratch()) : nullptr;
  if (sink && ks > 1) {  // a printed program allocates the workspace itself
    L.g.scratch = reinterpret_cast<_Float16 *>(kEmitScratch);
  }
  L.results = plan.ring;
  L.strips = plan.strips;
  // (whole blocks of one weight meet in no workgroup, and no more do sums past the fold's LDS)
  bool const takes_gate = gate != nullptr && (plan.strips || (ks == 1 ? plan.pairs : P.forloop_range * 2048 <= s.max_lds));
  L.g.gate = takes_gate ? gate : nullptr;
  dim3 const grid(P.grid[0] * plan.groups, P.grid[1], P.grid[2]);
  int rc = 0;
  if (plan.pairs) {
    rc = G.M <= 8 ? (G.wcm ? launch_stream_pairs<true, 0>(L, grid, lds) : launch_stream_pairs<false, 0>(L, grid, lds))
                  : (G.wcm ? launch_stream_pairs<true, 1>(L, grid, lds) : launch_stream_pairs<false, 1>(L, grid, lds));
  }
#define MI355_STREAM_CASE(NBV, PROV, LORAV, MTV)                                            \
  if (!plan.pairs && G.nb == NBV && G.pro == PROV && G.lora == LORAV && mt == MTV) {        \
    rc = G.wcm ? launch_stream_one<NBV, PROV, LORAV, true, MTV>(L, grid, lds)               \
               : launch_stream_one<NBV, PROV, LORAV, false, MTV>(L, grid, lds);             \
  }
  MI355_STREAM_CASE(1, PRO_NONE, false, 1)
  MI355_STREAM_CASE(1, PRO_NONE, false, 2)
  MI355_STREAM_CASE(1, PRO_NONE, false, 4)
  MI355_STREAM_CASE(1, PRO_EXP, false, 1)
  MI355_STREAM_CASE(1, PRO_SILU, false, 1)
  MI355_STREAM_CASE(2, PRO_NONE, false, 1)
  MI355_STREAM_CASE(1, PRO_SILU_MUL, false, 1)
  MI355_STREAM_CASE(1, PRO_NONE, true, 1)
#undef MI355_STREAM_CASE
  if (rc == 1 && ks > 1) {
    if (sink) {
      sink->scratch_bytes = std::max(sink->scratch_bytes, plan.slab);
    }
    rc = launch_combine(L.g, G.nb, dim3(P.grid[0], P.grid[1], P.grid[2]));
  }
  if (rc == 1) {
    *gated = takes_gate;
    s.last().kernel_id = MI355_KERNEL_F16_GEMM;
    s.last().workgroups = grid.x * grid.y * grid.z;
    s.last().threads = 256;
    s.last().lds_bytes = lds;
    s.last().row_split = ks;
  }
  return rc;
}

}  // namespace

std::string gemm_params_literal(GemmParams const &A, char const *var) { return literal(A, var); }

bool gemm_applicable(DevProgram const &P) {
  GMatch G;
  return gmatch(P, G);
}

// A gated MLP's operators: the first makes G and U, the second multiplies silu(G) * U.  Every block of columns of the
// second, and in the one-launch kernel every 16 of them, makes that product of 16 x k values again, a chain of an
// exponential, a reciprocal and a dozen instructions for each; where the first's kernel has both sums in a workgroup
// it makes it once, into the queue's memory for operand copies, and the second is a plain product.  (G and U are
// written as before.)  8 x 4096 x 14336, column-major: both 71.9 -> 68.0 us; 100 drawn gated MLPs 0.87 of the time in the
// mean, 0.70 - 1.01.  A launch of its own for the product takes back what it gives (us, separate operators / with it, row-major:
// 16 rows x 2496 x 5952 39.4 / 40.1, 8 x 1088 x 4288 17.6 / 19.1).
// For-loops past what the fold keeps in LDS stay: the second's plain product then takes the one-launch kernel, where
// result slots leave half the wavefronts (8 rows x 1408 x 14272 in 64-k iterations 19.6 us in ranges, 25.9 there).
bool gate_pair(DevProgram const &first, DevProgram const &second, GateRequest &R) {
  GMatch A, B;
  if (!gmatch(first, A) || !gmatch(second, B) || A.nb != 2 || B.pro != PRO_SILU_MUL || A.M != B.M ||
      second.forloop_range * 1024 > state().max_lds) {
    return false;
  }
  DevOp const &o0 = first.ops[A.o0], &o1 = first.ops[A.o1], &g = second.ops[B.a0], &u = second.ops[B.a1];
  if (first.out[o0.io] != second.in[g.io] || first.out[o1.io] != second.in[u.io]) {
    return false;
  }
  // the first makes all of [M][columns] side by side, the second reads all of it iteration by iteration
  int const columns = o0.d_cols;
  int pieces = 1;
  for (int i = 0; i < 3; i++) {
    if (first.grid[i] > 1) {
      if (o0.row_bs[i] != 0 || o0.g_bs[i] != 0 || o0.col_bs[i] != A.NC || o1.row_bs[i] != 0 || o1.g_bs[i] != 0 || o1.col_bs[i] != A.NC) {
        return false;
      }
      pieces *= first.grid[i];
    }
    if (second.grid[i] > 1 && (g.row_bs[i] || g.col_bs[i] || g.g_bs[i] || u.row_bs[i] || u.col_bs[i] || u.g_bs[i])) {
      return false;
    }
  }
  int dims = (first.grid[0] > 1) + (first.grid[1] > 1) + (first.grid[2] > 1);
  bool const walks = second.forloop_range == 1 || (g.col_fs == B.KT && g.row_fs == 0 && g.g_fs == 0 && u.col_fs == B.KT && u.row_fs == 0 && u.g_fs == 0);
  if (dims > 1 || pieces * A.NC != columns || o1.d_cols != columns || g.d_cols != columns || u.d_cols != columns || !walks ||
      second.forloop_range * B.KT != columns) {
    return false;
  }
  R.elements = (size_t)A.M * columns;
  return true;
}

int try_launch_gemm(DevProgram const &P, GateRequest *request, bool second) {
  GMatch G;
  if (!gmatch(P, G)) {
    return 0;
  }
  State &s = state();
  _Float16 *const made = request != nullptr ? static_cast<_Float16 *>(request->h) : nullptr, *const gate = second ? nullptr : made;
  bool gated = false;
  GMatch by_itself = G;
  if (second) {
    G.pro = PRO_NONE;
    G.a1 = -1;
    if (G.wcm) {  // (column-major strips in one launch are what its prologue kept it from: 16 rows x 1408 x 6400 23.1 -> 16.8 us)
      by_itself = G;
    }
  }
  GemmParams A{};
  int const extents[4] = {P.grid[0], P.grid[1], P.grid[2], P.forloop_range};
  bool fits = true;
  auto in_tile = [&](int i) { return gtile(P.ops[i], P.in[P.ops[i].io], extents, fits); };
  A.a0 = in_tile(G.a0);
  if (second) {
    A.a0.ptr = made;
  }
  A.a1 = G.a1 >= 0 ? in_tile(G.a1) : A.a0;
  A.b0 = in_tile(G.b0);
  A.b1 = G.b1 >= 0 ? in_tile(G.b1) : A.b0;
  A.la = G.la >= 0 ? in_tile(G.la) : A.a0;
  A.lb = G.lb >= 0 ? in_tile(G.lb) : A.a0;
  A.o0 = gtile(P.ops[G.o0], P.out[P.ops[G.o0].io], extents, fits);
  A.o1 = G.o1 >= 0 ? gtile(P.ops[G.o1], P.out[P.ops[G.o1].io], extents, fits) : A.o0;
  if (!fits) {
    return 0;  // a tensor of more than 2^31 elements: the generic interpreter takes the plan
  }
  A.M = G.M;
  A.KT = G.KT;
  A.forloop_range = P.forloop_range;
  auto with_gate = [&](int rc) -> int { return rc == 1 && gate != nullptr && !gated ? 0 : rc; };
  if (int const rc = try_launch_lanes(P, G, by_itself, A, gate, &gated)) {
    return with_gate(rc);
  }
  if (int const rc = try_launch_stream(P, G, A, gate, &gated)) {
    return with_gate(rc);
  }
  if (!G.whole || s.any_size_kernels) {
    return with_gate(launch_gemm_tiles(A, TileGemmPlan{{P.grid[0], P.grid[1], P.grid[2]}, G.pro, G.nb, G.rank, G.NC, G.wcm}));
  }
  int const mt = G.M <= 16 ? 1 : (G.M <= 32 ? 2 : 4);
  long long const blocks = (long long)P.grid[0] * P.grid[1] * P.grid[2];
  // Ranges per block: the split that minimises (rounds of resident workgroups) x
  // (iterations per workgroup + a fixed cost per workgroup + the combine's cost per range),
  // with two workgroups resident per compute unit.  Never more ranges than iterations.
  int ksplit = 1;
  {
    double best = 1e30;
    for (int cand = 1; cand <= P.forloop_range; cand++) {
      int const per = (P.forloop_range + cand - 1) / cand;
      if ((P.forloop_range + per - 1) / per != cand) {
        continue;  // would leave empty ranges
      }
      long long const rounds = (blocks * cand + 511) / 512;
      double const cost = (double)rounds * (per + 1.5 + 0.15 * cand);
      if (cost < best - 1e-9) {
        best = cost;
        ksplit = cand;
      }
    }
  }
  long long const scratch_elems = blocks * P.forloop_range * G.nb * G.M * 64;
  EmitSink *const sink = emit_sink();
  if (ksplit > 1 && (scratch_elems * 2 > (long long)(sink ? kEmitScratchBytes : s.scratch_bytes))) {
    ksplit = 1;
  }
  A.ksplit = ksplit;
  A.scratch = static_cast<_Float16 *>(s.scratch());
  if (sink) {  // a printed program allocates the workspace itself
    A.scratch = ksplit > 1 ? reinterpret_cast<_Float16 *>(kEmitScratch) : nullptr;
    if (ksplit > 1) {
      sink->scratch_bytes = std::max<size_t>(sink->scratch_bytes, (size_t)scratch_elems * 2);
    }
  }
  int const tile_lds = (16 * mt * G.KT + G.nb * 64 * G.KT + (G.lora ? 16 * G.KT + 64 * 16 : 0)) * 2;
  int const out_lds = G.nb * 16 * mt * (64 + 8) * 2;
  int const lds = tile_lds > out_lds ? tile_lds : out_lds;
  if (lds > s.max_lds || (long long)P.grid[0] * ksplit > 2147483647LL) {
    return 0;
  }
  dim3 grid(P.grid[0] * ksplit, P.grid[1], P.grid[2]);
  int rc = 0;
#define MI355_GEMM_CASE(MTV, NBV, PROV, LORAV)                                        \
  if (mt == MTV && G.nb == NBV && G.pro == PROV && G.lora == LORAV) {                 \
    rc = G.wcm ? launch_kt<MTV, NBV, PROV, LORAV, true>(A, grid, lds)                 \
               : launch_kt<MTV, NBV, PROV, LORAV, false>(A, grid, lds);               \
  }
  MI355_GEMM_CASE(1, 1, PRO_NONE, false)
  MI355_GEMM_CASE(2, 1, PRO_NONE, false)
  MI355_GEMM_CASE(4, 1, PRO_NONE, false)
  MI355_GEMM_CASE(1, 1, PRO_EXP, false)
  MI355_GEMM_CASE(1, 1, PRO_SILU, false)
  MI355_GEMM_CASE(1, 2, PRO_NONE, false)
  MI355_GEMM_CASE(1, 1, PRO_SILU_MUL, false)
  MI355_GEMM_CASE(1, 1, PRO_NONE, true)
#undef MI355_GEMM_CASE
  if (rc == 1 && ksplit > 1) {
    rc = launch_combine(A, G.nb, dim3(P.grid[0], P.grid[1], P.grid[2]));
  }
  if (rc == 1) {
    s.last().kernel_id = MI355_KERNEL_F16_GEMM;
    s.last().workgroups = grid.x * grid.y * grid.z;
    s.last().threads = 256;
    s.last().lds_bytes = lds;
    s.last().row_split = ksplit;
  }
  return with_gate(rc);
}

}  // namespace mi355
