// The kernel-level fp16 matmul: C = A . B in fp32 with one fp16 rounding per element, optionally with
// the element-wise consumer of C applied as it is stored.  Three kernels: f16_gemm_any_kernel
// (f16_gemm.h) takes any shape and layout, f16_gemm_nt_kernel streams large k-contiguous operands
// straight into LDS, f16_matmul_kernel takes rows of fewer than eight elements.
#include "f16_gemm.h"
#include "common.h"
#include "f16_gemm_choice.h"

#include <algorithm>
#include <array>
#include <utility>

namespace mi355 {

typedef float float16v __attribute__((ext_vector_type(16)));
constexpr int kThreads = 256;

// The general-purpose GEMM: any shape, either storage order of the operands (element (r, c) of
// A at r * a_rs + c * a_cs, likewise B), unaligned bases.  64x64 output tile per workgroup,
// four wavefronts each owning a 32x32 quadrant, k advanced 32 at a time through LDS, both
// tiles staged k-contiguous with rows padded by 8 halfs.  Element by element, so nothing is too
// small or too odd for it: rows shorter than the 8 elements of a chunk run here.
__global__ __launch_bounds__(kThreads) void f16_matmul_kernel(_Float16 const *__restrict__ A,
                                                             _Float16 const *__restrict__ B,
                                                             _Float16 *__restrict__ C, int m,
                                                             int n, int k, int a_rs, int a_cs,
                                                             int b_rs, int b_cs) {
  constexpr int T = 64, TK = 32, LD = TK + 8;
  __shared__ __attribute__((aligned(16))) _Float16 As[T][LD];
  __shared__ __attribute__((aligned(16))) _Float16 Bs[T][LD];
  int const tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  int const row0 = blockIdx.y * T, col0 = blockIdx.x * T;
  size_t const b = blockIdx.z;
  A += b * (size_t)m * k;
  B += b * (size_t)k * n;
  C += b * (size_t)m * n;
  int const wr = (wave / 2) * 32, wc = (wave % 2) * 32;
  float16v acc;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    acc[i] = 0.0f;
  }
  // a thread stages 8 elements of each tile per step, walking the direction that is
  // contiguous in memory: along k (8 consecutive k of one row) or along the rows / columns
  // (one k of 8 consecutive rows / columns)
  bool const a_along_k = a_cs == 1, b_along_k = b_rs == 1;
  for (int k0 = 0; k0 < k; k0 += TK) {
    {
      int const r = a_along_k ? tid / 4 : (tid % 8) * 8, kk = a_along_k ? (tid % 4) * 8 : tid / 8;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        int const rr = a_along_k ? r : r + j, kj = a_along_k ? kk + j : kk;
        int const gr = row0 + rr, gk = k0 + kj;
        As[rr][kj] = (gr < m && gk < k) ? A[(size_t)gr * a_rs + (size_t)gk * a_cs] : (_Float16)0.0f;
      }
    }
    {
      int const c = b_along_k ? tid / 4 : (tid % 8) * 8, kk = b_along_k ? (tid % 4) * 8 : tid / 8;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        int const cc = b_along_k ? c : c + j, kj = b_along_k ? kk + j : kk;
        int const gc = col0 + cc, gk = k0 + kj;
        Bs[cc][kj] = (gk < k && gc < n) ? B[(size_t)gk * b_rs + (size_t)gc * b_cs] : (_Float16)0.0f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < TK; ks += 16) {
      half8 a = *reinterpret_cast<half8 const *>(&As[wr + lane % 32][ks + 8 * (lane / 32)]);
      half8 bb = *reinterpret_cast<half8 const *>(&Bs[wc + lane % 32][ks + 8 * (lane / 32)]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bb, acc, 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < 16; r++) {
    int row = row0 + wr + (r / 4) * 8 + (lane / 32) * 4 + (r % 4);
    int col = col0 + wc + lane % 32;
    if (row < m && col < n) {
      C[(size_t)row * n + col] = static_cast<_Float16>(acc[r]);
    }
  }
}

// ---------------------------------------------------------------------------------------
// Streaming GEMM for operands whose reduction index is contiguous: A [m][k] row-major and B
// column-major, i.e. B^T [n][k] -- the form every plan of the reference declares its weights in
// (cpp_examples/lora.cc:36-41).  C = A . B, fp32 accumulation, one fp16 rounding per element.
//
//  * a workgroup owns a BM x BN tile of C, its wavefronts WM x WN sub-tiles (256 x 256 with
//    eight wavefronts of 128 x 64);
//  * k advances 32 at a time through a ring of four LDS stages.  A stage is BM + BN rows of 64
//    bytes, filled by direct-to-LDS loads (global_load_lds_dwordx4: no registers, no LDS store
//    instructions) issued three stages ahead; a wavefront waits for its own loads
//    (s_waitcnt vmcnt), one barrier per stage publishes everybody's;
//  * rows are 4 chunks of 16 bytes; chunk q of row r sits at position q ^ ((r >> 2) & 3), so the
//    sixteen rows a 16-lane read phase touches fall on sixteen different bank groups (the lane
//    -> global chunk map of the loads applies the swizzle, since a direct load writes its 64
//    chunks in lane order);
//  * v_mfma_f32_32x32x16_f16, operands one plain 16-byte LDS read per lane, all twelve operand
//    reads of a stage issued before its sixteen matrix instructions;
//  * the tile leaves through LDS as 16-byte row segments; rows and columns past the matrix are
//    clamped on load and masked on store (m and n are arbitrary, k a multiple of 32);
//  * workgroup ids are renumbered so that an XCD (whose 32 compute units share one L2) works on
//    a compact block of tiles: 4 tile rows deep, walked column by column.
struct GemmArgs {
  _Float16 const *A, *Bt;  // [batch][m][k], [batch][n][k]
  _Float16 *C;             // [batch][m][n]
  int m, n, k;
  int tiles_m, tiles_n, tiles_per_batch;
  unsigned total;          // workgroups
};

constexpr int kGemmStages = 4, kGemmBK = 32;

template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN)) void f16_gemm_nt_kernel(GemmArgs const G) {
  constexpr int NW = (BM / WM) * (BN / WN), NT = 64 * NW;
  constexpr int STAGE_HALFS = (BM + BN) * kGemmBK;
  constexpr int AI = BM * 4 / NT, BI = BN * 4 / NT;  // direct loads per thread and stage
  constexpr int TM = WM / 32, TN = WN / 32;
  static_assert(BM * 4 % NT == 0 && BN * 4 % NT == 0, "a stage must split evenly over the threads");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  _Float16 *const ring = reinterpret_cast<_Float16 *>(lds);
  int const tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);

  // ---- which tile: XCD-aware renumbering, then groups of four tile rows -----------------
  unsigned id = blockIdx.x;
  if (G.total % 8 == 0) {
    id = (id % 8) * (G.total / 8) + id / 8;
  }
  int const batch = (int)(id / (unsigned)G.tiles_per_batch);
  int const t = (int)(id % (unsigned)G.tiles_per_batch);
  int const per_group = 4 * G.tiles_n, group = t / per_group, first_m = 4 * group;
  int const gsz = (G.tiles_m - first_m) < 4 ? (G.tiles_m - first_m) : 4;
  int const tile_m = first_m + (t % per_group) % gsz, tile_n = (t % per_group) / gsz;
  int const row0 = tile_m * BM, col0 = tile_n * BN;
  _Float16 const *const Ab = G.A + (size_t)batch * G.m * G.k + (size_t)row0 * G.k;
  _Float16 const *const Bb = G.Bt + (size_t)batch * G.n * G.k + (size_t)col0 * G.k;

  // ---- this lane's share of a stage's loads (byte offsets from the tile's first element) --
  uint32_t a_off[AI], b_off[BI];
#pragma unroll
  for (int i = 0; i < AI; i++) {
    int const p = i * NT + tid, r = p / 4, pos = p % 4;
    int const rr = row0 + r < G.m ? r : G.m - 1 - row0;  // rows past the matrix re-read the last one
    a_off[i] = 2u * (uint32_t)(rr * G.k + 8 * (pos ^ ((r >> 2) & 3)));
  }
#pragma unroll
  for (int i = 0; i < BI; i++) {
    int const p = i * NT + tid, r = p / 4, pos = p % 4;
    int const rr = col0 + r < G.n ? r : G.n - 1 - col0;
    b_off[i] = 2u * (uint32_t)(rr * G.k + 8 * (pos ^ ((r >> 2) & 3)));
  }
  uint32_t const ring_addr = gemm_lds_address(ring);
  auto issue = [&](int kt) {
    uint32_t const stage = ring_addr + 2u * (uint32_t)((kt % kGemmStages) * STAGE_HALFS);
    _Float16 const *ag = Ab + (size_t)kt * kGemmBK, *bg = Bb + (size_t)kt * kGemmBK;
#pragma unroll
    for (int i = 0; i < AI; i++) {
      gemm_dma16(ag, a_off[i], stage + 16u * (uint32_t)(i * NT + wave * 64));
    }
#pragma unroll
    for (int i = 0; i < BI; i++) {
      gemm_dma16(bg, b_off[i], stage + 2u * (uint32_t)(BM * kGemmBK) + 16u * (uint32_t)(i * NT + wave * 64));
    }
  };

  // ---- operand reads: row (lane % 32) of a 32-row block, chunk 2 s + lane / 32 of its row -----
  int const wm0 = (wave / (BN / WN)) * WM, wn0 = (wave % (BN / WN)) * WN;
  int const l32 = lane & 31, hi = lane >> 5, swz = (l32 >> 2) & 3;
  int const x0 = ((0 + hi) ^ swz) << 3, x1 = ((2 + hi) ^ swz) << 3;  // halfs, k steps 0 and 1
  int const a_lane = (wm0 + l32) * kGemmBK, b_lane = BM * kGemmBK + (wn0 + l32) * kGemmBK;

  float16v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
      for (int e = 0; e < 16; e++) {
        acc[i][j][e] = 0.0f;
      }
    }
  }

  int const KT = G.k / kGemmBK;
  constexpr int LPS = AI + BI;  // loads per thread and stage
#pragma unroll
  for (int st = 0; st < kGemmStages - 1; st++) {
    if (st < KT) {
      issue(st);
    }
  }
  // operand reads of k step `s` (16 k) of the stage in ring slot `slot`
  auto read_step = [&](int slot, int s, half8 (&af)[TM], half8 (&bf)[TN]) {
    _Float16 const *stage = ring + slot * STAGE_HALFS;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      af[i] = *reinterpret_cast<half8 const *>(stage + a_lane + 32 * i * kGemmBK + (s ? x1 : x0));
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      bf[j] = *reinterpret_cast<half8 const *>(stage + b_lane + 32 * j * kGemmBK + (s ? x1 : x0));
    }
  };
  auto multiply = [&](half8 const (&af)[TM], half8 const (&bf)[TN]) {
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
      for (int j = 0; j < TN; j++) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
      }
    }
  };
  // stage `kt` has landed (this wavefront's share) when at most the stages issued after it --
  // up to stage kt + 2 by then -- are outstanding
  auto landed = [&](int kt) {
    int const later = (KT - 1 - kt) < 2 ? (KT - 1 - kt) : 2;
    if (later == 2) {
      gemm_wait_vm<2 * LPS>();
    } else if (later == 1) {
      gemm_wait_vm<LPS>();
    } else {
      gemm_wait_vm<0>();
    }
  };
  // The loop is skewed by half a stage so that every batch of operand reads is followed by
  // eight matrix instructions on operands that are already in registers: the second k step of
  // stage kt is read before the first one is multiplied, and the first k step of stage kt + 1
  // -- published by the barrier in the middle -- before the second one is.
  half8 a0[TM], b0[TN], a1[TM], b1[TN];
  landed(0);
  __syncthreads();
  if (kGemmStages - 1 < KT) {
    issue(kGemmStages - 1);
  }
  read_step(0, 0, a0, b0);
  // (The last stage stands behind the loop: the multiplications would otherwise wait for the next stage's reads,
  // which one of the two ways there does not make.)
  for (int kt = 0; kt + 1 < KT; kt++) {
    read_step(kt % kGemmStages, 1, a1, b1);
    multiply(a0, b0);
    landed(kt + 1);
    // (this wavefront's reads of stage kt are in registers before it lets the others go on)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();  // stage kt + 1 is there for everybody; stage kt is in everybody's registers
    if (kt + kGemmStages < KT) {
      issue(kt + kGemmStages);  // into the slot stage kt leaves
    }
    read_step((kt + 1) % kGemmStages, 0, a0, b0);
    multiply(a1, b1);
  }
  read_step((KT - 1) % kGemmStages, 1, a1, b1);
  multiply(a0, b0);
  multiply(a1, b1);

  // ---- the tile leaves through LDS: each wavefront its own WM x WN piece -------------------
  __syncthreads();  // the last stage's operand reads are done everywhere
  constexpr int LDW = WN;
  _Float16 *const piece = ring + wave * WM * LDW;
  static_assert(NW * WM * LDW * 2 <= kGemmStages * STAGE_HALFS * 2, "pieces must fit the ring");
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
      for (int e = 0; e < 16; e++) {
        // acc[e] = C[32 i + 8 (e / 4) + 4 (lane / 32) + e % 4][32 j + lane % 32]
        piece[(32 * i + 8 * (e / 4) + 4 * hi + (e % 4)) * LDW + 32 * j + l32] = static_cast<_Float16>(acc[i][j][e]);
      }
    }
  }
  // (a wavefront reads back only what it wrote: its own LDS operations complete in order)
  __builtin_amdgcn_wave_barrier();
  _Float16 *const Cb = G.C + (size_t)batch * G.m * G.n;
  constexpr int CPR = WN / 8;  // 16-byte chunks per row of the piece
  for (int e = lane; e < WM * CPR; e += 64) {
    int const r = e / CPR, c8 = (e % CPR) * 8;
    int const row = row0 + wm0 + r, col = col0 + wn0 + c8;
    if (row < G.m && col < G.n) {
      half8 const v = *reinterpret_cast<half8 const *>(piece + r * LDW + c8);
      if (col + 8 <= G.n) {
        *reinterpret_cast<half8_any *>(Cb + (size_t)row * G.n + col) = v;
      } else {
        for (int x = 0; x < 8 && col + x < G.n; x++) {
          Cb[(size_t)row * G.n + col + x] = v[x];
        }
      }
    }
  }
}

// out[b][c][r] = in[b][r][c] through a 64 x 64 LDS tile: the row-major copy of a column-major
// tensor (or the other way round) for the operators that index their inputs flat.
__global__ __launch_bounds__(kThreads) void f16_transpose_kernel(_Float16 const *__restrict__ in,
                                                                _Float16 *__restrict__ out, int rows,
                                                                int cols) {
  __shared__ _Float16 tile[64][66];
  size_t const b = blockIdx.z;
  in += b * (size_t)rows * cols;
  out += b * (size_t)rows * cols;
  int const r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  for (int e = threadIdx.x; e < 64 * 64; e += kThreads) {
    int const r = e / 64, c = e % 64;
    if (r0 + r < rows && c0 + c < cols) {
      tile[r][c] = in[(size_t)(r0 + r) * cols + c0 + c];
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 64 * 64; e += kThreads) {
    int const c = e / 64, r = e % 64;
    if (r0 + r < rows && c0 + c < cols) {
      out[(size_t)(c0 + c) * rows + r0 + r] = tile[r][c];
    }
  }
}

// C[i] = fp16(sum over the k ranges of partial[s][i]), added in fp32 in range order, and the
// consumer.  Four elements a thread: a 16-byte load per range.  `n` elements of a matrix; a batch is one of n elements
// but where it is two products, whose second follows the first in the same thread: its consumer may read the first's.
template <int PRODUCTS>
__global__ void f16_gemm_fold_kernel(AnyGemm const G, size_t n) {
  size_t const stride = (size_t)gridDim.x * blockDim.x * 4;
  for (size_t i = (blockIdx.x * (size_t)blockDim.x + threadIdx.x) * 4; i < n; i += stride) {
    int const left = n - i < 4 ? (int)(n - i) : 4;
    for (int product = 0; product < PRODUCTS; product++) {
      _Float16 *const C = G.C + product * G.c_step, *const E = G.E + product * G.e_step;
      _Float16 const *const X = G.X + product * G.x_step;
      int const epilogue = product == 0 ? G.epilogue : G.epilogue2;
      float4v r = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int s = 0; s < G.ksplit; s++) {
        float const *p = G.partial + ((size_t)s * PRODUCTS + product) * n + i;
        if (left == 4) {
          float4v const v = *reinterpret_cast<float4_any const *>(p);
#pragma unroll
          for (int e = 0; e < 4; e++) {
            r[e] += v[e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < 3; e++) {
            r[e] += e < left ? p[e] : 0.0f;
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if (e < left) {
          _Float16 const v = static_cast<_Float16>(r[e]);
          C[i + e] = v;
          if (epilogue != EPI_NONE) {
            float const x = epilogue >= EPI_ADD ? static_cast<float>(X[i + e]) : 0.0f;
            E[i + e] = static_cast<_Float16>(epilogue_value(epilogue, static_cast<float>(v), x));
          }
        }
      }
    }
  }
}

static int launch_transpose(_Float16 const *in, _Float16 *out, int batch, int rows, int cols) {
  dim3 grid((cols + 63) / 64, (rows + 63) / 64, batch);
  MI355_HIP(launch_kernel(f16_transpose_kernel, grid, kThreads, 0, state().stream(), in, out, rows, cols));
  return MI355_OK;
}

template <int BM, int BN, int WM, int WN>
static int launch_gemm_nt(GemmArgs &G, int batch) {
  constexpr int threads = 64 * (BM / WM) * (BN / WN);
  constexpr int lds = kGemmStages * (BM + BN) * kGemmBK * 2;
  G.tiles_m = (G.m + BM - 1) / BM;
  G.tiles_n = (G.n + BN - 1) / BN;
  G.tiles_per_batch = G.tiles_m * G.tiles_n;
  long long const total = (long long)G.tiles_per_batch * batch;
  if (total > 2147483647LL) {
    return fail(MI355_ERR_UNSUPPORTED, "matmul has too many output tiles");
  }
  G.total = (unsigned)total;
  auto *fn = f16_gemm_nt_kernel<BM, BN, WM, WN>;
  MI355_GRANT_LDS(fn, lds);
  MI355_HIP(launch_kernel(fn, G.total, threads, lds, state().stream(), G));
  return MI355_OK;
}

// ---- the tiles of f16_gemm_choice.h: instantiations and launches ----------------------------------
namespace {

struct TileKernel {
  void (*fn)(AnyGemm);
  int lds;
  void (*deep)(AnyGemm) = nullptr;  // four stages ahead instead of two
};
template <bool A_KC, int I>
constexpr GemmTile kTile = kGemmTiles[I];
template <int I>
constexpr GemmTile kTile<false, I> = kGemmTilesColumnMajorA[I];

template <int I, bool A_KC, bool B_KC>
constexpr TileKernel tile_kernel() {
  constexpr GemmTile t = kTile<A_KC, I>;
  if constexpr (t.kind == STAGED) {
    constexpr int lds = any_gemm_lds<t.bm, t.bn, t.wm, t.wn, t.kg, A_KC, B_KC>();
    if constexpr (t.bm <= 64 && t.bn == 64) {
      return {f16_gemm_any_kernel<t.bm, t.bn, t.wm, t.wn, t.kg, A_KC, B_KC>, lds, f16_gemm_any_kernel<t.bm, t.bn, t.wm, t.wn, t.kg, A_KC, B_KC, 4>};
    } else {
      return {f16_gemm_any_kernel<t.bm, t.bn, t.wm, t.wn, t.kg, A_KC, B_KC>, lds};
    }
  } else if constexpr (t.kind == DIRECT) {
    return {f16_gemm_direct_kernel<t.bm, t.bn, t.wm, t.wn, B_KC>, direct_gemm_lds<t.bm, t.bn>()};
  } else {
    return {f16_gemm_waves_kernel<t.bm, t.bn, kWavesRing, B_KC>, waves_gemm_lds<t.bm, t.bn, kWavesRing>()};
  }
}
template <bool A_KC, bool B_KC, size_t... I>
TileKernel tile_kernel_at(int i, std::index_sequence<I...>) {
  static constexpr std::array<TileKernel, sizeof...(I)> all = {tile_kernel<(int)I, A_KC, B_KC>()...};
  return all[i];
}
TileKernel tile_kernel_of(int i, bool a_kc, bool b_kc) {
  using Row = std::make_index_sequence<sizeof(kGemmTiles) / sizeof(GemmTile)>;
  using Col = std::make_index_sequence<sizeof(kGemmTilesColumnMajorA) / sizeof(GemmTile)>;
  if (a_kc) {
    return b_kc ? tile_kernel_at<true, true>(i, Row{}) : tile_kernel_at<true, false>(i, Row{});
  }
  return b_kc ? tile_kernel_at<false, true>(i, Col{}) : tile_kernel_at<false, false>(i, Col{});
}

// The geometry of these tiles in so many ranges.
int place_tiles(AnyGemm &G, int batch, GemmTile const &t, int ksplit) {
  G.tiles_m = (G.m + t.bm - 1) / t.bm;
  G.tiles_n = (G.n + t.bn - 1) / t.bn;
  G.group = G.tiles_m * t.bm <= 512 && (size_t)G.k * G.n >= (2u << 20) ? G.tiles_m : 4;
  G.ksplit = ksplit;
  G.steps_per_range = t.kind == WAVES ? (G.k / 32 + G.ksplit - 1) / G.ksplit : (G.k / 64 + G.ksplit * t.kg - 1) / (G.ksplit * t.kg);
  G.partial = static_cast<float *>(state().scratch());
  long long const total = (long long)G.tiles_m * G.tiles_n * batch * G.ksplit;
  if (total > 2147483647LL) {
    return fail(MI355_ERR_UNSUPPORTED, "matmul has too many output tiles");
  }
  G.total = (unsigned)total;
  return MI355_OK;
}

int launch_gemm_tiles(AnyGemm &G, int batch, bool a_kc, bool b_kc, GemmChoice const &choice, bool two = false) {
  GemmTile const &t = (a_kc ? kGemmTiles : kGemmTilesColumnMajorA)[choice.tile];
  TileKernel const kernel = tile_kernel_of(choice.tile, a_kc, b_kc);
  if (int rc = place_tiles(G, batch, t, choice.ksplit)) {
    return rc;
  }
  // Stages further ahead where a range is long (un-fused MLPs, us: 182 x 1830 x 1807 41.6 -> 33.3, 300 x 1027 x 2049 39.3
  // -> 33.9, 500 x 1999 x 3001 78.0 -> 75.1); a short one has them all in its last stages, which load under conditions
  // (from 6 on, 34 x 1455 x 790 27.7 -> 29.2).
  auto *const fn = kernel.deep != nullptr && G.steps_per_range >= 16 ? kernel.deep : kernel.fn;
  MI355_GRANT_LDS(fn, kernel.lds);
  MI355_HIP(launch_kernel(fn, G.total, t.threads(), kernel.lds, state().stream(), G));
  if (G.ksplit > 1) {
    size_t const n = (size_t)batch * G.m * G.n / (two ? 2 : 1), blocks = (n / 4 + kThreads) / kThreads;
    MI355_HIP(launch_kernel(two ? f16_gemm_fold_kernel<2> : f16_gemm_fold_kernel<1>, (unsigned)std::min<size_t>(blocks, 4096), kThreads, 0,
                            state().stream(), G, n));
  }
  return MI355_OK;
}

// Both products in every workgroup, columns of each side by side.
template <int HALF, int WN, bool B_KC>
int launch_gemm_two(AnyGemm &G) {
  auto *const fn = f16_gemm_direct_kernel<64, 2 * HALF, 32, WN, B_KC, true>;
  constexpr int lds = direct_gemm_lds<64, 2 * HALF>();
  if (int rc = place_tiles(G, 1, GemmTile{DIRECT, 64, HALF, 32, WN, 1}, 1)) {
    return rc;
  }
  MI355_GRANT_LDS(fn, lds);
  MI355_HIP(launch_kernel(fn, G.total, 64 * 2 * (2 * HALF / WN), lds, state().stream(), G));
  return MI355_OK;
}

// The matmul, and the consumer where the kernel that runs applies it: *applied says whether.
int run_matmul(AnyGemm G, int batch, int a_column_major, int b_column_major, bool *applied) {
  *applied = false;
  int const m = G.m, n = G.n, k = G.k;
  if (batch < 0 || m < 0 || n < 0 || k < 0) {
    return fail(MI355_ERR_INVALID, "negative matmul extent");
  }
  if (batch == 0 || m == 0 || n == 0) {
    return MI355_OK;
  }
  if (batch > 65535) {
    return fail(MI355_ERR_UNSUPPORTED, "batch %d exceeds grid.z", batch);
  }
  if (state().f16_matmul_route == 1 && k > 0) {  // an empty sum is zeros from the kernel below
    return vendor_gemm(G.A, G.B, G.C, batch, m, n, k, a_column_major, b_column_major);
  }
  bool const aligned = ((reinterpret_cast<uintptr_t>(G.A) | reinterpret_cast<uintptr_t>(G.B)) & 15) == 0;
  GemmChoice const choice =
      choose_gemm({batch, m, n, k, a_column_major != 0, b_column_major != 0, aligned, state().scratch() == nullptr ? 0 : state().scratch_bytes,
                   state().planes() == nullptr ? 0 : state().planes_bytes});
  // Transposed copies go into this queue's plane memory (the fingerprint matmuls' workspace: work of one
  // queue is ordered, so the two never overlap).
  char *room = state().planes();
  if (choice.copy_a) {  // the buffer is [k][m] per matrix
    auto *at = reinterpret_cast<_Float16 *>(room);
    if (int rc = launch_transpose(G.A, at, batch, k, m)) {
      return rc;
    }
    G.A = at;
    room += ((size_t)batch * m * k * 2 + 255) & ~(size_t)255;
  }
  if (choice.copy_b) {  // the buffer is [k][n] per matrix
    auto *bt = reinterpret_cast<_Float16 *>(room);
    if (int rc = launch_transpose(G.B, bt, batch, k, n)) {
      return rc;
    }
    G.B = bt;
  }
  if (choice.route == GEMM_BIG) {
    GemmArgs N{G.A, G.B, G.C, m, n, k, 0, 0, 0, 0};
    return launch_gemm_nt<256, 256, 128, 64>(N, batch);
  }
  if (choice.route == GEMM_TILES) {
    *applied = true;
    G.epilogue2 = G.epilogue;
    G.a_rows = m;
    G.b_step = (long long)k * n;
    G.c_step = G.x_step = G.e_step = (long long)m * n;
    return launch_gemm_tiles(G, batch, !a_column_major || choice.copy_a, b_column_major != 0, choice);
  }
  dim3 grid((n + 63) / 64, (m + 63) / 64, batch);
  MI355_HIP(launch_kernel(f16_matmul_kernel, grid, kThreads, 0, state().stream(), G.A, G.B, G.C, m, n, k, a_column_major ? 1 : k,
                          a_column_major ? m : 1, b_column_major ? 1 : n, b_column_major ? k : 1));
  return MI355_OK;
}

}  // namespace
}  // namespace mi355

using namespace mi355;

extern "C" int mi355_f16_matmul_layout(void const *A, void const *B, void *C, int batch, int m,
                                       int n, int k, int a_column_major, int b_column_major) {
  MI355_REQUIRE_INIT();
  AnyGemm G{};
  G.A = static_cast<_Float16 const *>(A);
  G.B = static_cast<_Float16 const *>(B);
  G.C = static_cast<_Float16 *>(C);
  G.m = m;
  G.n = n;
  G.k = k;
  bool applied;
  return run_matmul(G, batch, a_column_major, b_column_major, &applied);
}

extern "C" int mi355_f16_matmul(void const *A, void const *B, void *C, int batch, int m, int n,
                                int k) {
  return mi355_f16_matmul_layout(A, B, C, batch, m, n, k, 0, 0);
}

static bool consumer_of(int op, int x_first, int *epilogue) {
  switch (op) {
    case 0: *epilogue = EPI_NONE; return true;
    case KN_EXP_OP: *epilogue = EPI_EXP; return true;
    case KN_SILU_OP: *epilogue = EPI_SILU; return true;
    case KN_ADD_OP: *epilogue = EPI_ADD; return true;
    case KN_MUL_OP: *epilogue = EPI_MUL; return true;
    case KN_DIV_OP: *epilogue = x_first ? EPI_RDIV : EPI_DIV; return true;
    default: return false;
  }
}

extern "C" int mi355_f16_matmul_then(void const *A, void const *B, void *C, int batch, int m, int n, int k,
                                     int a_column_major, int b_column_major, int op, void const *X, int x_first, void *E) {
  MI355_REQUIRE_INIT();
  bool const binary = op == KN_ADD_OP || op == KN_MUL_OP || op == KN_DIV_OP;
  if (!binary && op != KN_EXP_OP && op != KN_SILU_OP) {
    return fail(MI355_ERR_UNSUPPORTED, "op %d after a matmul", op);
  }
  AnyGemm G{};
  G.A = static_cast<_Float16 const *>(A);
  G.B = static_cast<_Float16 const *>(B);
  G.C = static_cast<_Float16 *>(C);
  G.X = static_cast<_Float16 const *>(X);
  G.E = static_cast<_Float16 *>(E);
  G.m = m;
  G.n = n;
  G.k = k;
  consumer_of(op, x_first, &G.epilogue);
  bool applied;
  if (int rc = run_matmul(G, batch, a_column_major, b_column_major, &applied)) {
    return rc;
  }
  size_t const count = (size_t)batch * m * n;
  if (applied || count == 0) {
    return MI355_OK;
  }
  if (!binary) {
    return mi355_f16_unary(op, C, E, count);
  }
  int const dims[3] = {batch, m, n};
  return mi355_f16_binary(op, x_first ? X : C, dims, x_first ? C : X, dims, E, dims, 3);
}

extern "C" int mi355_f16_matmul_two(void const *A, int a_column_major, int b_column_major, int batch, int m, int n, int k,
                                    mi355_matmul_out const *first, mi355_matmul_out const *second, int *taken) {
  MI355_REQUIRE_INIT();
  if (first == nullptr || second == nullptr || taken == nullptr) {
    return fail(MI355_ERR_INVALID, "no products or no place for the answer");
  }
  *taken = 0;
  AnyGemm G{};
  G.A = static_cast<_Float16 const *>(A);
  G.B = static_cast<_Float16 const *>(first->B);
  G.C = static_cast<_Float16 *>(first->C);
  G.X = static_cast<_Float16 const *>(first->X);
  G.E = static_cast<_Float16 *>(first->E);
  G.m = m;
  G.n = n;
  G.k = k;
  if (!consumer_of(first->op, first->x_first, &G.epilogue) || !consumer_of(second->op, second->x_first, &G.epilogue2)) {
    return fail(MI355_ERR_UNSUPPORTED, "op after a matmul");
  }
  uintptr_t const all = reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(first->B) | reinterpret_cast<uintptr_t>(second->B);
  uintptr_t const results = reinterpret_cast<uintptr_t>(first->C) | reinterpret_cast<uintptr_t>(second->C) |
                            reinterpret_cast<uintptr_t>(first->E) | reinterpret_cast<uintptr_t>(second->E) |
                            reinterpret_cast<uintptr_t>(first->X) | reinterpret_cast<uintptr_t>(second->X);
  if (batch != 1 || m <= 0 || n <= 0 || k <= 0 || ((all | results) & 1) != 0 || state().f16_matmul_route == 1) {
    return MI355_OK;
  }
  auto elements = [](void const *from, void const *to) {
    return (long long)(reinterpret_cast<intptr_t>(to) - reinterpret_cast<intptr_t>(from)) / 2;
  };
  G.a_rows = 0;
  G.b_step = elements(first->B, second->B);
  G.c_step = elements(first->C, second->C);
  G.x_step = elements(first->X, second->X);
  G.e_step = elements(first->E, second->E);
  bool const reads_first = G.epilogue2 >= EPI_ADD && (second->X == first->C || (first->E != nullptr && second->X == first->E));
  GemmTwoChoice const two = choose_gemm_two({1, m, n, k, a_column_major != 0, b_column_major != 0, (all & 15) == 0,
                                             state().scratch() == nullptr ? 0 : state().scratch_bytes,
                                             state().planes() == nullptr ? 0 : state().planes_bytes}, reads_first);
  if (two.half != 0) {
    *taken = 1;
    if (two.half == 128) {
      return b_column_major ? launch_gemm_two<128, 64, true>(G) : launch_gemm_two<128, 64, false>(G);
    }
    return b_column_major ? launch_gemm_two<64, 32, true>(G) : launch_gemm_two<64, 32, false>(G);
  }
  if (!two.tiles) {
    return MI355_OK;
  }
  *taken = 1;
  return launch_gemm_tiles(G, 2, !a_column_major, b_column_major != 0, two.choice, true);
}

extern "C" int mi355_f16_transpose(void const *in, void *out, int batch, int rows, int cols) {
  MI355_REQUIRE_INIT();
  if (batch < 0 || rows < 0 || cols < 0) {
    return fail(MI355_ERR_INVALID, "negative transpose extent");
  }
  if (batch == 0 || rows == 0 || cols == 0) {
    return MI355_OK;
  }
  if (batch > 65535 || (rows + 63) / 64 > 65535) {
    return fail(MI355_ERR_UNSUPPORTED, "transpose grid out of range");
  }
  if (in == out) {
    return fail(MI355_ERR_INVALID, "transpose in place");
  }
  return launch_transpose(static_cast<_Float16 const *>(in), static_cast<_Float16 *>(out), batch, rows, cols);
}
