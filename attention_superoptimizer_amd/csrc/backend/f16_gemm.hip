// The kernel-level fp16 matmul: C = A . B in fp32 with one fp16 rounding per element, optionally with
// the element-wise consumer of C applied as it is stored.  Three kernels: f16_gemm_any_kernel
// (f16_gemm.h) takes any shape and layout, f16_gemm_nt_kernel streams large k-contiguous operands
// straight into LDS, f16_matmul_kernel takes rows of fewer than eight elements.
#include "f16_gemm.h"
#include "common.h"

#include <algorithm>
#include <cmath>
#include <vector>

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
  for (int kt = 0; kt < KT; kt++) {
    int const slot = kt % kGemmStages;
    read_step(slot, 1, a1, b1);
    multiply(a0, b0);
    if (kt + 1 < KT) {
      landed(kt + 1);
      // (this wavefront's reads of stage kt are in registers before it lets the others go on)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __syncthreads();  // stage kt + 1 is there for everybody; stage kt is in everybody's registers
      if (kt + kGemmStages < KT) {
        issue(kt + kGemmStages);  // into the slot stage kt leaves
      }
      read_step((kt + 1) % kGemmStages, 0, a0, b0);
    }
    multiply(a1, b1);
  }

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
  bool const vec = G.n % 8 == 0;
  for (int e = lane; e < WM * CPR; e += 64) {
    int const r = e / CPR, c8 = (e % CPR) * 8;
    int const row = row0 + wm0 + r, col = col0 + wn0 + c8;
    if (row < G.m && col < G.n) {
      half8 const v = *reinterpret_cast<half8 const *>(piece + r * LDW + c8);
      if (vec && col + 8 <= G.n) {
        *reinterpret_cast<half8 *>(Cb + (size_t)row * G.n + col) = v;
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
// consumer.  Four elements a thread: a 16-byte load per range.
__global__ void f16_gemm_fold_kernel(AnyGemm const G, size_t n) {
  size_t const stride = (size_t)gridDim.x * blockDim.x * 4;
  for (size_t i = (blockIdx.x * (size_t)blockDim.x + threadIdx.x) * 4; i < n; i += stride) {
    float4v r = {0.0f, 0.0f, 0.0f, 0.0f};
    int const left = n - i < 4 ? (int)(n - i) : 4;
    for (int s = 0; s < G.ksplit; s++) {
      float const *p = G.partial + (size_t)s * n + i;
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
        G.C[i + e] = v;
        if (G.epilogue != EPI_NONE) {
          float const x = G.epilogue >= EPI_ADD ? static_cast<float>(G.X[i + e]) : 0.0f;
          G.E[i + e] = static_cast<_Float16>(epilogue_value(G.epilogue, static_cast<float>(v), x));
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

// ---- f16_gemm_any_kernel: instantiations and the choice between them -------------------------
namespace {

// f16_gemm_any_kernel, f16_gemm_direct_kernel, f16_gemm_waves_kernel
enum TileKind { STAGED, DIRECT, WAVES };
struct AnyTile {
  int bm, bn, wm, wn, kg, lds;
  TileKind kind;
  void (*fn)(AnyGemm);
  int threads() const { return 64 * (bm / wm) * (bn / wn) * kg; }
};
template <int BM, int BN, int WM, int WN, int KG, bool A_KC, bool B_KC>
AnyTile any_tile() {
  return {BM, BN, WM, WN, KG, any_gemm_lds<BM, BN, WM, WN, KG, A_KC, B_KC>(), STAGED, f16_gemm_any_kernel<BM, BN, WM, WN, KG, A_KC, B_KC>};
}
template <int BM, int BN, int WM, int WN, bool B_KC>
AnyTile direct_tile() {
  return {BM, BN, WM, WN, 1, direct_gemm_lds<BM, BN>(), DIRECT, f16_gemm_direct_kernel<BM, BN, WM, WN, B_KC>};
}
template <int BM, int BN, int RING, bool B_KC>
AnyTile waves_tile() {
  return {BM, BN, BM, BN, 4, waves_gemm_lds<BM, BN, RING>(), WAVES, f16_gemm_waves_kernel<BM, BN, RING, B_KC>};
}
// [A k-contiguous][B k-contiguous]; a column-major A is rare (a layout search may ask for one), so
// it gets the middle tiles only
template <bool B_KC>
std::vector<AnyTile> any_tiles_row_major_a() {
  return {any_tile<16, 64, 16, 16, 1, true, B_KC>(),  any_tile<16, 64, 16, 16, 2, true, B_KC>(),
          any_tile<32, 64, 32, 16, 1, true, B_KC>(),  any_tile<32, 64, 32, 16, 2, true, B_KC>(),
          any_tile<64, 64, 32, 32, 1, true, B_KC>(),  any_tile<64, 64, 32, 32, 2, true, B_KC>(),
          any_tile<64, 128, 32, 64, 1, true, B_KC>(), any_tile<64, 128, 32, 64, 2, true, B_KC>(),
          any_tile<128, 128, 64, 64, 1, true, B_KC>(), direct_tile<64, 64, 32, 32, B_KC>(),
          direct_tile<64, 128, 32, 64, B_KC>(),        direct_tile<128, 64, 64, 32, B_KC>(),
          waves_tile<16, 64, 4, B_KC>(),               waves_tile<32, 64, 4, B_KC>()};
}
std::vector<AnyTile> const &any_tiles(bool a_kc, bool b_kc) {
  static std::vector<AnyTile> const row[2] = {any_tiles_row_major_a<false>(), any_tiles_row_major_a<true>()};
  static std::vector<AnyTile> const col[2] = {
      {any_tile<64, 64, 32, 32, 1, false, false>(), any_tile<64, 64, 32, 32, 2, false, false>()},
      {any_tile<64, 64, 32, 32, 1, false, true>(), any_tile<64, 64, 32, 32, 2, false, true>()}};
  return (a_kc ? row : col)[b_kc ? 1 : 0];
}

// Microseconds a tile shape is expected to take: a line fitted to 27,000 timed launches (114 shapes,
// m from 1 to 2048, n and k from 64 to 5504; the choice it makes is 2.6 % above the best on
// average).  A launch, then either the latency of its k stages one after another (0.24 us each) or,
// with the compute units full, what they have to move: 128-byte rows through the vector cache, into
// LDS and from there to the operands, and the matrix instructions.  k ranges need a second launch.
// (The kernels that load LDS directly: 3.2 us, and 35 bytes a cycle per compute unit; a lone workgroup
// waits 1.4 times as long for a stage, but not where wavefronts go their own ways.  15 shapes, within 15 %.)
double any_gemm_cost(AnyTile const &t, int batch, int m, int n, int k, int ksplit) {
  if (t.kind != STAGED) {
    double const stages = (k / 32 + 2 * ksplit - 1) / (2 * ksplit), stage = (t.bm + t.bn) * 128.0 / 35.0 / 2400.0;
    double per_cu = (double)((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn) * batch * ksplit / 256.0;
    if (t.kind == WAVES || per_cu < 3.0) {
      per_cu = std::ceil(per_cu);  // (the compute unit with the most workgroups is the last to finish)
    }
    double const us = 3.2 + stages * stage * std::max(per_cu, t.kind == DIRECT ? 1.4 : 1.0) + per_cu * 0.9e-4 * t.bm * t.bn;
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

int launch_gemm_any(AnyGemm &G, int batch, bool a_kc, bool b_kc) {
  AnyTile const *best = nullptr;
  double least = 0.0;
  int ksplit = 1;
  size_t const range_bytes = (size_t)batch * G.m * G.n * sizeof(float);
  bool const chunks = a_kc && (b_kc || G.n % 8 == 0) &&
                      ((reinterpret_cast<uintptr_t>(G.A) | reinterpret_cast<uintptr_t>(G.B)) & 15) == 0;
  for (AnyTile const &t : any_tiles(a_kc, b_kc)) {
    if (t.kind != STAGED && (!chunks || G.k % (t.kind == DIRECT ? 64 : 32) != 0)) {
      continue;
    }
    for (int s : {1, 2, 3, 4, 6, 8, 12, 16}) {
      // (a range is a stage per group at least, and the ranges' sums fit this queue's scratch)
      if (s > 1 && (G.k / 64 < s * (t.kind == WAVES ? 1 : t.kg) || state().scratch() == nullptr || range_bytes * s > state().scratch_bytes)) {
        break;
      }
      double const us = any_gemm_cost(t, batch, G.m, G.n, G.k, s);
      if (best == nullptr || us < least) {
        best = &t;
        least = us;
        ksplit = s;
      }
    }
  }
  G.tiles_m = (G.m + best->bm - 1) / best->bm;
  G.tiles_n = (G.n + best->bn - 1) / best->bn;
  G.tiles_per_batch = G.tiles_m * G.tiles_n;
  G.ksplit = ksplit;
  G.steps_per_range = best->kind == WAVES ? (G.k / 32 + ksplit - 1) / ksplit
                                          : (G.k / 64 + ksplit * best->kg - 1) / (ksplit * best->kg);
  G.partial = static_cast<float *>(state().scratch());
  long long const total = (long long)G.tiles_per_batch * batch * ksplit;
  if (total > 2147483647LL) {
    return fail(MI355_ERR_UNSUPPORTED, "matmul has too many output tiles");
  }
  G.total = (unsigned)total;
  MI355_GRANT_LDS(best->fn, best->lds);
  MI355_HIP(launch_kernel(best->fn, G.total, best->threads(), best->lds, state().stream(), G));
  if (ksplit > 1) {
    size_t const n = (size_t)batch * G.m * G.n, blocks = (n / 4 + kThreads) / kThreads;
    MI355_HIP(launch_kernel(f16_gemm_fold_kernel, (unsigned)std::min<size_t>(blocks, 4096), kThreads, 0, state().stream(), G, n));
  }
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
  // 256 x 256 tiles once they alone fill the chip.  That kernel wants k contiguous in both operands,
  // k in whole steps of 32 and 16-byte aligned rows; an operand stored the other way round is first
  // copied transposed into this queue's plane memory (the fingerprint matmuls' workspace: work of
  // one queue is ordered, so the two never overlap).
  long long const big_tiles = (long long)((m + 255) / 256) * ((n + 255) / 256) * batch;
  bool const aligned = ((reinterpret_cast<uintptr_t>(G.A) | reinterpret_cast<uintptr_t>(G.B)) & 15) == 0;
  size_t const a_bytes = a_column_major ? (size_t)batch * m * k * 2 : 0;
  size_t const b_bytes = b_column_major ? 0 : (size_t)batch * k * n * 2;
  size_t const a_room = (a_bytes + 255) & ~(size_t)255;
  bool const fits = state().planes() != nullptr && a_room + b_bytes <= state().planes_bytes;
  if (big_tiles >= 192 && k >= 256 && k % kGemmBK == 0 && aligned && fits && (size_t)std::max(m, n) * (size_t)k < ((size_t)1 << 30)) {
    GemmArgs N{G.A, G.B, G.C, m, n, k, 0, 0, 0, 0};
    if (a_column_major) {  // the buffer is [k][m] per matrix
      auto *at = reinterpret_cast<_Float16 *>(state().planes());
      if (int rc = launch_transpose(G.A, at, batch, k, m)) {
        return rc;
      }
      N.A = at;
    }
    if (!b_column_major) {  // the buffer is [k][n] per matrix
      auto *bt = reinterpret_cast<_Float16 *>(state().planes() + a_room);
      if (int rc = launch_transpose(G.B, bt, batch, k, n)) {
        return rc;
      }
      N.Bt = bt;
    }
    return launch_gemm_nt<256, 256, 128, 64>(N, batch);
  }
  // Byte offsets inside a tile are 31-bit numbers; a contiguous direction shorter than a chunk of
  // eight goes element by element.
  int const a_row = a_column_major ? m : k, b_row = b_column_major ? k : n;
  if (std::min(a_row, b_row) >= 8 && std::max(a_row, b_row) < (1 << 22)) {
    *applied = true;
    return launch_gemm_any(G, batch, !a_column_major, b_column_major != 0);
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
  G.epilogue = op == KN_EXP_OP    ? EPI_EXP
               : op == KN_SILU_OP ? EPI_SILU
               : op == KN_ADD_OP  ? EPI_ADD
               : op == KN_MUL_OP  ? EPI_MUL
               : x_first          ? EPI_RDIV
                                  : EPI_DIV;
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
