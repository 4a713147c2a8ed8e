// Kernels of the kernel-level fp16 matmul that take any shape: C = A . B for a batch of matrices,
// either storage order of each operand, any alignment, an element-wise consumer applied on the way
// out.  Launches and the choice between instantiations: f16_gemm.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mi355 {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
// 16 bytes anywhere an element may start (rows of an odd length): the same instructions, the
// compiler is told not to count on their alignment
typedef half8 half8_any __attribute__((aligned(2)));
typedef float4v float4_any __attribute__((aligned(4)));

// What happens to an element after its rounding to fp16, besides being stored: E = op(C) or
// E = C op X, the consumer of a matmul whose result it is (both are written).
enum : int { EPI_NONE = 0, EPI_EXP, EPI_SILU, EPI_ADD, EPI_MUL, EPI_DIV, EPI_RDIV /* X / C */ };

struct AnyGemm {
  _Float16 const *A, *B;
  _Float16 *C;
  _Float16 const *X;  // second operand of a binary consumer: [batch][m][n]
  _Float16 *E;        // the consumer's result
  int epilogue, epilogue2;  // of the first matrix of the batch; of the others
  int m, n, k;
  int tiles_m, tiles_n;
  int group;       // tile rows that a column of tiles goes down (gemm_tile)
  unsigned total;  // workgroups
  // k in `ksplit` ranges, a workgroup each; with more than one a range's fp32 sums go to
  // partial[range][batch][m][n] and f16_gemm_fold_kernel adds them
  int ksplit, steps_per_range;
  int a_rows;  // from a matrix of A to the next: m
  float *partial;
  // elements from a matrix of the other operands to the next.  Two products of the same A are a batch of two with
  // a_rows = 0 and these as the tensors happen to lie.
  long long b_step, c_step, x_step, e_step;
};
// (two lines of kernel arguments, both asked for at the start: a field of a third, first read on the way out, was 0.1 us)
static_assert(sizeof(AnyGemm) == 128, "two cache lines");

__device__ __forceinline__ float f16_unary_value(bool exp, float x) { return exp ? __expf(x) : x / (1.0f + __expf(-x)); }

__device__ __forceinline__ float epilogue_value(int op, float c, float x) {
  switch (op) {
    case EPI_EXP: return f16_unary_value(true, c);
    case EPI_SILU: return f16_unary_value(false, c);
    case EPI_ADD: return c + x;
    case EPI_MUL: return c * x;
    case EPI_DIV: return c / x;
    default: return x / c;
  }
}

// Drops the first `s` elements of a chunk (0 <= s <= 8): the rest moves to the front, zeros follow.
__device__ __forceinline__ half8 chunk_drop(half8 v, int s) {
  typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
  u64x2 const x = __builtin_bit_cast(u64x2, v);
  int const b = 16 * (s & 3);
  uint64_t const lo = s & 4 ? x.y : x.x, hi = s & 4 ? 0 : x.y;
  u64x2 r = {b ? (lo >> b) | (hi << (64 - b)) : lo, hi >> b};
  if (s >= 8) {
    r = u64x2{0, 0};
  }
  return __builtin_bit_cast(half8, r);
}

// One operand's share of the work of a thread: its 16-byte chunks of a stage of R rows (columns for
// B) x 64 k.  KC: k is contiguous in memory, an LDS row is a matrix row.  Otherwise the row index
// is contiguous, an LDS row is one k, and the MFMA operand comes from a transposing read.
// Everything stays inside the matrix: rows past it re-read its last row, a chunk that would cross
// the end of a row (of k, or of columns) is read from where it ends there and shifted.
template <int R, int NT, bool KC>
struct OperandStage {
  static constexpr int BK = 64, CHUNKS = R * BK / 8, CH = (CHUNKS + NT - 1) / NT;
  static constexpr int LD = KC ? BK + 8 : R + 8;  // halfs
  static constexpr int HALFS = (KC ? R : BK) * LD;
  _Float16 const *base;
  int ld, k, row_of[CH], pos_of[CH];
  uint32_t off[CH];  // bytes from the stage's first element
  int cut[CH];       // elements to drop from the front (row index contiguous: columns past the edge)
  bool ragged;

  __device__ __forceinline__ void init(_Float16 const *matrix, int rows, int row0, int k_, int tid) {
    k = k_;
    ld = KC ? k : rows;
    base = matrix + (KC ? (size_t)row0 * ld : (size_t)row0);
    ragged = !KC && row0 + R > rows && rows % 8 != 0;
#pragma unroll
    for (int i = 0; i < CH; i++) {
      int q = i * NT + tid;
      q = q < CHUNKS ? q : CHUNKS - 1;
      cut[i] = 0;
      if (KC) {
        row_of[i] = q / (BK / 8);
        pos_of[i] = 8 * (q % (BK / 8));
        int const r = row0 + row_of[i] < rows ? row_of[i] : rows - 1 - row0;
        off[i] = 2u * (uint32_t)(r * ld + pos_of[i]);
      } else {
        row_of[i] = q / (R / 8);
        pos_of[i] = 8 * (q % (R / 8));
        int const left = rows - row0 - pos_of[i];
        int const back = left >= 8 ? 0 : 8 - left;
        cut[i] = back < 8 ? back : 0;
        off[i] = 2u * (uint32_t)(row_of[i] * ld + pos_of[i]) - 2u * (uint32_t)back;  // (wraps when negative)
      }
    }
  }
  // (a negative offset happens only left of the stage's first element, never of the matrix's)
  __device__ __forceinline__ half8 fetch(_Float16 const *p, uint32_t o) const {
    return *reinterpret_cast<half8_any const *>(reinterpret_cast<char const *>(p) + (int)o);
  }
  // stage of 64 whole k
  __device__ __forceinline__ void load(half8 (&r)[CH], int stage) const {
    _Float16 const *p = base + (KC ? (size_t)(BK * stage) : (size_t)(BK * stage) * ld);
#pragma unroll
    for (int i = 0; i < CH; i++) {
      r[i] = fetch(p, off[i]);
    }
  }
  // the last stage, of `tail` < 64 k
  __device__ __forceinline__ void load_tail(half8 (&r)[CH], int stage, int tail) const {
    _Float16 const *p = base + (KC ? (size_t)(BK * stage) : (size_t)(BK * stage) * ld);
#pragma unroll
    for (int i = 0; i < CH; i++) {
      if (KC) {
        int const over = pos_of[i] + 8 - tail;  // elements of the chunk past the row's end
        r[i] = fetch(p, off[i] - (over > 0 ? 2u * (uint32_t)over : 0u));
      } else {
        int const over = row_of[i] - (tail - 1);
        r[i] = fetch(p, off[i] - (over > 0 ? 2u * (uint32_t)(over * ld) : 0u));
      }
    }
  }
  __device__ __forceinline__ void mask_tail(half8 (&r)[CH], int tail) const {
#pragma unroll
    for (int i = 0; i < CH; i++) {
      int over = KC ? pos_of[i] + 8 - tail : (row_of[i] < tail ? 0 : 8);
      over = over < 0 ? 0 : over > 8 ? 8 : over;
      if (KC || over == 8) {
        r[i] = chunk_drop(r[i], over);
      }
    }
  }
  __device__ __forceinline__ void store(half8 const (&r)[CH], _Float16 *tile, int tid) const {
#pragma unroll
    for (int i = 0; i < CH; i++) {
      half8 v = r[i];
      if (!KC && ragged) {
        v = chunk_drop(v, cut[i]);
      }
      if (CHUNKS % NT == 0 || i * NT + tid < CHUNKS) {
        *reinterpret_cast<half8 *>(tile + row_of[i] * LD + pos_of[i]) = v;
      }
    }
  }
  // operand of rows r0 .. r0 + 15, k step s of 32: lane (g, c) holds [r0 + c][32 s + 8 g .. + 7]
  __device__ __forceinline__ static half8 operand(_Float16 const *tile, int r0, int s, int lane) {
    int const g = lane / 16, c = lane % 16;
    if (KC) {
      return *reinterpret_cast<half8 const *>(tile + (r0 + c) * LD + 32 * s + 8 * g);
    }
    typedef short short4v __attribute__((ext_vector_type(4)));
    typedef short4v __attribute__((address_space(3))) *lds_p;
    _Float16 const *p = tile + (32 * s + 8 * g + (c >> 2)) * LD + r0 + 4 * (c & 3);
    half4 const lo = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                   (lds_p)(__attribute__((address_space(3))) void *)p));
    half4 const hi = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                   (lds_p)(__attribute__((address_space(3))) void *)(p + 4 * LD)));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

// Which tile, batch and k range: an XCD (one L2) gets consecutive ids; the k ranges of a tile sit next to
// each other, and tiles go down `group` tile rows before they move to the next columns: all of up to 512 rows where B
// is larger than an L2, else four ([300, 2048] . [2048, 5504], five rows of tiles, whose columns a second group would
// fetch again, 15.3 -> 14.1 us, [426, 128] . [128, 2575] 4.1 -> 4.3).
__device__ __forceinline__ void gemm_tile(AnyGemm const &G, int bm, int bn, int &split, int &batch, int &row0, int &col0) {
  unsigned const xcd = blockIdx.x % 8, each = G.total / 8, more = G.total % 8;
  unsigned id = xcd * each + (xcd < more ? xcd : more) + blockIdx.x / 8;
  split = (int)(id % (unsigned)G.ksplit);
  id /= (unsigned)G.ksplit;
  unsigned const tiles = (unsigned)(G.tiles_m * G.tiles_n);
  batch = (int)(id / tiles);
  int const t0 = (int)(id % tiles);
  int const per_group = G.group * G.tiles_n, first_m = G.group * (t0 / per_group);
  int const gsz = (G.tiles_m - first_m) < G.group ? (G.tiles_m - first_m) : G.group;
  row0 = (first_m + (t0 % per_group) % gsz) * bm;
  col0 = (t0 % per_group) / gsz * bn;
}

// The way out of a workgroup's sums: fp16 rows and the consumer's result, or a k range's fp32 sums.  `tile`
// is LDS nothing else uses any more; `owner`: wavefronts that hold sums.
template <int BM, int BN, int TM, int TN, int NT>
__device__ __forceinline__ void gemm_store(AnyGemm const &G, float4v const (&acc)[TM][TN], _Float16 *tile, bool owner, int lane,
                                           int split, int batch, int row0, int col0, int wm0, int wn0) {
  // acc[i][j][e] = C[wm0 + 16 i + lane % 16][wn0 + 16 j + 4 (lane / 16) + e]
  int const g = lane / 16, c = lane % 16;
  if (G.ksplit > 1) {
    if (owner) {
      int const batches = (int)(G.total / (unsigned)(G.ksplit * G.tiles_m * G.tiles_n));
      float *const P = G.partial + ((size_t)split * batches + batch) * (size_t)G.m * G.n;
#pragma unroll
      for (int i = 0; i < TM; i++) {
        int const row = row0 + wm0 + 16 * i + c;
#pragma unroll
        for (int j = 0; j < TN; j++) {
          int const col = col0 + wn0 + 16 * j + 4 * g;
          if (row < G.m && col + 4 <= G.n) {
            *reinterpret_cast<float4_any *>(P + (size_t)row * G.n + col) = acc[i][j];
          } else if (row < G.m) {
#pragma unroll
            for (int e = 0; e < 3; e++) {
              if (col + e < G.n) {
                P[(size_t)row * G.n + col + e] = acc[i][j][e];
              }
            }
          }
        }
      }
    }
    return;
  }
  // ---- out through LDS: rows of 16-byte chunks
  constexpr int LDC = BN + 8;
  if (owner) {
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
      for (int j = 0; j < TN; j++) {
        *reinterpret_cast<half4 *>(tile + (wm0 + 16 * i + c) * LDC + wn0 + 16 * j + 4 * g) =
            __builtin_convertvector(acc[i][j], half4);
      }
    }
  }
  __syncthreads();
  _Float16 *const C = G.C + batch * G.c_step, *const E = G.E + batch * G.e_step;
  _Float16 const *const X = G.X + batch * G.x_step;
  int const epilogue = batch == 0 ? G.epilogue : G.epilogue2;
  for (int e = threadIdx.x; e < BM * (BN / 8); e += NT) {
    int const r = e / (BN / 8), c8 = 8 * (e % (BN / 8)), row = row0 + r, col = col0 + c8;
    if (row < G.m && col < G.n) {
      half8 const v = *reinterpret_cast<half8 const *>(tile + r * LDC + c8);
      size_t const at = (size_t)row * G.n + col;
      if (col + 8 <= G.n) {
        *reinterpret_cast<half8_any *>(C + at) = v;
        if (epilogue != EPI_NONE) {
          half8 x = v;
          if (epilogue >= EPI_ADD) {
            x = *reinterpret_cast<half8_any const *>(X + at);
          }
          half8 y;
#pragma unroll
          for (int u = 0; u < 8; u++) {
            y[u] = static_cast<_Float16>(epilogue_value(epilogue, static_cast<float>(v[u]), static_cast<float>(x[u])));
          }
          *reinterpret_cast<half8_any *>(E + at) = y;
        }
      } else {
#pragma unroll
        for (int u = 0; u < 7; u++) {
          if (col + u < G.n) {
            C[at + u] = v[u];
            if (epilogue != EPI_NONE) {
              float const x = epilogue >= EPI_ADD ? static_cast<float>(X[at + u]) : 0.0f;
              E[at + u] = static_cast<_Float16>(epilogue_value(epilogue, static_cast<float>(v[u]), x));
            }
          }
        }
      }
    }
  }
}

// A workgroup owns a BM x BN tile of C and a range of k.  Its KG groups of wavefronts (WM x WN of the
// tile per wavefront) take a part of the range each and add their sums up in LDS at the end: with few
// tiles that is what keeps a compute unit busy.  A stage of 64 k goes global -> registers (PF stages
// ahead) -> LDS (two buffers, one barrier a stage) -> MFMA operands.  Registers rather than direct
// loads to LDS in between, because that is where a chunk of an odd-length row can be shifted and
// masked.  The partial stage at the end of k comes FIRST, so that the loop itself has no conditions
// around its loads and every wait can leave the newest stage in flight.
//
// What bounds it: launch and the latency of a stage (0.24 us) for small products, the vector cache
// and LDS traffic of a stage beside its matrix instructions for large ones (64 x 64: 384 cycles of
// LDS against 128 of MFMA).  Before, odd sizes went element by element through f16_matmul_kernel and
// row-major weights through a transposed copy: [8, 500, 1000] . [1000, 64] 67 -> 6.4 us,
// [300, 2048] . [2048, 5504] row-major 39 -> 20 us, [100, 320] . [320, 755] 46 -> 4.2 us,
// [1024, 2048] . [2048, 5504] 42 us (550 TFLOP/s).
template <int BM, int BN, int WM, int WN, int KG, bool A_KC, bool B_KC, int PF = 2>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN) * KG) void f16_gemm_any_kernel(AnyGemm const G) {
  constexpr int NTG = 64 * (BM / WM) * (BN / WN), NT = NTG * KG;
  constexpr int TM = WM / 16, TN = WN / 16;
  using SA = OperandStage<BM, NTG, A_KC>;
  using SB = OperandStage<BN, NTG, B_KC>;
  constexpr int BUF = SA::HALFS + SB::HALFS;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int const kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NTG);
  int const tid = threadIdx.x % NTG, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  _Float16 *const bufs = reinterpret_cast<_Float16 *>(lds) + kg * 2 * BUF;

  int split, batch, row0, col0;
  gemm_tile(G, BM, BN, split, batch, row0, col0);

  SA sa;
  SB sb;
  sa.init(G.A + (size_t)batch * G.a_rows * G.k, G.m, row0, G.k, tid);
  sb.init(G.B + batch * G.b_step, G.n, col0, G.k, tid);

  // This group's stages: whole stages [first, first + own) and, in the last range, the tail.
  int const whole = G.k / 64, tail = G.k % 64, ranges = G.ksplit * KG, range = split * KG + kg;
  int const first = range * G.steps_per_range < whole ? range * G.steps_per_range : whole;
  int const own = (whole - first) < G.steps_per_range ? (whole - first) : G.steps_per_range;
  int const lead = tail != 0 && range == ranges - 1 ? 1 : 0, T = own + lead;
  // (all groups of a workgroup meet at its barriers equally often)
  int const steps = KG == 1 ? T : G.steps_per_range + (tail != 0 ? 1 : 0);

  float4v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
      acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  half8 ra[PF][SA::CH], rb[PF][SB::CH];
  auto load = [&](int slot, int t) {  // (stages past this group's own re-read one: never multiplied)
    int const s = first + t - lead < whole - 1 ? first + t - lead : whole - 1;
    sa.load(ra[slot], s);
    sb.load(rb[slot], s);
  };
  auto store = [&](int slot, int t) {
    _Float16 *const buf = bufs + (t & 1) * BUF;
    sa.store(ra[slot], buf, tid);
    sb.store(rb[slot], buf + SA::HALFS, tid);
  };
  int const wm0 = (wave / (BN / WN)) * WM, wn0 = (wave % (BN / WN)) * WN;
  struct Operands {
    half8 a[TM], b[TN];
  };
  auto read = [&](Operands &x, int t, int s) {
    _Float16 const *const buf = bufs + (t & 1) * BUF;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      x.a[i] = SA::operand(buf, wm0 + 16 * i, s, lane);
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      x.b[j] = SB::operand(buf + SA::HALFS, wn0 + 16 * j, s, lane);
    }
  };
  auto multiply = [&](Operands const &x, int t) {
    if (KG == 1 || t < T) {
#pragma unroll
      for (int i = 0; i < TM; i++) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.b[j], x.a[i], acc[i][j], 0, 0, 0);
        }
      }
    }
  };
  if (steps > 0) {
    if (lead) {
      sa.load_tail(ra[0], whole, tail);
      sb.load_tail(rb[0], whole, tail);
    } else if (whole > 0) {
      load(0, 0);
    }
#pragma unroll
    for (int u = 1; u < PF; u++) {
      if (steps > u) {
        load(u, u);
      }
    }
    if (lead) {
      sa.mask_tail(ra[0], tail);
      sb.mask_tail(rb[0], tail);
    }
    store(0, 0);
    __syncthreads();
    // Skewed by half a stage: every batch of operand reads is followed by the multiplications of
    // the batch before it.
    Operands x0, x1;
    read(x0, 0, 0);
    int t = 0;
    for (; t + 2 * PF - 1 < steps; t += PF) {
#pragma unroll
      for (int u = 0; u < PF; u++) {
        load(u, t + u + PF);
        read(x1, t + u, 1);
        multiply(x0, t + u);
        store((u + 1) % PF, t + u + 1);
        __syncthreads();
        read(x0, t + u + 1, 0);
        multiply(x1, t + u);
      }
    }
#pragma unroll
    for (int u = 0; u < 2 * PF - 1; u++) {  // the last stages
      if (t + u < steps) {
        if (u < PF - 1 && t + u + PF < steps) {
          load(u, t + u + PF);
        }
        read(x1, t + u, 1);
        multiply(x0, t + u);
        if (t + u + 1 < steps) {
          store((u + 1) % PF, t + u + 1);
        }
        __syncthreads();
        if (t + u + 1 < steps) {
          read(x0, t + u + 1, 0);
        }
        multiply(x1, t + u);
      }
    }
  }

  // ---- the groups' sums, in group order
  if (KG > 1) {
    float4v *const sums = reinterpret_cast<float4v *>(lds);  // [KG - 1][TM * TN][NTG]
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < TM; i++) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
          sums[((kg - 1) * TM * TN + i * TN + j) * NTG + tid] = acc[i][j];
        }
      }
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int u = 1; u < KG; u++) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
#pragma unroll
          for (int j = 0; j < TN; j++) {
            float4v const v = sums[((u - 1) * TM * TN + i * TN + j) * NTG + tid];
#pragma unroll
            for (int e = 0; e < 4; e++) {
              acc[i][j][e] += v[e];
            }
          }
        }
      }
    }
  }
  gemm_store<BM, BN, TM, TN, NT>(G, acc, reinterpret_cast<_Float16 *>(lds) + (KG - 1) * TM * TN * NTG * 8, kg == 0, lane, split, batch,
                                 row0, col0, wm0, wn0);
}

template <int BM, int BN, int WM, int WN, int KG, bool A_KC, bool B_KC>
constexpr int any_gemm_lds() {
  constexpr int NTG = 64 * (BM / WM) * (BN / WN);
  constexpr int stages = KG * 2 * (OperandStage<BM, NTG, A_KC>::HALFS + OperandStage<BN, NTG, B_KC>::HALFS) * 2;
  constexpr int out = (KG - 1) * (WM / 16) * (WN / 16) * NTG * 16 + BM * (BN + 8) * 2;
  return stages > out ? stages : out;
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ uint32_t gemm_lds_address(void const *p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void const *)p;
}
__device__ __forceinline__ void gemm_dma16(_Float16 const *gbase, uint32_t lane_byte_offset, uint32_t lds_wave_base) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds_wave_base)), "v"(lane_byte_offset), "s"(gbase)
               : "m0", "memory");
}
template <int N>
__device__ __forceinline__ void gemm_wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
#pragma clang diagnostic pop

// Where the 16-byte chunk q of row r of an LDS tile lies in its row.  LDS has 64 banks, 256 bytes a cycle, and
// serves a 16-byte read in the lane groups {0-3, 12-15, 20-23, 24-27} and so on, an 8-byte one 32 lanes at a
// time; with these every operand read below is free of bank conflicts (measured over 16 wavefronts: 236 - 240
// bytes a cycle; rows of 64 bytes turned by r / 4 127; transposing reads 190, turned by r / 2 % 4 121).
__device__ __forceinline__ int turned_k64(int r, int q) { return q ^ (r / 2 % 8); }     // rows of 64 k
__device__ __forceinline__ int turned_k32(int r, int q) { return q ^ (-(r / 4) & 3); }  // rows of 32 k
template <int R>  // a row is one k of R = 64 or 128 columns, read transposing
__device__ __forceinline__ int turned_columns(int r, int q) {
  static_assert(R == 64 || R == 128, "columns of a tile");
  return q ^ (2 * (R == 64 ? r / 2 % 2 + 2 * (r / 8 % 2) : r % 4 + 4 * (r / 8 % 2)));
}

// Products whose rows are whole 16-byte chunks and whose k is whole stages of 64: f16_gemm_any_kernel's
// tiles and k ranges, but a stage goes to LDS directly (global_load_lds_dwordx4), without the registers and
// the LDS stores of the way through them; a ring of three stages, two in flight.  A direct load writes its
// 64 chunks in lane order: a lane fetches the chunk that belongs in its place.
//
// What bounds it: the 35 bytes a cycle that a compute unit gets from its caches (64 x 64 x 64: 470 cycles,
// of matrix instructions 128), whatever the number of stages in flight; so a wide tile where there are
// tiles enough.  f16_gemm_any_kernel and here: [300, 2048] . [2048, 5504] row-major 20.1 and 16.2 us,
// [1024, 2048] . [2048, 5504] 39.6 and 35.4, [2048, 2048] . [2048, 2048] 28.9 and 24.4 (704 TFLOP/s).
template <int R, int NT, bool KC>
struct DirectStage {
  static constexpr int BK = 64, CH = R * BK / 8 / NT, LD = KC ? BK : R, HALFS = R * BK;
  static_assert(R * BK / 8 % NT == 0, "a stage splits evenly over the threads");
  _Float16 const *base;
  size_t step;       // elements from a stage to the next
  uint32_t off[CH];  // bytes from the stage's first element

  __device__ __forceinline__ static int turned(int r, int q) {
    if constexpr (KC) {
      return turned_k64(r, q);
    } else {
      return turned_columns<R>(r, q);
    }
  }

  // (rows and chunks past the matrix re-read its last ones)
  __device__ __forceinline__ void init(_Float16 const *matrix, int rows, int row0, int k, int tid) {
    base = matrix + (KC ? (size_t)row0 * k : (size_t)row0);
    step = KC ? (size_t)BK : (size_t)BK * rows;
#pragma unroll
    for (int i = 0; i < CH; i++) {
      int const p = i * NT + tid;
      if (KC) {
        int const r = p / 8, rr = row0 + r < rows ? r : rows - 1 - row0;
        off[i] = 2u * (uint32_t)(rr * k + 8 * turned(r, p % 8));
      } else {
        int const r = p / (R / 8), q = 8 * turned(r, p % (R / 8));
        off[i] = 2u * (uint32_t)(r * rows + (row0 + q + 8 <= rows ? q : rows - 8 - row0));
      }
    }
  }
  __device__ __forceinline__ void issue(int stage, uint32_t lds, int wave) const {
    _Float16 const *const p = base + (size_t)stage * step;
#pragma unroll
    for (int i = 0; i < CH; i++) {
      gemm_dma16(p, off[i], lds + 16u * (uint32_t)(i * NT + wave * 64));
    }
  }
  // operand of rows r0 .. r0 + 15, k step s of 32: lane (g, c) holds [r0 + c][32 s + 8 g .. + 7]
  __device__ __forceinline__ static half8 operand(_Float16 const *tile, int r0, int s, int lane) {
    int const g = lane / 16, c = lane % 16;
    if (KC) {
      return *reinterpret_cast<half8 const *>(tile + (r0 + c) * LD + 8 * turned(c, 4 * s + g));  // (16 divides r0)
    }
    typedef short short4v __attribute__((ext_vector_type(4)));
    typedef short4v __attribute__((address_space(3))) *lds_p;
    int const r = 32 * s + 8 * g + (c >> 2), q = r0 / 8 + ((c & 3) >> 1), in = 4 * (c & 1);
    _Float16 const *const p = tile + r * LD + 8 * turned(r, q) + in, *const p4 = tile + (r + 4) * LD + 8 * turned(r + 4, q) + in;
    half4 const lo = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                   (lds_p)(__attribute__((address_space(3))) void *)p));
    half4 const hi = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                   (lds_p)(__attribute__((address_space(3))) void *)p4));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

constexpr int kDirectRing = 3;

// Both of two products of one A (TWO): half of a tile's columns are of the second, a wavefront's all
// of one, and each half leaves as a product by itself does.  A is fetched once, and a launch of 64 x 64 + 64 or
// 128 + 128 columns has less to wait for than two: [300, 2048] . [2048, 5504] twice 26.1 us, one by one 2 x 17.8.  What
// bounds it: the LDS traffic of a stage, 1100 cycles of 1600 with 128 columns of each.
template <int BM, int BN, int WM, int WN, bool B_KC, bool TWO = false>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN)) void f16_gemm_direct_kernel(AnyGemm const G) {
  constexpr int NT = 64 * (BM / WM) * (BN / WN), TM = WM / 16, TN = WN / 16, COLS = TWO ? BN / 2 : BN;
  static_assert(COLS % WN == 0, "a wavefront has columns of one product");
  using SA = DirectStage<BM, NT, true>;
  using SB = DirectStage<COLS, NT, B_KC>;
  constexpr int STAGE = SA::HALFS + (TWO ? 2 : 1) * SB::HALFS, LPS = SA::CH + (TWO ? 2 : 1) * SB::CH;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  _Float16 *const ring = reinterpret_cast<_Float16 *>(lds);
  int const tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);

  int split, batch, row0, col0;
  gemm_tile(G, BM, COLS, split, batch, row0, col0);
  SA sa;
  SB sb, sb2;
  sa.init(G.A + (size_t)batch * G.a_rows * G.k, G.m, row0, G.k, tid);
  sb.init(G.B + batch * G.b_step, G.n, col0, G.k, tid);
  if (TWO) {
    sb2.init(G.B + G.b_step, G.n, col0, G.k, tid);
  }
  int const whole = G.k / 64, first = split * G.steps_per_range < whole ? split * G.steps_per_range : whole;
  int const T = (whole - first) < G.steps_per_range ? (whole - first) : G.steps_per_range;
  int const wm0 = (wave / (BN / WN)) * WM, col = (wave % (BN / WN)) * WN, second = TWO ? col / COLS : 0, wn0 = col - second * COLS;

  float4v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
      acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  uint32_t const ring_at = gemm_lds_address(ring);
  auto issue = [&](int t, int slot) {
    uint32_t const at = ring_at + 2u * (uint32_t)(slot * STAGE);
    sa.issue(first + t, at, wave);
    sb.issue(first + t, at + 2u * (uint32_t)SA::HALFS, wave);
    if (TWO) {
      sb2.issue(first + t, at + 2u * (uint32_t)(SA::HALFS + SB::HALFS), wave);
    }
  };
  struct Operands {
    half8 a[TM], b[TN];
  };
  auto read = [&](Operands &x, int slot, int s) {
    _Float16 const *const buf = ring + slot * STAGE;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      x.a[i] = SA::operand(buf, wm0 + 16 * i, s, lane);
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      x.b[j] = SB::operand(buf + SA::HALFS + second * SB::HALFS, wn0 + 16 * j, s, lane);
    }
  };
  auto multiply = [&](Operands const &x) {
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
      for (int j = 0; j < TN; j++) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.b[j], x.a[i], acc[i][j], 0, 0, 0);
      }
    }
  };
  // stage t has landed (this wavefront's share) when at most stage t + 1 is outstanding
  auto landed = [&](int t) {
    if (t + 1 < T) {
      gemm_wait_vm<LPS>();
    } else {
      gemm_wait_vm<0>();
    }
  };
  // Skewed by half a stage: every batch of operand reads is followed by the multiplications of the batch
  // before it.  The last stage stands behind the loop: with a condition around the reads of the next one, the
  // multiplications behind it wait for those reads too (the compiler's count of LDS reads in flight is the
  // least of the two ways there), and reading and multiplying take turns ([300, 2048] . [2048, 5504] row-major
  // 18.5 -> 17.6 us, [1024, 2048] . [2048, 5504] 39.7 -> 38.0).
  if (T > 0) {
    issue(0, 0);
    if (T > 1) {
      issue(1, 1);
    }
    landed(0);
    __syncthreads();
    if (T > 2) {
      issue(2, 2);
    }
    Operands x0, x1;
    read(x0, 0, 0);
    int slot = 0;
    for (int t = 0; t + 1 < T; t++) {
      int const next = slot + 1 < kDirectRing ? slot + 1 : 0;
      read(x1, slot, 1);
      multiply(x0);
      landed(t + 1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wavefront's reads of stage t are in registers
      __syncthreads();                                    // stage t + 1 is there, stage t is free
      if (t + 3 < T) {
        issue(t + 3, slot);
      }
      read(x0, next, 0);
      multiply(x1);
      slot = next;
    }
    read(x1, slot, 1);
    multiply(x0);
    multiply(x1);
    __syncthreads();
  }
  gemm_store<BM, COLS, TM, TN, NT>(G, acc, ring, second == 0, lane, split, batch, row0, col0, wm0, wn0);
  if (TWO) {  // (a thread stores the same elements of both: a consumer may read the first's)
    __syncthreads();
    gemm_store<BM, COLS, TM, TN, NT>(G, acc, ring, second == 1, lane, split, 1, row0, col0, wm0, wn0);
  }
}

template <int BM, int BN>
constexpr int direct_gemm_lds() {
  constexpr int ring = kDirectRing * (BM + BN) * 128, out = BM * (BN + 8) * 2;
  return ring > out ? ring : out;
}

// Products whose rows are whole 16-byte chunks and whose k is whole steps of 32.  A workgroup's tile is as
// before, but each of its four wavefronts has ALL of the tile and every fourth step of k: an element of an
// operand then leaves LDS once per workgroup rather than once per wavefront that shares its row, and a
// wavefront needs no barrier until the four sums are added up.  A step goes to the wavefront's own ring in
// LDS by direct loads (global_load_lds_dwordx4), RING - 1 of them in flight while one is multiplied from
// registers.
//
// What bounds it: as above; the operand reads and barriers it saves count where the tile is small and the
// steps of a workgroup are a chain: 0.14 us for 64 k of a 16 x 64 tile (f16_gemm_any_kernel: 0.24).
// [16, 2048] . [2048, 5504] 10.2 -> 7.5 us, [96, 512] . [512, 1024] 5.5 -> 4.7, [512, 4096] . [4096, 512]
// 13.0 -> 12.1.
template <int R, bool KC>
struct WaveStage {
  static constexpr int BK = 32, CH = R * BK / 8 / 64, LD = KC ? BK : R, HALFS = R * BK;
  _Float16 const *base;
  size_t step;       // elements from a step of k to the next
  uint32_t off[CH];  // bytes from the step's first element

  __device__ __forceinline__ static int turned(int r, int q) {
    if constexpr (KC) {
      return turned_k32(r, q);
    } else {
      return turned_columns<R>(r, q);
    }
  }

  // (rows and chunks past the matrix re-read its last ones)
  __device__ __forceinline__ void init(_Float16 const *matrix, int rows, int row0, int k, int lane) {
    base = matrix + (KC ? (size_t)row0 * k : (size_t)row0);
    step = KC ? (size_t)BK : (size_t)BK * rows;
#pragma unroll
    for (int i = 0; i < CH; i++) {
      int const p = i * 64 + lane;
      if (KC) {
        int const r = p / 4, rr = row0 + r < rows ? r : rows - 1 - row0;
        off[i] = 2u * (uint32_t)(rr * k + 8 * turned(r, p % 4));
      } else {
        int const r = p / (R / 8), q = 8 * turned(r, p % (R / 8));
        off[i] = 2u * (uint32_t)(r * rows + (row0 + q + 8 <= rows ? q : rows - 8 - row0));
      }
    }
  }
  __device__ __forceinline__ void issue(int t, uint32_t lds) const {
    _Float16 const *const p = base + (size_t)t * step;
#pragma unroll
    for (int i = 0; i < CH; i++) {
      gemm_dma16(p, off[i], lds + 1024u * (uint32_t)i);
    }
  }
  // operand of rows r0 .. r0 + 15: lane (g, c) holds [r0 + c][8 g .. + 7]
  __device__ __forceinline__ static half8 operand(_Float16 const *tile, int r0, int lane) {
    int const g = lane / 16, c = lane % 16;
    if (KC) {
      return *reinterpret_cast<half8 const *>(tile + (r0 + c) * LD + 8 * turned(c, g));  // (16 divides r0)
    }
    typedef short short4v __attribute__((ext_vector_type(4)));
    typedef short4v __attribute__((address_space(3))) *lds_p;
    int const r = 8 * g + (c >> 2), q = r0 / 8 + ((c & 3) >> 1), in = 4 * (c & 1);
    _Float16 const *const p = tile + r * LD + 8 * turned(r, q) + in, *const p4 = tile + (r + 4) * LD + 8 * turned(r + 4, q) + in;
    half4 const lo = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                   (lds_p)(__attribute__((address_space(3))) void *)p));
    half4 const hi = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                   (lds_p)(__attribute__((address_space(3))) void *)p4));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

template <int BM, int BN, int RING, bool B_KC>
__global__ __launch_bounds__(256) void f16_gemm_waves_kernel(AnyGemm const G) {
  constexpr int TM = BM / 16, TN = BN / 16, TQ = TN / 4;
  using SA = WaveStage<BM, true>;
  using SB = WaveStage<BN, B_KC>;
  constexpr int STEP = SA::HALFS + SB::HALFS, LPS = SA::CH + SB::CH;
  static_assert(RING >= 3 && RING <= 4 && (RING - 1) * LPS < 64, "waits for two or three steps");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int const lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  _Float16 *const ring = reinterpret_cast<_Float16 *>(lds) + wave * RING * STEP;

  int split, batch, row0, col0;
  gemm_tile(G, BM, BN, split, batch, row0, col0);
  SA sa;
  SB sb;
  sa.init(G.A + (size_t)batch * G.a_rows * G.k, G.m, row0, G.k, lane);
  sb.init(G.B + batch * G.b_step, G.n, col0, G.k, lane);
  // this range's steps [first, last); the wavefront's are first + wave, + 4, ..
  int const all = G.k / 32, first = split * G.steps_per_range < all ? split * G.steps_per_range : all;
  int const last = all - first < G.steps_per_range ? all : first + G.steps_per_range;
  int const T = (last - first - wave + 3) / 4;

  float4v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
      acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  uint32_t const ring_at = gemm_lds_address(ring);
  auto issue = [&](int t, int slot) {
    uint32_t const at = ring_at + 2u * (uint32_t)(slot * STEP);
    sa.issue(first + wave + 4 * t, at);
    sb.issue(first + wave + 4 * t, at + 2u * (uint32_t)SA::HALFS);
  };
  struct Operands {
    half8 a[TM], b[TN];
  };
  auto read = [&](Operands &x, int slot) {
    _Float16 const *const buf = ring + slot * STEP;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      x.a[i] = SA::operand(buf, 16 * i, lane);
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      x.b[j] = SB::operand(buf + SA::HALFS, 16 * j, lane);
    }
  };
  auto multiply = [&](Operands const &x) {
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
      for (int j = 0; j < TN; j++) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.b[j], x.a[i], acc[i][j], 0, 0, 0);
      }
    }
  };
  // step t has landed when at most the RING - 1 steps after it are outstanding
  auto landed = [&](int t) {
    int const later = T - 1 - t;
    if (later >= RING - 1) {
      gemm_wait_vm<(RING - 1) * LPS>();
    } else if (RING > 3 && later >= 2) {
      gemm_wait_vm<2 * LPS>();
    } else if (later >= 1) {
      gemm_wait_vm<LPS>();
    } else {
      gemm_wait_vm<0>();
    }
  };
#pragma unroll
  for (int t = 0; t < RING; t++) {
    if (t < T) {
      issue(t, t);
    }
  }
  // one step: its operands are in registers; the next one's are read and its slot filled again
  int slot = 0;
  auto advance = [&](Operands &next, Operands const &now, int t) {
    slot = slot + 1 < RING ? slot + 1 : 0;
    landed(t + 1);
    read(next, slot);
    multiply(now);
    if (t + 1 + RING < T) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the reads have left the slot)
      issue(t + 1 + RING, slot);
    }
  };
  if (T > 0) {
    Operands x0, x1;
    landed(0);
    read(x0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (RING < T) {
      issue(RING, 0);
    }
    int t = 0;  // (the last step or two behind the loop: see f16_gemm_direct_kernel)
    for (; t + 2 < T; t += 2) {
      advance(x1, x0, t);
      advance(x0, x1, t + 1);
    }
    if (t + 1 < T) {
      advance(x1, x0, t);
      multiply(x1);
    } else {
      multiply(x0);
    }
  }
  // ---- the wavefronts' sums, in wavefront order: each adds up a quarter of the columns
  float4v *const sums = reinterpret_cast<float4v *>(lds);  // [4 wavefronts][TM][TN][64]
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
      sums[((wave * TM + i) * TN + j) * 64 + lane] = acc[i][j];
    }
  }
  __syncthreads();
  float4v quarter[TM][TQ];
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TQ; j++) {
      float4v v = sums[(i * TN + wave * TQ + j) * 64 + lane];
#pragma unroll
      for (int w = 1; w < 4; w++) {
        float4v const x = sums[((w * TM + i) * TN + wave * TQ + j) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          v[e] += x[e];
        }
      }
      quarter[i][j] = v;
    }
  }
  __syncthreads();
  gemm_store<BM, BN, TM, TQ, 256>(G, quarter, reinterpret_cast<_Float16 *>(lds), true, lane, split, batch, row0, col0, 0,
                                  wave * TQ * 16);
}

template <int BM, int BN, int RING>
constexpr int waves_gemm_lds() {
  constexpr int ring = 4 * RING * (BM + BN) * 64, sums = 4 * BM * BN * 4;
  return ring > sums ? ring : sums;
}

}  // namespace mi355
