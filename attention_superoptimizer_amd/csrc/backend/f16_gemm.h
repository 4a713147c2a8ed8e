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
  int epilogue;
  int m, n, k;
  int tiles_m, tiles_n, tiles_per_batch;
  unsigned total;  // workgroups
  // k in `ksplit` ranges, a workgroup each; with more than one a range's fp32 sums go to
  // partial[range][batch][m][n] and f16_gemm_fold_kernel adds them
  int ksplit, steps_per_range;
  float *partial;
};

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
  static constexpr int LD = KC ? BK + 8 : R + 8;  // halfs; both strides spread a read over all banks
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

// A workgroup owns a BM x BN tile of C and a range of k.  Its KG groups of wavefronts (WM x WN of the
// tile per wavefront) take a part of the range each and add their sums up in LDS at the end: with few
// tiles that is what keeps a compute unit busy.  A stage of 64 k goes global -> registers (two stages
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
template <int BM, int BN, int WM, int WN, int KG, bool A_KC, bool B_KC>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN) * KG) void f16_gemm_any_kernel(AnyGemm const G) {
  constexpr int NTG = 64 * (BM / WM) * (BN / WN), NT = NTG * KG, PF = 2;
  constexpr int TM = WM / 16, TN = WN / 16;
  using SA = OperandStage<BM, NTG, A_KC>;
  using SB = OperandStage<BN, NTG, B_KC>;
  constexpr int BUF = SA::HALFS + SB::HALFS;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int const kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NTG);
  int const tid = threadIdx.x % NTG, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  _Float16 *const bufs = reinterpret_cast<_Float16 *>(lds) + kg * 2 * BUF;

  // Which tile: an XCD (one L2) gets consecutive ids; the k ranges of a tile sit next to each
  // other, and tiles go down four tile rows before they move to the next columns.
  unsigned const xcd = blockIdx.x % 8, each = G.total / 8, more = G.total % 8;
  unsigned id = xcd * each + (xcd < more ? xcd : more) + blockIdx.x / 8;
  int const split = (int)(id % (unsigned)G.ksplit);
  id /= (unsigned)G.ksplit;
  int const batch = (int)(id / (unsigned)G.tiles_per_batch), t0 = (int)(id % (unsigned)G.tiles_per_batch);
  int const per_group = 4 * G.tiles_n, first_m = 4 * (t0 / per_group);
  int const gsz = (G.tiles_m - first_m) < 4 ? (G.tiles_m - first_m) : 4;
  int const row0 = (first_m + (t0 % per_group) % gsz) * BM, col0 = (t0 % per_group) / gsz * BN;

  SA sa;
  SB sb;
  sa.init(G.A + (size_t)batch * G.m * G.k, G.m, row0, G.k, tid);
  sb.init(G.B + (size_t)batch * G.k * G.n, G.n, col0, G.k, tid);

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
    if (steps > 1) {
      load(1, 1);
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
    for (; t + PF + 1 < steps; t += 2) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
        load(u, t + u + PF);
        read(x1, t + u, 1);
        multiply(x0, t + u);
        store(1 - u, t + u + 1);
        __syncthreads();
        read(x0, t + u + 1, 0);
        multiply(x1, t + u);
      }
    }
#pragma unroll
    for (int u = 0; u < 3; u++) {  // the last one to three stages
      if (t + u < steps) {
        if (u == 0 && t + PF < steps) {
          load(0, t + PF);
        }
        read(x1, t + u, 1);
        multiply(x0, t + u);
        if (t + u + 1 < steps) {
          store((u + 1) % 2, t + u + 1);
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
  // acc[i][j][e] = C[wm0 + 16 i + lane % 16][wn0 + 16 j + 4 (lane / 16) + e]
  int const g = lane / 16, c = lane % 16;
  if (G.ksplit > 1) {
    if (kg == 0) {
      int const batches = (int)(G.total / (unsigned)(G.ksplit * G.tiles_per_batch));
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
  _Float16 *const tile = reinterpret_cast<_Float16 *>(lds) + (KG - 1) * TM * TN * NTG * 8;
  if (kg == 0) {
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
  size_t const matrix = (size_t)batch * G.m * G.n;
  for (int e = threadIdx.x; e < BM * (BN / 8); e += NT) {
    int const r = e / (BN / 8), c8 = 8 * (e % (BN / 8)), row = row0 + r, col = col0 + c8;
    if (row < G.m && col < G.n) {
      half8 const v = *reinterpret_cast<half8 const *>(tile + r * LDC + c8);
      size_t const at = matrix + (size_t)row * G.n + col;
      if (col + 8 <= G.n) {
        *reinterpret_cast<half8_any *>(G.C + at) = v;
        if (G.epilogue != EPI_NONE) {
          half8 x = v;
          if (G.epilogue >= EPI_ADD) {
            x = *reinterpret_cast<half8_any const *>(G.X + at);
          }
          half8 y;
#pragma unroll
          for (int u = 0; u < 8; u++) {
            y[u] = static_cast<_Float16>(epilogue_value(G.epilogue, static_cast<float>(v[u]), static_cast<float>(x[u])));
          }
          *reinterpret_cast<half8_any *>(G.E + at) = y;
        }
      } else {
#pragma unroll
        for (int u = 0; u < 7; u++) {
          if (col + u < G.n) {
            G.C[at + u] = v[u];
            if (G.epilogue != EPI_NONE) {
              float const x = G.epilogue >= EPI_ADD ? static_cast<float>(G.X[at + u]) : 0.0f;
              G.E[at + u] = static_cast<_Float16>(epilogue_value(G.epilogue, static_cast<float>(v[u]), x));
            }
          }
        }
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, int KG, bool A_KC, bool B_KC>
constexpr int any_gemm_lds() {
  constexpr int NTG = 64 * (BM / WM) * (BN / WN);
  constexpr int stages = KG * 2 * (OperandStage<BM, NTG, A_KC>::HALFS + OperandStage<BN, NTG, B_KC>::HALFS) * 2;
  constexpr int out = (KG - 1) * (WM / 16) * (WN / 16) * NTG * 16 + BM * (BN + 8) * 2;
  return stages > out ? stages : out;
}

}  // namespace mi355
