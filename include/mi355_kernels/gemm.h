// Device code of the fused skinny-GEMM kernels (gemm_fused_kernel and its fold gemm_combine_kernel,
// gemm_lanes_kernel) and the parameter blocks they take.  Header-only and free of host state:
// the backend library (gemm_fused.hip recognises the family, chooses kernel and launch shape) and
// the programs Graph::generate_hip_program writes both instantiate these templates.  They are
// what an emitted program of this backend runs where the reference emits Triton source
// (src/kernel/triton_code_gen.cc:84-352).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernarg.h"

namespace mi355 {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));

enum { PRO_NONE = 0, PRO_EXP = 1, PRO_SILU = 2, PRO_SILU_MUL = 3 };

// Where a tile of a device tensor starts: the element offset is linear in the block
// coordinates and the for-loop iteration, so the host folds the plan's row / column / batch
// strides into one stride per coordinate (a few scalar multiplies per tile address).
struct GTile {
  void const *ptr;
  int lin[4];  // elements per step of bx, by, bz and of the iteration (the host takes a plan on
               // these kernels only when every tile origin fits 31 bits: the parameter block
               // of the one-launch kernel then fits the scalar registers, and a tile address is
               // four 32-bit multiplies)
  int d_cols;  // row stride of the tensor
};

struct GemmParams {
  GTile a0, a1;      // activation-side tiles [M][KT] (a1: second operand of the gate form)
  GTile b0, b1;      // weight tiles [KT][64]
  GTile la, lb;      // lora: A tile [KT][r], B tile [r][64] (loop invariant), ranks r of 8, 16 and 32
  GTile o0, o1;      // outputs
  int M, KT;         // rows of the activation tile, k extent of one iteration
  int forloop_range;
  int ksplit;        // workgroups per logical block
  _Float16 *scratch; // [blocks][forloop_range][NB][M][64] fp16 product tiles (ksplit > 1)
  _Float16 *gate;    // two weights: where silu(first) * second goes as well, in the places of the first result; or null
};

__device__ __forceinline__ long long gtile_offset(GTile const &t, int bx, int by, int bz, int it) {
  return (long long)(bx * t.lin[0] + by * t.lin[1] + bz * t.lin[2] + it * t.lin[3]);
}

// 16-byte chunk `chunk` of row `row` in a swizzled LDS tile with LD halfs per row.
// `mask` = (chunks per row - 1) & 7 keeps the XOR inside the row for narrow tiles.
__device__ __forceinline__ int sw_chunk(int row, int chunk, int LD, int mask) {
  return row * LD + ((chunk ^ ((row ^ (row >> 3)) & mask)) << 3);
}

__device__ __forceinline__ float prologue(int pro, float x) {
  if (pro == PRO_EXP) {
    return __expf(x);
  }
  // x / (1 + exp(-x)): the quotient by a reciprocal, one correction, infinities and NaN as a division has
  // them.  Half the instructions of the full division, and for every fp16 x its result.
  float const d = 1.0f + __expf(-x), r = __builtin_amdgcn_rcpf(d), q = x * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, x), r, q), d, x);
}

// The prologue silu(g) * u, with the roundings of the operators it is made of.
__device__ __forceinline__ _Float16 gate_value(_Float16 g, _Float16 u) {
  _Float16 const silu = static_cast<_Float16>(prologue(PRO_SILU, static_cast<float>(g)));
  return static_cast<_Float16>(static_cast<float>(silu) * static_cast<float>(u));
}

// Transposing stage of a [R][C] tile (C contiguous, row stride ld) into dst[C][R]
// (swizzled, R halfs per row).  All loads first, then the register transposes and
// the LDS writes.  PPT = patches per thread (compile-time bound).
template <int PPT>
__device__ __forceinline__ void stage_weight(_Float16 const *__restrict__ src, int ld, int R, int C,
                                             _Float16 *__restrict__ dst, int tid, int nthreads) {
  int const cblocks = C / 8, patches = (R / 4) * cblocks;
  int const mask = ((R / 8) - 1) & 7;
  uint4v x[PPT][4];
#pragma unroll
  for (int i = 0; i < PPT; i++) {
    int p = tid + i * nthreads;
    if (p < patches) {
      int cb = p % cblocks, rb = p / cblocks;
      _Float16 const *s = src + (long long)(4 * rb) * ld + 8 * cb;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        x[i][j] = *reinterpret_cast<uint4v const *>(s + (long long)j * ld);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < PPT; i++) {
    int p = tid + i * nthreads;
    if (p < patches) {
      int cb = p % cblocks, rb = p / cblocks;
#pragma unroll
      for (int w = 0; w < 4; w++) {
        uint2v even, odd;
        even.x = (x[i][0][w] & 0xffffu) | (x[i][1][w] << 16);
        even.y = (x[i][2][w] & 0xffffu) | (x[i][3][w] << 16);
        odd.x = (x[i][0][w] >> 16) | (x[i][1][w] & 0xffff0000u);
        odd.y = (x[i][2][w] >> 16) | (x[i][3][w] & 0xffff0000u);
        int row = 8 * cb + 2 * w;
        *reinterpret_cast<uint2v *>(dst + sw_chunk(row, rb >> 1, R, mask) + (rb & 1) * 4) = even;
        *reinterpret_cast<uint2v *>(dst + sw_chunk(row + 1, rb >> 1, R, mask) + (rb & 1) * 4) = odd;
      }
    }
  }
}

// The two halves of stage_weight for tiles that are prefetched: the global loads of the
// next iteration's tile are issued before the current one is multiplied and the
// register transposes / LDS writes happen an iteration later.
template <int PPT>
__device__ __forceinline__ void load_weight(_Float16 const *__restrict__ src, int ld, int R, int C,
                                            uint4v (&x)[PPT][4], int tid, int nthreads) {
  int const cblocks = C / 8, patches = (R / 4) * cblocks;
#pragma unroll
  for (int i = 0; i < PPT; i++) {
    int p = tid + i * nthreads;
    if (p < patches) {
      int cb = p % cblocks, rb = p / cblocks;
      _Float16 const *s = src + (long long)(4 * rb) * ld + 8 * cb;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        x[i][j] = *reinterpret_cast<uint4v const *>(s + (long long)j * ld);
      }
    }
  }
}

template <int PPT>
__device__ __forceinline__ void store_weight(uint4v const (&x)[PPT][4], int R, int C,
                                             _Float16 *__restrict__ dst, int tid, int nthreads) {
  int const cblocks = C / 8, patches = (R / 4) * cblocks;
  int const mask = ((R / 8) - 1) & 7;
#pragma unroll
  for (int i = 0; i < PPT; i++) {
    int p = tid + i * nthreads;
    if (p < patches) {
      int cb = p % cblocks, rb = p / cblocks;
#pragma unroll
      for (int w = 0; w < 4; w++) {
        uint2v even, odd;  // byte permute: selector bytes 0-3 from the second operand
        even.x = __builtin_amdgcn_perm(x[i][1][w], x[i][0][w], 0x05040100u);
        even.y = __builtin_amdgcn_perm(x[i][3][w], x[i][2][w], 0x05040100u);
        odd.x = __builtin_amdgcn_perm(x[i][1][w], x[i][0][w], 0x07060302u);
        odd.y = __builtin_amdgcn_perm(x[i][3][w], x[i][2][w], 0x07060302u);
        int row = 8 * cb + 2 * w;
        *reinterpret_cast<uint2v *>(dst + sw_chunk(row, rb >> 1, R, mask) + (rb & 1) * 4) = even;
        *reinterpret_cast<uint2v *>(dst + sw_chunk(row + 1, rb >> 1, R, mask) + (rb & 1) * 4) = odd;
      }
    }
  }
}

// Column-major weights (a [R][C] tile stored column by column: C rows of R contiguous halfs,
// `ld` halfs apart) already have k contiguous: the same two halves without the transpose.
// The tile is dst[C][R], R / 8 chunks of 16 bytes per row; slot (i, j) of thread `tid` is chunk
// (4 i + j) * nthreads + tid, so that the lanes of one load or store instruction walk
// consecutive chunks of a row (whole cache lines per instruction).
template <int PPT>
__device__ __forceinline__ void load_weight_cm(_Float16 const *__restrict__ src, int ld, int R, int C,
                                               uint4v (&x)[PPT][4], int tid, int nthreads) {
  int const cpr = R / 8, chunks = C * cpr;
#pragma unroll
  for (int i = 0; i < PPT; i++) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      int const q = (4 * i + j) * nthreads + tid;
      if (q < chunks) {
        x[i][j] = *reinterpret_cast<uint4v const *>(src + (long long)(q / cpr) * ld + 8 * (q % cpr));
      }
    }
  }
}

template <int PPT>
__device__ __forceinline__ void store_weight_cm(uint4v const (&x)[PPT][4], int R, int C,
                                                _Float16 *__restrict__ dst, int tid, int nthreads) {
  int const cpr = R / 8, chunks = C * cpr;
  int const mask = (cpr - 1) & 7;
#pragma unroll
  for (int i = 0; i < PPT; i++) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      int const q = (4 * i + j) * nthreads + tid;
      if (q < chunks) {
        *reinterpret_cast<uint4v *>(dst + sw_chunk(q / cpr, q % cpr, R, mask)) = x[i][j];
      }
    }
  }
}

// MT m-tiles of 16 rows, NB weight matrices, 4 wavefronts = the 4 column tiles of a
// 64-column weight tile.  KTMAX bounds the staging register arrays.  WCM: every weight-side
// operand (weights, lora A and B) is a column-major tensor.
template <int MT, int NB, int PRO, bool LORA, int KTMAX, bool WCM>
__global__ __launch_bounds__(256) void gemm_fused_kernel(GemmParams const P) {
  fetch_kernel_arguments<sizeof(GemmParams), 2>();  // every line of the block, one trip (gridDim.x, .y are read)
  constexpr int NT = 256;
  constexpr int WPPT = ((KTMAX / 4) * 8 + NT - 1) / NT;  // weight patches per thread
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int const tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  int const g = lane / 16, c = lane % 16;
  int const M = P.M, KT = P.KT, F = P.forloop_range;
  int const kmask = ((KT / 8) - 1) & 7;

  // logical block and k range of this workgroup; consecutive ids share a block so the
  // block's partial products are written and read from one XCD's L2 where possible
  int const ks = blockIdx.x % P.ksplit;
  int const bx = blockIdx.x / P.ksplit, by = blockIdx.y, bz = blockIdx.z;
  int const per = (F + P.ksplit - 1) / P.ksplit;
  int const it_begin = ks * per, it_end = (it_begin + per) < F ? (it_begin + per) : F;
  int const block_linear = bx + (gridDim.x / P.ksplit) * (by + gridDim.y * bz);

  // LDS: activation tile [16*MT][KT] | weight tiles NB x [64][KT] | lora A^T [16][KT] |
  // lora B^T [64][16]
  _Float16 *a_lds = reinterpret_cast<_Float16 *>(lds);
  _Float16 *b_lds = a_lds + 16 * MT * KT;
  _Float16 *la_lds = b_lds + NB * 64 * KT;
  _Float16 *lb_lds = la_lds + (LORA ? 16 * KT : 0);

  if (LORA) {
    // B [16][64] -> B^T [64][16], loop invariant: 32 patches
    _Float16 const *src = static_cast<_Float16 const *>(P.lb.ptr) + gtile_offset(P.lb, bx, by, bz, 0);
    if (WCM) {  // already B^T [64][16]: 128 chunks, copied as they are
      uint4v x[1][4];
      load_weight_cm<1>(src, P.lb.d_cols, 16, 64, x, tid, NT);
      store_weight_cm<1>(x, 16, 64, lb_lds, tid, NT);
    } else {
      stage_weight<1>(src, P.lb.d_cols, 16, 64, lb_lds, tid, NT);
    }
  }

  _Float16 acc16[NB][MT][4];  // O[16mt + c][16*wave + 4g + r], used when ksplit == 1
#pragma unroll
  for (int b = 0; b < NB; b++) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        acc16[b][mt][r] = (_Float16)0.0f;
      }
    }
  }

  // Prefetch registers: the raw tiles of the next iteration.
  constexpr int APT = (16 * MT * (KTMAX / 8) + NT - 1) / NT;  // activation chunks per thread
  constexpr int LPPT = (KTMAX / 4) * 2 / NT + 1;             // lora A patches per thread
  uint4v wreg[NB][WPPT][4];
  uint4v lreg[LORA ? LPPT : 1][4];
  half8 areg[APT], ureg[PRO == PRO_SILU_MUL ? APT : 1];
  int const chunks_a = KT / 8;
  auto fetch = [&](int it) {
    _Float16 const *a0 = static_cast<_Float16 const *>(P.a0.ptr) + gtile_offset(P.a0, bx, by, bz, it);
    _Float16 const *a1 = PRO == PRO_SILU_MUL
                             ? static_cast<_Float16 const *>(P.a1.ptr) + gtile_offset(P.a1, bx, by, bz, it)
                             : a0;
#pragma unroll
    for (int i = 0; i < APT; i++) {
      int const e = tid + i * NT;
      int const row = e / chunks_a, ch = e % chunks_a;
      if (e < 16 * MT * chunks_a && row < M) {
        areg[i] = *reinterpret_cast<half8 const *>(a0 + (long long)row * P.a0.d_cols + 8 * ch);
        if (PRO == PRO_SILU_MUL) {
          ureg[i] = *reinterpret_cast<half8 const *>(a1 + (long long)row * P.a1.d_cols + 8 * ch);
        }
      }
    }
#pragma unroll
    for (int b = 0; b < NB; b++) {
      GTile const &bt = b == 0 ? P.b0 : P.b1;
      _Float16 const *src = static_cast<_Float16 const *>(bt.ptr) + gtile_offset(bt, bx, by, bz, it);
      if (WCM) {
        load_weight_cm<WPPT>(src, bt.d_cols, KT, 64, wreg[b], tid, NT);
      } else {
        load_weight<WPPT>(src, bt.d_cols, KT, 64, wreg[b], tid, NT);
      }
    }
    if (LORA) {
      _Float16 const *src = static_cast<_Float16 const *>(P.la.ptr) + gtile_offset(P.la, bx, by, bz, it);
      if (WCM) {
        load_weight_cm<LORA ? LPPT : 1>(src, P.la.d_cols, KT, 16, lreg, tid, NT);
      } else {
        load_weight<LORA ? LPPT : 1>(src, P.la.d_cols, KT, 16, lreg, tid, NT);
      }
    }
  };
  // registers -> LDS: activation tile as it is (prologue applied), weights transposed
  auto stash = [&]() {
#pragma unroll
    for (int i = 0; i < APT; i++) {
      int const e = tid + i * NT;
      int const row = e / chunks_a, ch = e % chunks_a;
      if (e < 16 * MT * chunks_a) {
        half8 v;
        if (row < M) {
          v = areg[i];
          if (PRO == PRO_EXP || PRO == PRO_SILU) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
              v[j] = static_cast<_Float16>(prologue(PRO, static_cast<float>(v[j])));
            }
          } else if (PRO == PRO_SILU_MUL) {
            half8 u = ureg[i];
#pragma unroll
            for (int j = 0; j < 8; j++) {
              _Float16 sg = static_cast<_Float16>(prologue(PRO_SILU, static_cast<float>(v[j])));
              v[j] = static_cast<_Float16>(static_cast<float>(sg) * static_cast<float>(u[j]));
            }
          }
        } else {
#pragma unroll
          for (int j = 0; j < 8; j++) {
            v[j] = (_Float16)0.0f;  // rows past M (M == 8) contribute nothing
          }
        }
        *reinterpret_cast<half8 *>(a_lds + sw_chunk(row, ch, KT, kmask)) = v;
      }
    }
#pragma unroll
    for (int b = 0; b < NB; b++) {
      if (WCM) {
        store_weight_cm<WPPT>(wreg[b], KT, 64, b_lds + b * 64 * KT, tid, NT);
      } else {
        store_weight<WPPT>(wreg[b], KT, 64, b_lds + b * 64 * KT, tid, NT);
      }
    }
    if (LORA) {
      if (WCM) {
        store_weight_cm<LORA ? LPPT : 1>(lreg, KT, 16, la_lds, tid, NT);
      } else {
        store_weight<LORA ? LPPT : 1>(lreg, KT, 16, la_lds, tid, NT);
      }
    }
  };
  bool const split = P.ksplit > 1;
  auto compute = [&](int it) {
    // ---- lora inner product, transposed: D^T = A^T . X^T (rows past M are zero) -----
    half4 dfrag = {(_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f};
    if (LORA) {
      float4v d = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int k0 = 0; k0 < KT; k0 += 32) {
        int ch = (k0 >> 3) + g;
        half8 a = *reinterpret_cast<half8 const *>(la_lds + sw_chunk(c, ch, KT, kmask));  // A^T[n=c]
        half8 x = *reinterpret_cast<half8 const *>(a_lds + sw_chunk(c, ch, KT, kmask));   // X[m=c]
        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, x, d, 0, 0, 0);
      }
      // d[r] = D[m = c][n = 4g + r]: the A fragment of a 16x16x16 MFMA over k = n
#pragma unroll
      for (int r = 0; r < 4; r++) {
        dfrag[r] = static_cast<_Float16>(d[r]);  // the [X.A] tile, fp16
      }
    }
    // ---- main products: wavefront `wave` owns output columns 16*wave .. +15 ---------
#pragma unroll
    for (int b = 0; b < NB; b++) {
      float4v o[MT];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        o[mt] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
      }
      _Float16 const *bt = b_lds + b * 64 * KT;
      for (int k0 = 0; k0 < KT; k0 += 32) {
        int ch = (k0 >> 3) + g;
        half8 w = *reinterpret_cast<half8 const *>(bt + sw_chunk(16 * wave + c, ch, KT, kmask));
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          half8 a = *reinterpret_cast<half8 const *>(a_lds + sw_chunk(16 * mt + c, ch, KT, kmask));
          // weights first: o[mt][r] = O[m = 16mt + c][n = 16 wave + 4g + r]
          o[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, a, o[mt], 0, 0, 0);
        }
      }
      if (LORA) {
        // + [X.A] . B over the 16 concatenated k; B^T rows hold 16 halfs (2 chunks)
        half4 w = *reinterpret_cast<half4 const *>(lb_lds + sw_chunk(16 * wave + c, g >> 1, 16, 1) +
                                                   (g & 1) * 4);
        o[0] = __builtin_amdgcn_mfma_f32_16x16x16f16(w, dfrag, o[0], 0, 0, 0);
      }
      if (split) {
        // this iteration's fp16 product tile goes to its slot of the scratch slab
        _Float16 *tile = P.scratch + (((long long)block_linear * F + it) * NB + b) * (long long)M * 64;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          half4 p16;
#pragma unroll
          for (int r = 0; r < 4; r++) {
            p16[r] = static_cast<_Float16>(o[mt][r]);
          }
          if (16 * mt + c < M) {
            *reinterpret_cast<half4 *>(tile + (16 * mt + c) * 64 + 16 * wave + 4 * g) = p16;
          }
        }
      } else {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            _Float16 p16 = static_cast<_Float16>(o[mt][r]);  // this iteration's product tile
            acc16[b][mt][r] = static_cast<_Float16>(static_cast<float>(acc16[b][mt][r]) +
                                                    static_cast<float>(p16));
          }
        }
      }
    }
  };

  // Steady state is branch-free: the next iteration's loads are issued as soon as this
  // iteration's tiles are in LDS and stay in flight while it is multiplied; the last
  // iteration is peeled.
  // A split for-loop leaves every iteration's tile in its own slot of the slab, so a workgroup
  // may walk its range in any order: each starts at a different iteration (rotating through the
  // range), so that at any moment the workgroups of the chip read at many different offsets
  // along k.  Started in step they would all sit at the same one or two offsets within the
  // operand's power-of-two row or column stride, i.e. on a fraction of the memory channels.
  int const n_it = it_end - it_begin;
  int const rot = split ? (int)((blockIdx.x / P.ksplit * 5u + blockIdx.y * 3u + blockIdx.z) % (unsigned)n_it) : 0;
  auto nth = [&](int i) {
    int const j = i + rot;
    return it_begin + (j >= n_it ? j - n_it : j);
  };
  fetch(nth(0));
  for (int i = 0; i + 1 < n_it; i++) {
    __syncthreads();  // previous iteration's tiles fully consumed
    stash();
    __syncthreads();
    fetch(nth(i + 1));
    __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the products
    compute(nth(i));
  }
  __syncthreads();
  stash();
  __syncthreads();
  compute(nth(n_it - 1));

  // ---- finish ---------------------------------------------------------------------------
  // A split for-loop has left every iteration's tile in the scratch slab.  Otherwise the
  // workgroup's fp16 sums go through LDS so that they leave as 16-byte row segments.
  if (split) {
    return;
  }
  constexpr int LDT = 64 + 8;
  _Float16 *t_lds = reinterpret_cast<_Float16 *>(lds);  // the tiles are dead by now
  __syncthreads();
#pragma unroll
  for (int b = 0; b < NB; b++) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      half4 v;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        v[r] = acc16[b][mt][r];
      }
      *reinterpret_cast<half4 *>(t_lds + (b * 16 * MT + 16 * mt + c) * LDT + 16 * wave + 4 * g) = v;
    }
  }
  __syncthreads();
  int const chunks = M * 8;  // 16-byte chunks of one [M][64] tile
#pragma unroll
  for (int b = 0; b < NB; b++) {
    GTile const &ot = b == 0 ? P.o0 : P.o1;
    _Float16 *og = static_cast<_Float16 *>(const_cast<void *>(ot.ptr)) + gtile_offset(ot, bx, by, bz, 0);
    for (int e = tid; e < chunks; e += NT) {
      int row = e / 8, col = (e % 8) * 8;
      *reinterpret_cast<uint4v *>(og + (long long)row * ot.d_cols + col) =
          *reinterpret_cast<uint4v const *>(t_lds + (b * 16 * MT + row) * LDT + col);
    }
  }
}

// Second pass of a split for-loop: adds the fp16 product tiles of every logical block in
// iteration order (fp16 rounding after each add: the rounding sequence of the sequential
// loop) and stores the block's output tile.  A separate launch rather than a last-arriver
// fix-up: the kernel boundary makes the slabs visible without device-scope fences,
// which on this part write back and invalidate a whole L2 each time (with a fence per
// workgroup the LoRA plan took 77 us instead of 13).
template <int NB>
__global__ __launch_bounds__(256) void gemm_combine_kernel(GemmParams const P) {
  fetch_kernel_arguments<sizeof(GemmParams), 2>();  // (gridDim.x, .y are read)
  int const tid = threadIdx.x, M = P.M, F = P.forloop_range;
  int const bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  int const block_linear = bx + gridDim.x * (by + gridDim.y * bz);
  long long const slab = (long long)NB * M * 64;  // one iteration's tiles
  _Float16 const *all = P.scratch + (long long)block_linear * F * slab;
  // 4-byte pieces (two neighbouring columns), so that even an 8-row tile keeps every thread
  // busy, and sixteen iterations' loads in flight per piece: the adds are a dependent chain,
  // the loads are not.
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  int const pieces = M * 32;
#pragma unroll
  for (int b = 0; b < NB; b++) {
    GTile const &ot = b == 0 ? P.o0 : P.o1;
    _Float16 *og = static_cast<_Float16 *>(const_cast<void *>(ot.ptr)) + gtile_offset(ot, bx, by, bz, 0);
    for (int e = tid; e < pieces; e += 256) {
      int row = e / 32, col = (e % 32) * 2;
      _Float16 const *sp = all + (long long)b * M * 64 + row * 64 + col;
      float a0 = 0.0f, a1 = 0.0f;  // hold fp16 values between the adds
      int q = 0;
      for (; q + 16 <= F; q += 16) {
        half2v v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) {
          v[u] = *reinterpret_cast<half2v const *>(sp + (long long)(q + u) * slab);
        }
#pragma unroll
        for (int u = 0; u < 16; u++) {
          a0 = static_cast<float>(static_cast<_Float16>(a0 + static_cast<float>(v[u][0])));
          a1 = static_cast<float>(static_cast<_Float16>(a1 + static_cast<float>(v[u][1])));
        }
      }
      if (q < F) {
        // the tail's loads go out together as well (past the end: the last tile again, left out
        // of the sums), not one latency after the other
        half2v v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) {
          int const it = q + u < F ? q + u : F - 1;
          v[u] = *reinterpret_cast<half2v const *>(sp + (long long)it * slab);
        }
#pragma unroll
        for (int u = 0; u < 16; u++) {
          if (q + u < F) {
            a0 = static_cast<float>(static_cast<_Float16>(a0 + static_cast<float>(v[u][0])));
            a1 = static_cast<float>(static_cast<_Float16>(a1 + static_cast<float>(v[u][1])));
          }
        }
      }
      half2v r;
      r[0] = static_cast<_Float16>(a0);
      r[1] = static_cast<_Float16>(a1);
      *reinterpret_cast<half2v *>(og + (long long)row * ot.d_cols + col) = r;
    }
  }
}

// The same for up to 160 iterations (what fits LDS).  A workgroup takes 8 rows of one output tile: all of its iterations' pieces (1 KB each) are loaded
// together into LDS, then added in order from there, so that the only trip to memory is one latency
// long (61 rows, 20 iterations, 40 blocks: 22.1 -> 14.6 us for the plan; no slower at 8 rows).
template <int NB>
__global__ __launch_bounds__(256 * NB) void gemm_fold_kernel(GemmParams const P) {
  fetch_kernel_arguments<sizeof(GemmParams), 2>();  // (gridDim.x, .y are read)
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];  // [F][8][64] fp16
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  int const tid = threadIdx.x % 256, lane = tid % 64, wave = tid / 64, M = P.M, F = P.forloop_range;
  // with a gate a workgroup is twice as many threads and has both weights
  int const sets = NB == 2 && P.gate != nullptr ? 2 : 1, set = threadIdx.x / 256;
  int const groups = (M + 7) / 8, per_block = groups * (NB / sets);
  int const bx = blockIdx.x / per_block, by = blockIdx.y, bz = blockIdx.z;
  int const part = blockIdx.x % per_block, b = sets == 2 ? set : part / groups, row0 = 8 * (part % groups);
  int const block_linear = bx + (gridDim.x / per_block) * (by + gridDim.y * bz);
  long long const slab = (long long)NB * M * 64;  // one iteration's tiles
  int const row = row0 + lane / 8 < M ? row0 + lane / 8 : M - 1;
  _Float16 const *src = P.scratch + (long long)block_linear * F * slab + (long long)b * M * 64 + row * 64 + 8 * (lane % 8);
  unsigned char *const mine = lds + set * F * 1024;
  for (int it = wave; it < F; it += 16) {
    uint4v v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (it + 4 * u < F) {
        v[u] = *reinterpret_cast<uint4v const *>(src + (it + 4 * u) * slab);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (it + 4 * u < F) {
        *reinterpret_cast<uint4v *>(mine + (it + 4 * u) * 1024 + 16 * lane) = v[u];
      }
    }
  }
  __syncthreads();
  int const r = tid / 32, col = 2 * (tid % 32);
  half2v a = {(_Float16)0.0f, (_Float16)0.0f};
#pragma unroll 8
  for (int it = 0; it < F; it++) {  // (a packed fp16 add is the exact sum rounded once)
    a += *reinterpret_cast<half2v const *>(mine + it * 1024 + 128 * r + 2 * col);
  }
  if (row0 + r < M) {
    GTile const &ot = b == 0 ? P.o0 : P.o1;
    _Float16 *og = static_cast<_Float16 *>(const_cast<void *>(ot.ptr)) + gtile_offset(ot, bx, by, bz, 0);
    *reinterpret_cast<half2v *>(og + (long long)(row0 + r) * ot.d_cols + col) = a;
  }
  if (sets == 2) {
    half2v *const other = reinterpret_cast<half2v *>(lds + F * 1024 + 128 * r + 2 * col);  // (the second set's, which only its thread has read)
    if (set == 1) {
      *other = a;
    }
    __syncthreads();
    if (set == 0 && row0 + r < M) {
      half2v const u = *other;
      *reinterpret_cast<half2v *>(P.gate + gtile_offset(P.o0, bx, by, bz, 0) + (long long)(row0 + r) * P.o0.d_cols + col) =
          half2v{gate_value(a[0], u[0]), gate_value(a[1], u[1])};
    }
  }
}

// ---------------------------------------------------------------------------------------
// One launch, no scratch: the output tile of a logical block is cut into 16-row x 16-column
// pieces and every piece is a workgroup of its own, so a plan with a handful of blocks still covers the
// chip.  Inside a workgroup the wavefronts are ITERATION LANES: lane ip takes iterations ip,
// ip + IP, ... of the for-loop and needs nobody else for them --
//   * its activation rows come as they lie in memory and are turned into MFMA operands through LDS, the
//     element-wise prologue is applied in registers;
//   * column-major weights come the same way; of row-major ones its 16-column strip of a tile ([KT][16], 32
//     contiguous bytes per k) is copied by direct-to-LDS loads into a buffer of its own and read back with
//     transposing LDS reads, which hand a lane the eight consecutive k of one column;
//   * one wait for all of its loads, then KT / 32 MFMAs per weight matrix (weights as the
//     first operand: a lane ends up with four consecutive columns of one row);
// so the workgroup is IP independent streams with no barrier in the loop.  Every iteration's
// product piece is rounded to fp16 into an LDS slot of its own; after ONE barrier the
// pieces are added in ITERATION order, rounding to fp16 after each add -- the arithmetic of
// the sequential loop (src/kernel/triton_code_gen.cc:223-232) -- and stored.
// Workgroup ids put the column pieces of a block on ids that are equal modulo 8, i.e. on
// one XCD: the 128-byte lines of a weight row that the pieces share are fetched into one L2.
struct LaneParams {
  GemmParams g;
  int gx, gy;        // the plan's grid (x, y): the logical block index is decoded from a flat id
  int blocks;        // logical blocks
  int mtiles;        // 16-row pieces per block
  int pieces;        // 16-column pieces per block
  int rank;          // of lora A
  int slot_base;     // byte offset of the product slots in LDS (after the lanes' buffers)
  // multiply-high division magics (fast_div_magic) of 8 * pieces * mtiles, pieces * mtiles, pieces, gx and gy:
  // the decode of the flat id is on the path to the first load
  uint32_t m_group, m_pieces, m_columns, m_gx, m_gy;
};

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lane_dma16(_Float16 const *gbase, uint32_t lane_byte_offset,
                                           uint32_t lds_wave_base) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds_wave_base)), "v"(lane_byte_offset),
                 "s"(gbase)
               : "m0", "memory");
}
#pragma clang diagnostic pop
__device__ __forceinline__ uint32_t lane_lds_address(void const *p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void const *)p;
}
// within 16 lanes, lane 4a + b names four halfs T[row0 + a][col0 + 4b ..]; lane i receives
// T[row0 + 0..3][col0 + i]
__device__ __forceinline__ half4 lane_tr16(_Float16 const *p) {
  typedef short short4v __attribute__((ext_vector_type(4)));
  short4v const v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (short4v __attribute__((address_space(3))) *)(__attribute__((address_space(3))) void *)(p));
  return __builtin_bit_cast(half4, v);
}

// Activations, and column-major weights (WCM: column n of a weight tile is KT contiguous halfs, so a piece's
// sixteen columns are sixteen streams of whole cache lines that no other workgroup touches), are
// [16][KT] tiles whose operands are 16 contiguous bytes.  They come in units of 64 k, a line of each row, into
// registers in the order they have in memory and become operands through 2 KB of LDS each: read as operands,
// sixteen lanes in a row would be sixteen rows, and a compute unit then gets 16 bytes a cycle from its
// vector cache against 59 (32 rows x 2240 x 1856 in 64-k iterations: 9.0 -> 5.5 us).
constexpr int kUnitBytes = 2048;  // [16][64 k]
// bytes of a wavefront's strips: the units being turned; row-major weights, the [16][16] piece of lora B
// (lora: 16-rank pieces of lora A, the last of them may hold 8)
constexpr int lanes_wave_bytes(int KT, int nb, int lora, bool wcm, int pro) {
  int const units = 1 + (pro == PRO_SILU_MUL ? 1 : 0) + (wcm ? nb + lora : 0);
  return units * kUnitBytes + (wcm ? 0 : (nb + lora) * KT * 32 + lora * 512);
}
// most iteration lanes of a workgroup: what the registers of three tiles in flight leave
constexpr int lanes_most(int KT, int lora) { return lora == 2 && KT == 256 ? 8 : 16; }
template <int KT, int NB, int PRO, int LORA, bool WCM>
__global__ __launch_bounds__(64 * lanes_most(KT, LORA)) void gemm_lanes_kernel(LaneParams const L) {
  fetch_kernel_arguments<sizeof(LaneParams), 4>();  // every line of the block, one trip (blockDim.x is read)
  GemmParams const &P = L.g;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int KS = KT / 32;                                // MFMA steps (and 1 KB loads) per strip
  constexpr int STRIPS = NB + LORA;
  constexpr int KU = (KT + 63) / 64;                         // units, the last one of 32 k where KT is an odd number of them
  constexpr int WAVE_BYTES = lanes_wave_bytes(KT, NB, LORA, WCM, PRO), UNITS = 1 + (PRO == PRO_SILU_MUL) + (WCM ? STRIPS : 0);
  int const tid = threadIdx.x, lane = tid % 64, IP = blockDim.x / 64;
  int const ip = __builtin_amdgcn_readfirstlane(tid / 64);  // (wave-uniform: addresses stay scalar)
  int const g = lane / 16, c = lane % 16;
  int const F = P.forloop_range, M = P.M;

  // flat id -> (logical block, row piece, column piece): ids that differ by 8 x piece index
  // share a block
  auto div = [](unsigned v, uint32_t magic) { return magic == 0 ? v : __umulhi(v, magic); };
  unsigned const S = (unsigned)(L.pieces * L.mtiles);
  unsigned const id = blockIdx.x;
  unsigned const eighth = id >> 3;
  int const blk = (int)(div(id, L.m_group) * 8 + (id & 7));
  int const sub = (int)(eighth - div(eighth, L.m_pieces) * S);
  if (blk >= L.blocks) {
    return;
  }
  int const mt = (int)div((unsigned)sub, L.m_columns), piece = sub - mt * L.pieces;
  unsigned const q1 = div((unsigned)blk, L.m_gx);  // blk / gx
  unsigned const q2 = div(q1, L.m_gy);             // blk / (gx * gy)
  int const bx = (int)((unsigned)blk - q1 * (unsigned)L.gx), by = (int)(q1 - q2 * (unsigned)L.gy), bz = (int)q2;
  int const n0 = 16 * piece;

  unsigned char *const units = lds + ip * WAVE_BYTES, *const mine = units + UNITS * kUnitBytes;
  _Float16 const *strip[STRIPS];
#pragma unroll
  for (int b = 0; b < STRIPS; b++) {
    strip[b] = reinterpret_cast<_Float16 const *>(mine + b * KT * 32);
  }
  _Float16 const *lb_piece = reinterpret_cast<_Float16 const *>(mine + STRIPS * KT * 32);
  _Float16 *slots = reinterpret_cast<_Float16 *>(lds + L.slot_base);  // [F][NB][16][16]

  // this lane's place in a strip load (64 lanes x 16 bytes = 32 rows of 32 bytes) and in the
  // transposing reads
  int const ld_row = lane / 2, ld_half = lane % 2;
  int const tr_off = (c / 4) * 16 + 4 * (c % 4);
  bool const row_ok = 16 * mt + c < M;         // activation row of this lane's fragments
  // units: lane l has chunk l % 8 of rows l / 8 and 8 + l / 8; chunk q of row r lies at q ^ (r / 2 % 8)
  int const l8 = lane / 8, ch8 = lane % 8;
  // (of a unit of 32 k: lane l has chunk l % 4 of row l / 4)
  int const l4 = lane / 4, ch4 = lane % 4;
  auto half_unit = [](int u) { return 64 * u + 32 == KT; };
  auto load_rows = [&](_Float16 const *tile, int ld, int row0, int rows, uint4v (&to)[KU][2]) {  // rows past `rows` re-read one
    auto at = [&](int r) { return tile + (long long)(row0 + r < rows ? row0 + r : rows - 1) * ld; };
#pragma unroll
    for (int u = 0; u < KU; u++) {
      if (half_unit(u)) {
        to[u][0] = *reinterpret_cast<uint4v const *>(at(l4) + 64 * u + 8 * ch4);
      } else {
        to[u][0] = *reinterpret_cast<uint4v const *>(at(l8) + 64 * u + 8 * ch8);
        to[u][1] = *reinterpret_cast<uint4v const *>(at(8 + l8) + 64 * u + 8 * ch8);
      }
    }
  };
  auto put_unit = [&](int which, int u, uint4v const (&from)[2]) {
    unsigned char *const to = units + which * kUnitBytes;
    if (half_unit(u)) {
      *reinterpret_cast<uint4v *>(to + 128 * l4 + 16 * (ch4 ^ (l4 / 2))) = from[0];
    } else {
      *reinterpret_cast<uint4v *>(to + 128 * l8 + 16 * (ch8 ^ (l8 / 2))) = from[0];
      *reinterpret_cast<uint4v *>(to + 128 * l8 + 1024 + 16 * (ch8 ^ (l8 / 2 + 4))) = from[1];
    }
  };
  auto operand = [&](int which, int s) {  // row c, k 32 s + 8 g ..
    return *reinterpret_cast<half8 const *>(units + which * kUnitBytes + 128 * c + 16 * ((4 * s + g) ^ (c / 2)));
  };

  half4 lb_frag[LORA > 0 ? LORA : 1];
  int const rank = L.rank;
  if (LORA > 0) {
    _Float16 const *src = static_cast<_Float16 const *>(P.lb.ptr) + gtile_offset(P.lb, bx, by, bz, 0);
    if (WCM) {
      // lora B^T[n0 + c][k = 16 q + 4g .. + 3]: 8 bytes, loop invariant
#pragma unroll
      for (int q = 0; q < LORA; q++) {
        lb_frag[q] = half4{(_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f};
        if (16 * q + 4 * g < rank) {
          lb_frag[q] = *reinterpret_cast<half4 const *>(src + (long long)(n0 + c) * P.lb.d_cols + 16 * q + 4 * g);
        }
      }
    } else if (lane < 32 * LORA) {
      // lora B [16 LORA][64], loop invariant: this piece's 16 columns, rows of 32 bytes
      lane_dma16(src + n0, (uint32_t)((ld_row * P.lb.d_cols + 8 * ld_half) * 2), lane_lds_address(lb_piece));
    }
  }

  for (int it = ip; it < F; it += IP) {
    // (the previous iteration's operand reads must be out of LDS before the transfers that
    // overwrite the strips are issued; the compiler would otherwise move them up among that
    // iteration's last matrix instructions, past the waits for those reads)
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    // ---- issue everything this iteration needs -------------------------------------------
    uint4v wr[WCM ? STRIPS : 1][KU][2], xr[KU][2], ur[KU][2];
#pragma unroll
    for (int b = 0; b < STRIPS; b++) {
      GTile const &bt = b >= NB ? P.la : (b == 0 ? P.b0 : P.b1);
      int const col0 = b >= NB ? 16 * (b - NB) : n0;
      if (WCM) {
        load_rows(static_cast<_Float16 const *>(bt.ptr) + gtile_offset(bt, bx, by, bz, it), bt.d_cols, col0,
                  b >= NB ? rank : col0 + 16, wr[WCM ? b : 0]);
      } else {
        _Float16 const *src = static_cast<_Float16 const *>(bt.ptr) + gtile_offset(bt, bx, by, bz, it) + col0;
        uint32_t const off = (uint32_t)((ld_row * bt.d_cols + 8 * ld_half) * 2);
#pragma unroll
        for (int j = 0; j < KS; j++) {
          lane_dma16(src + (long long)(32 * j) * bt.d_cols, off, lane_lds_address(strip[b]) + j * 1024);
        }
      }
    }
    load_rows(static_cast<_Float16 const *>(P.a0.ptr) + gtile_offset(P.a0, bx, by, bz, it), P.a0.d_cols, 16 * mt, M, xr);
    if (PRO == PRO_SILU_MUL) {
      load_rows(static_cast<_Float16 const *>(P.a1.ptr) + gtile_offset(P.a1, bx, by, bz, it), P.a1.d_cols, 16 * mt, M, ur);
    }
    if (!WCM) {
      // ---- one wait for all of it (direct-to-LDS loads and register loads do not complete in
      // one order, so nothing short of "all" says that a particular one has landed)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
      asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
#pragma unroll
      for (int u = 0; u < KU; u++) {
#pragma unroll
        for (int h = 0; h < (half_unit(u) ? 1 : 2); h++) {
          asm volatile("" : "+v"(xr[u][h]));  // (no use moves above the wait)
          if (PRO == PRO_SILU_MUL) {
            asm volatile("" : "+v"(ur[u][h]));
          }
        }
      }
#pragma clang diagnostic pop
    }
    float4v o[NB], d[LORA > 0 ? LORA : 1];
#pragma unroll
    for (int q = 0; q < LORA; q++) {
      d[q] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int b = 0; b < NB; b++) {
      o[b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // One row-major weight: every load is there, so all units are turned before the first product (a unit at a time
    // each would wait for its own way through LDS: exp of 4 rows x 384 x 768 in 256-k iterations 3.5 -> 3.2 us, SiLU(a) * u
    // of 4 x 3072 x 512 4.85 -> 4.6; with two weights or a LoRA tile, whose operand reads cover it, no gain).
    constexpr bool AHEAD = !WCM && STRIPS == 1;
    half8 xs[AHEAD ? KS : 1], us[AHEAD && PRO == PRO_SILU_MUL ? KS : 1];
    if (AHEAD) {
#pragma unroll
      for (int u = 0; u < KU; u++) {
        put_unit(0, u, xr[u]);
        if (PRO == PRO_SILU_MUL) {
          put_unit(1, u, ur[u]);
        }
        asm volatile("" ::: "memory");  // (a wavefront's LDS operations complete in order)
#pragma unroll
        for (int h = 0; h < (half_unit(u) ? 1 : 2); h++) {
          xs[AHEAD ? 2 * u + h : 0] = operand(0, h);
          if (PRO == PRO_SILU_MUL) {
            us[AHEAD && PRO == PRO_SILU_MUL ? 2 * u + h : 0] = operand(1, h);
          }
        }
        asm volatile("" ::: "memory");
      }
    }
#pragma unroll
    for (int u = 0; u < KU; u++) {
      if (!AHEAD) {
        put_unit(0, u, xr[u]);
        if (PRO == PRO_SILU_MUL) {
          put_unit(1, u, ur[u]);
        }
        if (WCM) {
#pragma unroll
          for (int b = 0; b < STRIPS; b++) {
            put_unit(UNITS - STRIPS + b, u, wr[WCM ? b : 0][u]);
          }
        }
        asm volatile("" ::: "memory");
      }
#pragma unroll
      for (int h = 0; h < (half_unit(u) ? 1 : 2); h++) {
        int const j = 2 * u + h;
        // ---- activation fragments: rows past M are zero, prologue in registers
        half8 x = AHEAD ? xs[AHEAD ? j : 0] : operand(0, h);
        if (PRO == PRO_EXP || PRO == PRO_SILU) {
#pragma unroll
          for (int e = 0; e < 8; e++) {
            x[e] = static_cast<_Float16>(prologue(PRO, static_cast<float>(x[e])));
          }
        } else if (PRO == PRO_SILU_MUL) {
          half8 const um = AHEAD ? us[AHEAD && PRO == PRO_SILU_MUL ? j : 0] : operand(1, h);
#pragma unroll
          for (int e = 0; e < 8; e++) {
            _Float16 const sg = static_cast<_Float16>(prologue(PRO_SILU, static_cast<float>(x[e])));
            x[e] = static_cast<_Float16>(static_cast<float>(sg) * static_cast<float>(um[e]));
          }
        }
        if (!row_ok) {
#pragma unroll
          for (int e = 0; e < 8; e++) {
            x[e] = (_Float16)0.0f;
          }
        }
        // ---- products: o[r] = O[m = c][n = n0 + 4g + r]; lora's inner one, transposed:
        // d[r] = (X.A)[m = c][n = 4g + r]
#pragma unroll
        for (int b = 0; b < STRIPS; b++) {
          half8 w;
          if (WCM) {
            w = operand(UNITS - STRIPS + b, h);
          } else {
            _Float16 const *wp = strip[b] + (32 * j + 8 * g) * 16 + tr_off;
            half4 const lo = lane_tr16(wp), hi = lane_tr16(wp + 64);
            w = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          }
          float4v &to = b >= NB ? d[b >= NB ? b - NB : 0] : o[b < NB ? b : 0];
          to = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, x, to, 0, 0, 0);
        }
      }
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int b = 0; b < NB; b++) {
#pragma unroll
      for (int q = 0; q < LORA; q++) {
        half4 dfrag;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          dfrag[r] = static_cast<_Float16>(16 * q + 4 * g < rank ? d[q][r] : 0.0f);
        }
        half4 const w = WCM ? lb_frag[q] : lane_tr16(lb_piece + 256 * q + (4 * g) * 16 + tr_off);  // B[k = 16 q + 4g ..][n = c]
        o[b] = __builtin_amdgcn_mfma_f32_16x16x16f16(w, dfrag, o[b], 0, 0, 0);
      }
      half4 p16;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        p16[r] = static_cast<_Float16>(o[b][r]);
      }
      *reinterpret_cast<half4 *>(slots + ((it * NB + b) * 16 + c) * 16 + 4 * g) = p16;
    }
  }
  __syncthreads();
  // ---- the saver: pieces added in iteration order, two neighbouring columns per thread ----
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  for (int e = tid; e < NB * 128; e += blockDim.x) {
    int const b = e / 128, r = (e % 128) / 8, col = (e % 8) * 2;
    _Float16 const *sp = slots + (b * 16 + r) * 16 + col;
    float a0 = 0.0f, a1 = 0.0f;  // hold fp16 values between the adds
    int q = 0;
    for (; q + 8 <= F; q += 8) {
      half2v v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        v[u] = *reinterpret_cast<half2v const *>(sp + (q + u) * NB * 256);
      }
#pragma unroll
      for (int u = 0; u < 8; u++) {
        a0 = static_cast<float>(static_cast<_Float16>(a0 + static_cast<float>(v[u][0])));
        a1 = static_cast<float>(static_cast<_Float16>(a1 + static_cast<float>(v[u][1])));
      }
    }
    for (; q < F; q++) {
      half2v const v = *reinterpret_cast<half2v const *>(sp + q * NB * 256);
      a0 = static_cast<float>(static_cast<_Float16>(a0 + static_cast<float>(v[0])));
      a1 = static_cast<float>(static_cast<_Float16>(a1 + static_cast<float>(v[1])));
    }
    if (16 * mt + r < M) {
      GTile const &ot = b == 0 ? P.o0 : P.o1;
      _Float16 *og = static_cast<_Float16 *>(const_cast<void *>(ot.ptr)) + gtile_offset(ot, bx, by, bz, 0);
      half2v out;
      out[0] = static_cast<_Float16>(a0);
      out[1] = static_cast<_Float16>(a1);
      *reinterpret_cast<half2v *>(og + (long long)(16 * mt + r) * ot.d_cols + n0 + col) = out;
    }
    if (NB == 2 && P.gate != nullptr) {
      *reinterpret_cast<half2v *>(slots + (b * 16 + r) * 16 + col) = half2v{(_Float16)a0, (_Float16)a1};  // (its own slot, which only it has read)
    }
  }
  if (NB == 2 && P.gate != nullptr) {
    __syncthreads();
    _Float16 *const to = P.gate + gtile_offset(P.o0, bx, by, bz, 0);
    for (int e = tid; e < 128; e += blockDim.x) {
      int const r = e / 8, col = (e % 8) * 2;
      half2v const x = *reinterpret_cast<half2v const *>(slots + r * 16 + col), u = *reinterpret_cast<half2v const *>(slots + (16 + r) * 16 + col);
      if (16 * mt + r < M) {
        *reinterpret_cast<half2v *>(to + (long long)(16 * mt + r) * P.o0.d_cols + n0 + col) = half2v{gate_value(x[0], u[0]), gate_value(x[1], u[1])};
      }
    }
  }
}

}  // namespace mi355
