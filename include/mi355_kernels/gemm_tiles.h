// gemm_tiles_kernel: the skinny-GEMM family of thread-block graphs (see gemm.h for its members) at
// any tile size: activation tiles of any number of rows, weight tiles of any multiple of 16
// columns, iterations of any multiple of 32 k, LoRA ranks 8, 16 and 32, weights in either storage
// order.  The kernels of gemm.h are built for 64-column tiles; what they do not take runs here
// instead of statement by statement in the generic LDS interpreter.
//
// A workgroup owns 16 MT rows x 16 CT columns of a logical block's output.  Its wavefronts are
// iteration lanes: lane ip takes iterations ip, ip + IP, ... of a round by itself, both operands of
// every product going from global memory into registers (eight consecutive k of a row or column
// are sixteen contiguous bytes; a row-major weight strip takes one trip through a private strip of
// LDS and a transposing read), and leaves each iteration's fp16 product in an LDS slot of its
// own.  After one barrier the round's slots are added in ITERATION order with one fp16 rounding
// per add: the sequence of roundings of the sequential loop (reference
// src/kernel/triton_code_gen.cc:223-232).  A round is the whole for-loop whenever its slots fit.
//
// What bounds it: the trip to memory for plans of a few MB (the loads of up to KS steps of 32 k go
// out together), the weight stream for larger ones.  Pieces of 16 columns put a workgroup on every
// compute unit for plans of a few dozen blocks; 32 columns halve the re-reading of the activations
// and make a row-major weight strip's rows 64 contiguous bytes.
#pragma once

#include "gemm.h"

namespace mi355 {

struct TileGemmParams {
  GemmParams g;   // (ksplit and scratch unused)
  int strips;     // column strips of 16 CT per block
  int slabs;      // row slabs of 16 MT per block
  int round;      // iterations per round (a multiple of the lanes, or the whole for-loop)
  int rank;       // lora: 8, 16 or 32 (0: no lora)
  int cols;       // columns of a weight tile
  uint32_t m_strips, m_slabs;  // division magics (fast_div_magic)
};

// Steps of 32 k whose loads are in flight together.
constexpr int gemm_tiles_steps(int MT, int NB, bool LORA) { return MT == 1 && NB == 1 && !LORA ? 8 : 4; }

// Most iteration lanes of a workgroup: sixteen where 128 registers hold a lane's operands.
constexpr int gemm_tiles_lanes(int MT, int CT, int NB, int PRO, bool LORA) {
  return MT == 1 && CT == 1 && NB == 1 && !LORA && PRO != PRO_SILU_MUL ? 16 : 8;
}

template <int MT, int CT, int NB, int PRO, bool LORA, bool WCM>
__global__ __launch_bounds__(64 * gemm_tiles_lanes(MT, CT, NB, PRO, LORA)) void gemm_tiles_kernel(TileGemmParams const L) {
  fetch_kernel_arguments<sizeof(TileGemmParams), 4>();  // (blockDim.x is read)
  GemmParams const &P = L.g;
  constexpr int KS = gemm_tiles_steps(MT, NB, LORA);
  constexpr int RT = LORA ? 2 : 0;              // 16-wide pieces of the rank
  constexpr int LDO = 16 * CT + 4;              // slot row stride (halfs)
  constexpr int SLOT = NB * 16 * MT * LDO;
  constexpr int OWN = NB * MT * CT;             // 8-byte pieces a thread adds up, one wavefront
  constexpr int SW = 16 * CT + 8, LW = 40;      // row strides of the transposing strips
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int const tid = threadIdx.x, NT = blockDim.x, IP = NT / 64, lane = tid % 64;
  int const ip = __builtin_amdgcn_readfirstlane(tid / 64);
  int const gq = lane / 16, c = lane % 16, a4 = c >> 2, b4 = c & 3;
  int const F = P.forloop_range, M = P.M, steps = P.KT / 32;

  auto div = [](unsigned v, uint32_t magic) { return magic == 0 ? v : __umulhi(v, magic); };
  unsigned const q1 = div(blockIdx.x, L.m_strips), q2 = div(q1, L.m_slabs);
  int const n0 = 16 * CT * (int)(blockIdx.x - q1 * (unsigned)L.strips);
  int const row0 = 16 * MT * (int)(q1 - q2 * (unsigned)L.slabs);
  int const bx = (int)q2, by = blockIdx.y, bz = blockIdx.z;

  _Float16 *const slots = reinterpret_cast<_Float16 *>(lds);  // [1 or 2][round][SLOT]
  bool const rounds = L.round < F;
  // (row-major weights: a strip of 32 k per lane, and one of the lora A tile)
  _Float16 *const w_strip = slots + (rounds ? 2 : 1) * L.round * SLOT + ip * (32 * SW + (LORA ? 32 * LW : 0));
  _Float16 *const l_strip = w_strip + 32 * SW;

  int rows[MT];  // activation rows of this lane's fragments (past the tile: its last row, not stored)
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    rows[mt] = row0 + 16 * mt + c < M ? row0 + 16 * mt + c : M - 1;
  }

  // lora B^T[n0 + 16 ct + c][k = 16 rt + 4g .. + 3], loop invariant; k past the rank is zero
  half4 lb[LORA ? CT : 1][LORA ? RT : 1];
  if (LORA) {
    _Float16 const *src = static_cast<_Float16 const *>(P.lb.ptr) + gtile_offset(P.lb, bx, by, bz, 0);
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
#pragma unroll
      for (int rt = 0; rt < RT; rt++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          int const k = 16 * rt + 4 * gq + e, n = n0 + 16 * ct + c;
          lb[ct][rt][e] = (_Float16)0.0f;
          if (k < L.rank) {
            lb[ct][rt][e] = src[WCM ? (long long)n * P.lb.d_cols + k : (long long)k * P.lb.d_cols + n];
          }
        }
      }
    }
  }

  half4 acc[OWN];  // this thread's pieces of the result (fp16 sums)
#pragma unroll
  for (int i = 0; i < OWN; i++) {
    acc[i] = half4{(_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f};
  }

  int buf = 0;
  for (int r0 = 0; r0 < F; r0 += L.round, buf ^= 1) {
    _Float16 *const round = slots + buf * L.round * SLOT;
    int const r_end = r0 + L.round < F ? r0 + L.round : F;
    for (int it = r0 + ip; it < r_end; it += IP) {
      _Float16 const *const a0 = static_cast<_Float16 const *>(P.a0.ptr) + gtile_offset(P.a0, bx, by, bz, it);
      _Float16 const *const a1 = static_cast<_Float16 const *>(P.a1.ptr) + gtile_offset(P.a1, bx, by, bz, it);
      _Float16 const *const la = static_cast<_Float16 const *>(P.la.ptr) + gtile_offset(P.la, bx, by, bz, it);
      float4v o[NB][MT][CT], d[LORA ? MT : 1][LORA ? RT : 1];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
          for (int ct = 0; ct < CT; ct++) {
            o[b][mt][ct] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
          }
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
          d[LORA ? mt : 0][LORA ? rt : 0] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
      for (int s0 = 0; s0 < steps; s0 += KS) {
        // ---- the loads of up to KS steps of 32 k
        uint4v w[NB][KS][CT], x[KS][MT], u[PRO == PRO_SILU_MUL ? KS : 1][MT], lr[LORA ? KS : 1][LORA ? RT : 1];
#pragma unroll
        for (int s = 0; s < KS; s++) {
          if (s0 + s < steps) {
            int const k0 = 32 * (s0 + s);
#pragma unroll
            for (int b = 0; b < NB; b++) {
              GTile const &bt = b == 0 ? P.b0 : P.b1;
              _Float16 const *wg = static_cast<_Float16 const *>(bt.ptr) + gtile_offset(bt, bx, by, bz, it);
#pragma unroll
              for (int ct = 0; ct < CT; ct++) {
                // column-major: W^T[n0 + 16 ct + c][k0 + 8g ..]; row-major: chunk 64 ct + lane of
                // the strip [32 k][16 CT columns]
                long long const off = WCM ? (long long)(n0 + 16 * ct + c) * bt.d_cols + k0 + 8 * gq
                                          : (long long)(k0 + (64 * ct + lane) / (2 * CT)) * bt.d_cols + n0 + 8 * (lane % (2 * CT));
                w[b][s][ct] = *reinterpret_cast<uint4v const *>(wg + off);
              }
            }
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
              x[s][mt] = *reinterpret_cast<uint4v const *>(a0 + (long long)rows[mt] * P.a0.d_cols + k0 + 8 * gq);
              if (PRO == PRO_SILU_MUL) {
                u[PRO == PRO_SILU_MUL ? s : 0][mt] =
                    *reinterpret_cast<uint4v const *>(a1 + (long long)rows[mt] * P.a1.d_cols + k0 + 8 * gq);
              }
            }
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
              if (16 * rt < L.rank) {
                // column-major: A^T[rank index][k0 + 8g ..] (past the rank: its last row, dropped
                // below); row-major: the [32 k][rank] strip, 16 bytes a lane
                int const n = 16 * rt + c < L.rank ? 16 * rt + c : L.rank - 1;
                int const cpr = L.rank / 8, q = 64 * rt + lane;
                int const qr = q / cpr < 32 ? q / cpr : 31;  // (rank 8: half of the lanes hold the strip)
                long long const off = WCM ? (long long)n * P.la.d_cols + k0 + 8 * gq
                                          : (long long)(k0 + qr) * P.la.d_cols + 8 * (q % cpr);
                lr[LORA ? s : 0][LORA ? rt : 0] = *reinterpret_cast<uint4v const *>(la + off);
              }
            }
          }
        }
        // ---- products, weights first: o[r] = O[m = c][n = 4g + r]
#pragma unroll
        for (int s = 0; s < KS; s++) {
          if (s0 + s < steps) {
            half8 xf[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
              half8 v = __builtin_bit_cast(half8, x[s][mt]);
              if (PRO == PRO_EXP || PRO == PRO_SILU) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                  v[e] = static_cast<_Float16>(prologue(PRO, static_cast<float>(v[e])));
                }
              } else if (PRO == PRO_SILU_MUL) {
                half8 const um = __builtin_bit_cast(half8, u[PRO == PRO_SILU_MUL ? s : 0][mt]);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                  _Float16 const sg = static_cast<_Float16>(prologue(PRO_SILU, static_cast<float>(v[e])));
                  v[e] = static_cast<_Float16>(static_cast<float>(sg) * static_cast<float>(um[e]));
                }
              }
              xf[mt] = v;
            }
#pragma unroll
            for (int b = 0; b < NB; b++) {
              if (!WCM) {
#pragma unroll
                for (int ct = 0; ct < CT; ct++) {
                  *reinterpret_cast<uint4v *>(w_strip + ((64 * ct + lane) / (2 * CT)) * SW + 8 * (lane % (2 * CT))) = w[b][s][ct];
                }
                asm volatile("" ::: "memory");  // (a wavefront's LDS operations complete in order)
              }
#pragma unroll
              for (int ct = 0; ct < CT; ct++) {
                half8 wf;
                if (WCM) {
                  wf = __builtin_bit_cast(half8, w[b][s][ct]);
                } else {
                  _Float16 const *wp = w_strip + (8 * gq + a4) * SW + 16 * ct + 4 * b4;
                  half4 const lo = lane_tr16(wp), hi = lane_tr16(wp + 4 * SW);
                  wf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                }
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                  o[b][mt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, xf[mt], o[b][mt][ct], 0, 0, 0);
                }
              }
              asm volatile("" ::: "memory");
            }
            if (LORA) {
              if (!WCM) {
#pragma unroll
                for (int rt = 0; rt < RT; rt++) {
                  int const cpr = L.rank / 8, q = 64 * rt + lane;
                  if (16 * rt < L.rank && q < 32 * cpr) {
                    *reinterpret_cast<uint4v *>(l_strip + (q / cpr) * LW + 8 * (q % cpr)) = lr[LORA ? s : 0][LORA ? rt : 0];
                  }
                }
                asm volatile("" ::: "memory");
              }
#pragma unroll
              for (int rt = 0; rt < RT; rt++) {
                if (16 * rt < L.rank) {
                  half8 af;
                  if (WCM) {
                    af = __builtin_bit_cast(half8, lr[LORA ? s : 0][LORA ? rt : 0]);
                  } else {
                    _Float16 const *ap = l_strip + (8 * gq + a4) * LW + 16 * rt + 4 * b4;
                    half4 const lo = lane_tr16(ap), hi = lane_tr16(ap + 4 * LW);
                    af = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                  }
#pragma unroll
                  for (int mt = 0; mt < MT; mt++) {
                    d[LORA ? mt : 0][LORA ? rt : 0] =
                        __builtin_amdgcn_mfma_f32_16x16x32_f16(af, xf[mt], d[LORA ? mt : 0][LORA ? rt : 0], 0, 0, 0);
                  }
                }
              }
              asm volatile("" ::: "memory");
            }
          }
        }
      }
      if (LORA) {
        // + [X.A] . B over the concatenated k: d[r] = (X.A)[m = c][n = 16 rt + 4g + r], rounded to
        // fp16 (the materialised tile); columns past the rank are zero
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
          if (16 * rt < L.rank) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
              half4 df;
#pragma unroll
              for (int r = 0; r < 4; r++) {
                df[r] = 16 * rt + 4 * gq + r < L.rank ? static_cast<_Float16>(d[LORA ? mt : 0][LORA ? rt : 0][r]) : (_Float16)0.0f;
              }
#pragma unroll
              for (int ct = 0; ct < CT; ct++) {
                o[0][mt][ct] = __builtin_amdgcn_mfma_f32_16x16x16f16(lb[LORA ? ct : 0][LORA ? rt : 0], df, o[0][mt][ct], 0, 0, 0);
              }
            }
          }
        }
      }
      // ---- this iteration's product, fp16, to its slot
      _Float16 *const slot = round + (it - r0) * SLOT;
#pragma unroll
      for (int b = 0; b < NB; b++) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
          for (int ct = 0; ct < CT; ct++) {
            half4 p;
#pragma unroll
            for (int r = 0; r < 4; r++) {
              p[r] = static_cast<_Float16>(o[b][mt][ct][r]);
            }
            *reinterpret_cast<half4 *>(slot + (b * 16 * MT + 16 * mt + c) * LDO + 16 * ct + 4 * gq) = p;
          }
        }
      }
    }
    __syncthreads();
    // ---- the round's products in iteration order, one fp16 rounding per add (a packed fp16 add
    // is the exact sum rounded once)
#pragma unroll
    for (int i = 0; i < OWN; i++) {
      int const e = tid + i * NT;
      if (e < NB * 16 * MT * 4 * CT) {
        _Float16 const *src = round + (e / (4 * CT)) * LDO + 4 * (e % (4 * CT));
        int const n = r_end - r0;
        int q = 0;
        for (; q + 8 <= n; q += 8) {  // (the loads are independent, only the adds are a chain)
          half4 v[8];
#pragma unroll
          for (int j = 0; j < 8; j++) {
            v[j] = *reinterpret_cast<half4 const *>(src + (q + j) * SLOT);
          }
#pragma unroll
          for (int j = 0; j < 8; j++) {
            acc[i] = acc[i] + v[j];
          }
        }
        for (; q < n; q++) {
          acc[i] = acc[i] + *reinterpret_cast<half4 const *>(src + q * SLOT);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < OWN; i++) {
    int const e = tid + i * NT;
    if (e < NB * 16 * MT * 4 * CT) {
      int const r = e / (4 * CT), b = r / (16 * MT), row = row0 + r % (16 * MT), col = n0 + 4 * (e % (4 * CT));
      if (row < M) {
        GTile const &ot = b == 0 ? P.o0 : P.o1;
        *reinterpret_cast<half4 *>(static_cast<_Float16 *>(const_cast<void *>(ot.ptr)) + gtile_offset(ot, bx, by, bz, 0) +
                                   (long long)row * ot.d_cols + col) = acc[i];
      }
    }
  }
}

}  // namespace mi355
