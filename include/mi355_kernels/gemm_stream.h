// gemm_stream_kernel: the skinny-GEMM family (gemm.h: plain, two-weight, gate, lora) where the weights'
// bytes are what costs: 64-column weight tiles, iterations of whole 64 k, up to 64 activation rows,
// either storage order of the weights.
//
// A workgroup owns the 64 columns of a logical block and a range of the for-loop; each of its four
// wavefronts takes every fourth iteration of the range and needs nobody else for it: a ring of LDS
// slots of its own (64 columns x 64 k of one weight matrix, whole 128-byte lines, and the activations'
// 64 k beside it) is filled by direct-to-LDS loads several 
// in flight, no register waits for memory and no barrier stands in the loop.  Column-major weights are
// read back as they are, row-major ones with transposing reads; chunks are XOR-swizzled on the way in
// so that both are free of bank conflicts.
//
// An iteration's product is rounded to fp16 into a slot of its own -- in LDS when the workgroup has the
// whole for-loop, in the scratch slab gemm_combine_kernel adds up when ranges share a block -- and the
// slots are added in ITERATION order with one rounding per add: the arithmetic of the sequential loop
// (reference src/kernel/triton_code_gen.cc:223-232).
//
// What bounds it is memory: 235 MB (two weights of 4096 x 14336, column-major) 57 us in the one-launch
// kernel, 45 here (5.2 TB/s; a kernel that only reads them takes 38); 118 MB, one weight, 19 us (6.2).
// The gate's activations (silu of 14336 x 16 values in every column block) are vector work on top:
// 25 us for 117 MB.
#pragma once

#include "gemm.h"

namespace mi355 {

struct StreamParams {
  GemmParams g;
  int results;  // byte offset of the iterations' results in LDS (one range only)
};
// Slots per wavefront.  A third one changes nothing (118 MB of weights: 19.0 us with either), two
// workgroups on a compute unit, which two slots leave room for, do.
constexpr int kStreamRing = 2;

template <int N>
__device__ __forceinline__ void stream_wait() {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
#pragma clang diagnostic pop
}

// Bytes of a slot: the weight tile, then activation rows (and the gate's second operand), then lora A.
constexpr int stream_slot_bytes(int pro, bool lora, int mt) {
  return 8192 + 2048 * mt * (pro == PRO_SILU_MUL ? 2 : 1) + (lora ? 2048 : 0);
}

template <int NB, int PRO, bool LORA, bool WCM, int MT>
__global__ __launch_bounds__(256) void gemm_stream_kernel(StreamParams const S) {
  fetch_kernel_arguments<sizeof(StreamParams), 2>();
  GemmParams const &P = S.g;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int W = 4, SLOT = stream_slot_bytes(PRO, LORA, MT);
  constexpr int X_LOADS = 2 * MT * (PRO == PRO_SILU_MUL ? 2 : 1) + (LORA ? 2 : 0);  // besides the weights' 8
  constexpr int X_AT = 8192, U_AT = X_AT + 2048 * MT, LA_AT = U_AT + (PRO == PRO_SILU_MUL ? 2048 * MT : 0);
  int const tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  int const g = lane / 16, c = lane % 16;
  int const M = P.M, F = P.forloop_range, subs = P.KT / 64;
  constexpr int R = kStreamRing;

  int const gx = gridDim.x / P.ksplit;
  int const ks = blockIdx.x % P.ksplit;  // (the ranges of a block next to each other)
  int const bx = blockIdx.x / P.ksplit, by = blockIdx.y, bz = blockIdx.z;
  int const per = (F + P.ksplit - 1) / P.ksplit;
  int const it_begin = ks * per, n_it = (it_begin + per < F ? it_begin + per : F) - it_begin;
  int const block_linear = bx + gx * (by + gridDim.y * bz);
  // This wavefront's iterations, starting at another one in each workgroup: started in step, all would
  // read at the same offsets of a power-of-two column stride, a fraction of the memory channels.
  int const n_mine = (n_it - wave + W - 1) / W;
  int const rot = n_mine > 1 ? (int)((unsigned)block_linear % (unsigned)n_mine) : 0;
  auto nth = [&](int i) {
    int const j = i + rot;
    return it_begin + wave + W * (j >= n_mine ? j - n_mine : j);
  };

  unsigned char *const mine = lds + wave * R * SLOT;
  uint32_t const mine_at = lane_lds_address(mine);

  // ---- loads: lane l of a load writes the 16 bytes at 16 l of its KB ------------------------------
  // weights, load j of 8: column-major, columns 8 j + l / 8, chunk l % 8 of the column's 64 k;
  // row-major, k rows 8 j + l / 8, chunk l % 8 of the row's 64 columns.  Both swizzled by the row of
  // the LDS tile (the chunk a lane FETCHES moves, its place is fixed).
  auto swizzle = [](int row) { return WCM ? (row >> 1) & 7 : (((row >> 1) & 1) | ((row >> 2) & 2)) << 1; };
  int const l8 = lane / 8, ch8 = lane % 8;
  uint32_t w_off[2][NB];  // rows 8 j + l8: the swizzle of rows 8 apart differs, so even and odd j
#pragma unroll
  for (int b = 0; b < NB; b++) {
    int const ld = b == 0 ? P.b0.d_cols : P.b1.d_cols;
    w_off[0][b] = 2u * (uint32_t)(l8 * ld + 8 * (ch8 ^ swizzle(l8)));
    w_off[1][b] = 2u * (uint32_t)(l8 * ld + 8 * (ch8 ^ swizzle(8 + l8)));
  }
  // activation rows 8 j + l / 8 (rows past the tile re-read its last one: theirs are not stored)
  uint32_t x_off[2 * MT], u_off[PRO == PRO_SILU_MUL ? 2 * MT : 1];
#pragma unroll
  for (int j = 0; j < 2 * MT; j++) {
    int const row = 8 * j + l8, rr = row < M ? row : M - 1;
    uint32_t const chunk = 8u * (uint32_t)(ch8 ^ ((row >> 1) & 7));
    x_off[j] = 2u * ((uint32_t)(rr * P.a0.d_cols) + chunk);
    if (PRO == PRO_SILU_MUL) {
      u_off[j] = 2u * ((uint32_t)(rr * P.a1.d_cols) + chunk);
    }
  }
  // lora A: column-major like the weights (16 columns), row-major k rows 32 j + l / 2 of 32 bytes
  auto issue = [&](int it, int sub, int b, int slot) {
    uint32_t const at = mine_at + (uint32_t)(slot * SLOT);
    GTile const &bt = b == 0 ? P.b0 : P.b1;
    _Float16 const *w = static_cast<_Float16 const *>(bt.ptr) + gtile_offset(bt, bx, by, bz, it) +
                        (WCM ? (long long)(64 * sub) : (long long)(64 * sub) * bt.d_cols);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      lane_dma16(w + (long long)(8 * j) * bt.d_cols, w_off[j & 1][b], at + (uint32_t)(1024 * j));
    }
    if (b == 0) {
      _Float16 const *x = static_cast<_Float16 const *>(P.a0.ptr) + gtile_offset(P.a0, bx, by, bz, it) + 64 * sub;
#pragma unroll
      for (int j = 0; j < 2 * MT; j++) {
        lane_dma16(x, x_off[j], at + (uint32_t)(X_AT + 1024 * j));
      }
      if (PRO == PRO_SILU_MUL) {
        _Float16 const *u = static_cast<_Float16 const *>(P.a1.ptr) + gtile_offset(P.a1, bx, by, bz, it) + 64 * sub;
#pragma unroll
        for (int j = 0; j < 2 * MT; j++) {
          lane_dma16(u, u_off[j], at + (uint32_t)(U_AT + 1024 * j));
        }
      }
      if (LORA) {
        _Float16 const *la = static_cast<_Float16 const *>(P.la.ptr) + gtile_offset(P.la, bx, by, bz, it) +
                             (WCM ? (long long)(64 * sub) : (long long)(64 * sub) * P.la.d_cols);
#pragma unroll
        for (int j = 0; j < 2; j++) {
          uint32_t const off = WCM ? 2u * (uint32_t)(l8 * P.la.d_cols + 8 * (ch8 ^ swizzle(8 * j + l8)))
                                   : 2u * (uint32_t)((lane / 2) * P.la.d_cols + 8 * (lane % 2));
          lane_dma16(la + (long long)(WCM ? 8 * j : 32 * j) * P.la.d_cols, off, at + (uint32_t)(LA_AT + 1024 * j));
        }
      }
    }
  };
  // operand of 16 weight columns from 16 t, k step s of 32: lane (g, c) holds [k = 32 s + 8 g ..][16 t + c]
  auto weights = [&](unsigned char const *slot, int t, int s) {
    if (WCM) {
      int const row = 16 * t + c;
      return *reinterpret_cast<half8 const *>(slot + 128 * row + 16 * ((4 * s + g) ^ swizzle(row)));
    }
    int const row = 32 * s + 8 * g + (c >> 2);  // (rows 4 apart share a swizzle but for bit 1: 4 -> same)
    auto at = [&](int r) {
      return reinterpret_cast<_Float16 const *>(slot + 128 * r + 16 * ((2 * t + ((c & 3) >> 1)) ^ swizzle(r)) + 8 * (c & 1));
    };
    half4 const lo = lane_tr16(at(row)), hi = lane_tr16(at(row + 4));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto rows = [&](unsigned char const *x, int mt, int s) {
    int const row = 16 * mt + c;
    return *reinterpret_cast<half8 const *>(x + 128 * row + 16 * ((4 * s + g) ^ ((row >> 1) & 7)));
  };

  half4 lb_frag[4];  // lora B[4 g ..][16 t + c], loop invariant
  if (LORA) {
    _Float16 const *lb = static_cast<_Float16 const *>(P.lb.ptr) + gtile_offset(P.lb, bx, by, bz, 0);
#pragma unroll
    for (int t = 0; t < 4; t++) {
      if (WCM) {
        lb_frag[t] = *reinterpret_cast<half4 const *>(lb + (long long)(16 * t + c) * P.lb.d_cols + 4 * g);
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          lb_frag[t][r] = lb[(long long)(4 * g + r) * P.lb.d_cols + 16 * t + c];
        }
      }
    }
    stream_wait<0>();  // (before the counted loads begin)
#pragma unroll
    for (int t = 0; t < 4; t++) {
      asm volatile("" : "+v"(lb_frag[t]));
    }
  }

  // ---- the loop: step = one weight matrix's 64 k ---------------------------------------------------
  int const total = n_mine > 0 ? n_mine * subs * NB : 0;
  int i_it = 0, i_sub = 0, i_b = 0, i_slot = 0, issued = 0;  // the next step to issue
  auto issue_next = [&]() {
    if (NB == 1 || i_b == 0) {
      issue(nth(i_it), i_sub, 0, i_slot);
    } else {
      issue(nth(i_it), i_sub, 1, i_slot);
    }
    issued++;
    i_slot = i_slot + 1 == R ? 0 : i_slot + 1;
    if (NB == 2) {
      i_b ^= 1;
    }
    if (NB == 1 || i_b == 0) {
      i_sub++;
      if (i_sub == subs) {
        i_sub = 0;
        i_it++;
      }
    }
  };
  for (int s = 0; s < R && s < total; s++) {
    issue_next();
  }
  int slot = 0, step = 0;
  for (int i = 0; i < n_mine; i++) {
    float4v o[NB][4][MT], d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < NB; b++) {
#pragma unroll
      for (int t = 0; t < 4; t++) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          o[b][t][mt] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
    }
    for (int sub = 0; sub < subs; sub++) {
      half8 x[MT][2];
#pragma unroll
      for (int b = 0; b < NB; b++, step++) {
        // this step has landed when only the loads of the one after it are outstanding
        if (issued - 1 > step) {
          stream_wait<NB == 1 ? 8 + X_LOADS : 8>();
        } else {
          stream_wait<0>();
        }
        unsigned char const *const at = mine + slot * SLOT;
        half8 w[4][2], la[2];
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
          for (int t = 0; t < 4; t++) {
            w[t][s] = weights(at, t, s);
          }
        }
        half8 u[PRO == PRO_SILU_MUL ? MT : 1][2];
        if (b == 0) {
#pragma unroll
          for (int s = 0; s < 2; s++) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
              x[mt][s] = rows(at + X_AT, mt, s);
              if (PRO == PRO_SILU_MUL) {
                u[mt][s] = rows(at + U_AT, mt, s);
              }
            }
            if (LORA) {
              if (WCM) {
                la[s] = *reinterpret_cast<half8 const *>(at + LA_AT + 128 * c + 16 * ((4 * s + g) ^ swizzle(c)));
              } else {
                _Float16 const *ap = reinterpret_cast<_Float16 const *>(at + LA_AT) + (32 * s + 8 * g + (c >> 2)) * 16 + 4 * (c & 3);
                half4 const lo = lane_tr16(ap), hi = lane_tr16(ap + 64);
                la[s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
              }
            }
          }
        }
        // the slot is in registers: the step that takes it next may fly
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (issued < total) {
          issue_next();
        }
        slot = slot + 1 == R ? 0 : slot + 1;
        if (b == 0) {
          if (PRO != PRO_NONE) {
#pragma unroll
            for (int s = 0; s < 2; s++) {
#pragma unroll
              for (int mt = 0; mt < MT; mt++) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                  _Float16 v = static_cast<_Float16>(prologue(PRO == PRO_EXP ? PRO_EXP : PRO_SILU, static_cast<float>(x[mt][s][e])));
                  if (PRO == PRO_SILU_MUL) {
                    v = static_cast<_Float16>(static_cast<float>(v) * static_cast<float>(u[mt][s][e]));
                  }
                  x[mt][s][e] = v;
                }
              }
            }
          }
          if (LORA) {
#pragma unroll
            for (int s = 0; s < 2; s++) {
              d = __builtin_amdgcn_mfma_f32_16x16x32_f16(la[s], x[0][s], d, 0, 0, 0);
            }
          }
        }
        // weights first: o[b][t][mt][r] = O[16 mt + c][16 t + 4 g + r]
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
          for (int t = 0; t < 4; t++) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
              o[b][t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[t][s], x[mt][s], o[b][t][mt], 0, 0, 0);
            }
          }
        }
      }
    }
    int const it = nth(i);
    if (LORA) {
      // + [X.A] . B: d[r] = (X.A)[c][4 g + r] is the operand of a product over the 16 ranks
      half4 df;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        df[r] = static_cast<_Float16>(d[r]);
      }
#pragma unroll
      for (int t = 0; t < 4; t++) {
        o[0][t][0] = __builtin_amdgcn_mfma_f32_16x16x16f16(lb_frag[t], df, o[0][t][0], 0, 0, 0);
      }
    }
    // ---- this iteration's product, fp16 ----------------------------------------------------------
#pragma unroll
    for (int b = 0; b < NB; b++) {
      long long const tile = (long long)M * 64;
      _Float16 *const to = P.ksplit > 1 ? P.scratch + (((long long)block_linear * F + it) * NB + b) * tile
                                        : reinterpret_cast<_Float16 *>(lds + S.results) + (it * NB + b) * (int)tile;
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        if (16 * mt + c < M) {
#pragma unroll
          for (int t = 0; t < 4; t++) {
            *reinterpret_cast<half4 *>(to + (16 * mt + c) * 64 + 16 * t + 4 * g) = __builtin_convertvector(o[b][t][mt], half4);
          }
        }
      }
    }
  }
  if (P.ksplit > 1) {
    return;
  }
  // ---- the saver: the iterations' products in order ----------------------------------------------
  __syncthreads();
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  _Float16 const *const all = reinterpret_cast<_Float16 const *>(lds + S.results);
  for (int e = tid; e < NB * M * 16; e += 256) {
    int const b = e / (M * 16), q = e % (M * 16), row = q / 16, col = 4 * (q % 16);
    _Float16 const *src = all + b * M * 64 + row * 64 + col;
    half2v lo = {(_Float16)0.0f, (_Float16)0.0f}, hi = lo;
    for (int it = 0; it < F; it++) {  // (a packed fp16 add is the exact sum rounded once)
      half4 const v = *reinterpret_cast<half4 const *>(src + it * NB * M * 64);
      lo += half2v{v[0], v[1]};
      hi += half2v{v[2], v[3]};
    }
    GTile const &ot = b == 0 ? P.o0 : P.o1;
    _Float16 *og = static_cast<_Float16 *>(const_cast<void *>(ot.ptr)) + gtile_offset(ot, bx, by, bz, 0);
    *reinterpret_cast<half4 *>(og + (long long)row * ot.d_cols + col) = half4{lo[0], lo[1], hi[0], hi[1]};
  }
}

}  // namespace mi355
