// gemm_stream_kernel: the skinny-GEMM family (gemm.h: plain, two-weight, gate, lora) where the weights'
// bytes are what costs: 64-column weight tiles, iterations of whole 64 k, up to 64 activation rows,
// either storage order of the weights.
//
// A workgroup owns the 64 columns of a logical block and a range of the for-loop; each of its four
// wavefronts takes every fourth iteration of the range and needs nobody else for it: a ring of LDS
// slots of its own (64 columns x 64 k of one weight matrix, whole 128-byte lines, and the activations'
// 64 k beside it) is filled by direct-to-LDS loads, several
// in flight; no register waits for memory and no barrier stands in the loop.  Column-major weights are
// read back as they are, row-major ones with transposing reads; chunks are XOR-swizzled on the way in
// so that both are free of bank conflicts.
//
// An iteration's product is rounded to fp16 into a slot of its own -- in LDS when the workgroup has the
// whole for-loop, in the scratch slab gemm_combine_kernel adds up when ranges share a block -- and the
// slots are added in ITERATION order with one rounding per add: the arithmetic of the sequential loop
// (reference src/kernel/triton_code_gen.cc:223-232).
//
// Two weights are two sets of workgroups (for twice the activations' bytes): seven to a compute unit instead of
// three and a half leave less of the last round empty (two weights of 4096 x 14336: 44.3 -> 42.3 us).  Where that does not
// hold, few blocks or one workgroup a compute unit, gemm_stream_pairs_kernel takes both in a workgroup (the host's rule).
//
// What bounds it is memory: 235 MB (those two weights, column-major) 42 us (5.6 TB/s; a kernel that only reads
// them takes 38); 118 MB, one weight, 19 us (6.2).  The gate's activations (silu of 14336 x 16 values in every
// column block) are vector work on top: 24 us for 117 MB.  Up to 8 rows a slot holds 8, which leaves room for two
// workgroups also beside the gate's second operand, and a silu is made by one lane instead of two (gated MLP of
// 8 x 4096 x 14336: 78.9 -> 77.1 us).
#pragma once

#include <type_traits>

#include "gemm.h"

namespace mi355 {

struct StreamParams {
  GemmParams g;
  int results;  // byte offset of the iterations' results in LDS (one range only)
  int strips;   // a workgroup takes 16 columns and the whole for-loop (stream_columns)
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
// mt counts 16-row groups; 0 is one of 8 rows.
constexpr int stream_slot_bytes(int pro, bool lora, int mt) {
  return 8192 + (mt > 0 ? 2048 * mt : 1024) * (pro == PRO_SILU_MUL ? 2 : 1) + (lora ? 2048 : 0);
}

// TAKES: weights of a workgroup, 1 or both of two (the step of one, then the step of the other, on the same
// activations).
template <int NB, int PRO, bool LORA, bool WCM, int GROUPS, int TAKES = 1>
__device__ __forceinline__ void stream_block(StreamParams const &S) {
  GemmParams const &P = S.g;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int MT = GROUPS > 0 ? GROUPS : 1, EIGHTS = GROUPS > 0 ? 2 * GROUPS : 1;  // 16-row groups, loads of 8 rows
  constexpr int W = 4, SLOT = stream_slot_bytes(PRO, LORA, GROUPS);
  constexpr int X_LOADS = EIGHTS * (PRO == PRO_SILU_MUL ? 2 : 1) + (LORA ? 2 : 0);  // besides the weights' 8
  constexpr int X_AT = 8192, U_AT = X_AT + 1024 * EIGHTS, LA_AT = U_AT + (PRO == PRO_SILU_MUL ? 1024 * EIGHTS : 0);
  int const tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  int const g = lane / 16, c = lane % 16;
  int const M = P.M, F = P.forloop_range, subs = P.KT / 64;
  constexpr int R = kStreamRing;

  constexpr int SETS = NB / TAKES;
  int const gx = gridDim.x / (P.ksplit * SETS);
  int const ks = blockIdx.x % P.ksplit;  // (the ranges of a block next to each other)
  int const block_weight = blockIdx.x / P.ksplit, b0 = SETS == 2 ? block_weight % 2 : 0;
  int const bx = block_weight / SETS, by = blockIdx.y, bz = blockIdx.z;
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
  // rows 8 j + l8: the swizzle of rows 8 apart differs, so even and odd j
  uint32_t w_off[TAKES][2];
#pragma unroll
  for (int q = 0; q < TAKES; q++) {
    int const ld = NB == 2 && b0 + q == 1 ? P.b1.d_cols : P.b0.d_cols;
    w_off[q][0] = 2u * (uint32_t)(l8 * ld + 8 * (ch8 ^ swizzle(l8)));
    w_off[q][1] = 2u * (uint32_t)(l8 * ld + 8 * (ch8 ^ swizzle(8 + l8)));
  }
  // activation rows 8 j + l / 8 (rows past the tile re-read its last one: theirs are not stored)
  uint32_t x_off[EIGHTS], u_off[PRO == PRO_SILU_MUL ? EIGHTS : 1];
#pragma unroll
  for (int j = 0; j < EIGHTS; j++) {
    int const row = 8 * j + l8, rr = row < M ? row : M - 1;
    uint32_t const chunk = 8u * (uint32_t)(ch8 ^ ((row >> 1) & 7));
    x_off[j] = 2u * ((uint32_t)(rr * P.a0.d_cols) + chunk);
    if (PRO == PRO_SILU_MUL) {
      u_off[j] = 2u * ((uint32_t)(rr * P.a1.d_cols) + chunk);
    }
  }
  // lora A: column-major like the weights (16 columns), row-major k rows 32 j + l / 2 of 32 bytes
  auto issue = [&](int it, int sub, int q, int slot) {
    uint32_t const at = mine_at + (uint32_t)(slot * SLOT);
    GTile const &bt = NB == 2 && b0 + q == 1 ? P.b1 : P.b0;
    _Float16 const *w = static_cast<_Float16 const *>(bt.ptr) + gtile_offset(bt, bx, by, bz, it) +
                        (WCM ? (long long)(64 * sub) : (long long)(64 * sub) * bt.d_cols);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      lane_dma16(w + (long long)(8 * j) * bt.d_cols, w_off[q][j & 1], at + (uint32_t)(1024 * j));
    }
    if (q > 0) {
      return;
    }
    _Float16 const *x = static_cast<_Float16 const *>(P.a0.ptr) + gtile_offset(P.a0, bx, by, bz, it) + 64 * sub;
#pragma unroll
    for (int j = 0; j < EIGHTS; j++) {
      lane_dma16(x, x_off[j], at + (uint32_t)(X_AT + 1024 * j));
    }
    if (PRO == PRO_SILU_MUL) {
      _Float16 const *u = static_cast<_Float16 const *>(P.a1.ptr) + gtile_offset(P.a1, bx, by, bz, it) + 64 * sub;
#pragma unroll
      for (int j = 0; j < EIGHTS; j++) {
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
    int const row = GROUPS > 0 ? 16 * mt + c : c % 8;
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

  // ---- the loop: step = 64 k ----------------------------------------------------------------------
  int const total = n_mine > 0 ? n_mine * subs * TAKES : 0;
  int i_it = 0, i_sub = 0, i_q = 0, i_slot = 0, issued = 0;  // the next step to issue
  auto issue_next = [&]() {
    if (TAKES == 1 || i_q == 0) {
      issue(nth(i_it), i_sub, 0, i_slot);
    } else {
      issue(nth(i_it), i_sub, TAKES - 1, i_slot);
    }
    issued++;
    i_slot = i_slot + 1 == R ? 0 : i_slot + 1;
    if (TAKES == 2) {
      i_q ^= 1;
      if (i_q == 1) {
        return;
      }
    }
    i_sub++;
    if (i_sub == subs) {
      i_sub = 0;
      i_it++;
    }
  };
  for (int s = 0; s < R && s < total; s++) {
    issue_next();
  }
  int slot = 0, step = 0;
  for (int i = 0; i < n_mine; i++) {
    float4v o[TAKES][4][MT], d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < 4 * TAKES; t++) {
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        o[t / 4][t % 4][mt] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
    half8 x[MT][2];
    auto work = [&](auto which) {
      constexpr int q = decltype(which)::value;
      // this step has landed when only the loads of the one after it are outstanding
      if (issued - 1 > step) {
        stream_wait<q + 1 < TAKES ? 8 : 8 + X_LOADS>();
      } else {
        stream_wait<0>();
      }
      unsigned char const *const at = mine + slot * SLOT;
      half8 w[4][2], la[2], u[PRO == PRO_SILU_MUL ? MT : 1][2];
#pragma unroll
      for (int s = 0; s < 2; s++) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
          w[t][s] = weights(at, t, s);
        }
      }
#pragma unroll
      for (int s = 0; s < 2; s++) {
        if (q > 0) {
          continue;
        }
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
      // the slot is in registers: the step that takes it next may fly
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (issued < total) {
        issue_next();
      }
      slot = slot + 1 == R ? 0 : slot + 1;
      auto applied = [&](half8 v, half8 m) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
          v[e] = static_cast<_Float16>(prologue(PRO == PRO_EXP ? PRO_EXP : PRO_SILU, static_cast<float>(v[e])));
          if (PRO == PRO_SILU_MUL) {
            v[e] = static_cast<_Float16>(static_cast<float>(v[e]) * static_cast<float>(m[e]));
          }
        }
        return v;
      };
      if (PRO != PRO_NONE && GROUPS == 0) {
        // Eight rows: lanes c and c + 8 hold the same values of both k steps.  Each makes one step's and the
        // lower lane takes the other's from the upper (the upper lane's operands belong to rows that are not stored).
        bool const upper = c >= 8;
        half8 const v = applied(upper ? x[0][1] : x[0][0], upper ? u[0][PRO == PRO_SILU_MUL] : u[0][0]);
        x[0][0] = v;
        uint4v const bits = __builtin_bit_cast(uint4v, v);
        uint4v from;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          from[e] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)bits[e], 0x128, 0xf, 0xf, false);  // row_ror:8
        }
        x[0][1] = __builtin_bit_cast(half8, from);
      } else if (PRO != PRO_NONE) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
          for (int mt = 0; mt < MT; mt++) {
            x[mt][s] = applied(x[mt][s], u[PRO == PRO_SILU_MUL ? mt : 0][PRO == PRO_SILU_MUL ? s : 0]);
          }
        }
      }
      if (LORA) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(la[s], x[0][s], d, 0, 0, 0);
        }
      }
      // weights first: o[t][mt][r] = O[16 mt + c][16 t + 4 g + r]
#pragma unroll
      for (int s = 0; s < 2; s++) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
#pragma unroll
          for (int mt = 0; mt < MT; mt++) {
            o[q][t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[t][s], x[mt][s], o[q][t][mt], 0, 0, 0);
          }
        }
      }
      step++;
    };
    for (int sub = 0; sub < subs; sub++) {
      work(std::integral_constant<int, 0>{});
      if constexpr (TAKES == 2) {
        work(std::integral_constant<int, 1>{});
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
    long long const tile = (long long)M * 64;
#pragma unroll
    for (int q = 0; q < TAKES; q++) {
      _Float16 *const to = P.ksplit > 1 ? P.scratch + (((long long)block_linear * F + it) * NB + b0 + q) * tile
                                        : reinterpret_cast<_Float16 *>(lds + S.results) + (q * F + it) * (int)tile;
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        if (16 * mt + c < M) {
#pragma unroll
          for (int t = 0; t < 4; t++) {
            *reinterpret_cast<half4 *>(to + (16 * mt + c) * 64 + 16 * t + 4 * g) = __builtin_convertvector(o[q][t][mt], half4);
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
  if (TAKES == 2 && P.gate != nullptr) {  // both sums in one thread
    for (int e = tid; e < M * 16; e += 256) {
      int const row = e / 16, col = 4 * (e % 16);
      _Float16 const *src = reinterpret_cast<_Float16 const *>(lds + S.results) + row * 64 + col;
      half4 x[2];
#pragma unroll
      for (int q = 0; q < 2; q++) {
        half2v lo = {(_Float16)0.0f, (_Float16)0.0f}, hi = lo;
        for (int it = 0; it < F; it++) {
          half4 const v = *reinterpret_cast<half4 const *>(src + (q * F + it) * M * 64);
          lo += half2v{v[0], v[1]};
          hi += half2v{v[2], v[3]};
        }
        x[q] = half4{lo[0], lo[1], hi[0], hi[1]};
        GTile const &ot = q == 1 ? P.o1 : P.o0;
        _Float16 *const og = static_cast<_Float16 *>(const_cast<void *>(ot.ptr)) + gtile_offset(ot, bx, by, bz, 0);
        *reinterpret_cast<half4 *>(og + (long long)row * ot.d_cols + col) = x[q];
      }
      half4 h;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        h[j] = gate_value(x[0][j], x[1][j]);
      }
      *reinterpret_cast<half4 *>(P.gate + gtile_offset(P.o0, bx, by, bz, 0) + (long long)row * P.o0.d_cols + col) = h;
    }
    return;
  }
  for (int e = tid; e < TAKES * M * 16; e += 256) {
    int const q = TAKES == 1 || e < M * 16 ? 0 : 1, of = e - q * M * 16, row = of / 16, col = 4 * (of % 16);
    _Float16 const *src = reinterpret_cast<_Float16 const *>(lds + S.results) + q * F * M * 64 + row * 64 + col;
    half2v lo = {(_Float16)0.0f, (_Float16)0.0f}, hi = lo;
    for (int it = 0; it < F; it++) {  // (a packed fp16 add is the exact sum rounded once)
      half4 const v = *reinterpret_cast<half4 const *>(src + it * M * 64);
      lo += half2v{v[0], v[1]};
      hi += half2v{v[2], v[3]};
    }
    GTile const &ot = NB == 2 && b0 + q == 1 ? P.o1 : P.o0;
    _Float16 *const og = static_cast<_Float16 *>(const_cast<void *>(ot.ptr)) + gtile_offset(ot, bx, by, bz, 0);
    *reinterpret_cast<half4 *>(og + (long long)row * ot.d_cols + col) = half4{lo[0], lo[1], hi[0], hi[1]};
  }
}

// The same for column-major weights cut into strips of 16 columns, a workgroup with the whole for-loop each: no
// ranges to add up, so no slab and no second launch, for activations read four times as often.  Of two weights a strip
// is 8 columns of each: a workgroup then has both sums of a gated MLP and can make what its second product takes.
// Bound by memory: two weights of 4096 x 14336 against 8 rows 42.9 us, ranges and their fold 47.2;
// against 16 rows, and with a gated MLP's second product behind it, 79.5 against 82.5.  (With strips of 16 of one of
// them a pair of workgroups took 42.8 us, with 8 of each and SiLU(a) * u 43.8, and the second product 25.2 instead of 29.4.)
// A LoRA's A, 16 columns too, goes through the ring with every strip: 8 rows x 4096 x 4096 8.0 us, ranges and fold 11.1.
// Slots per wavefront: for two workgroups on a compute unit.
constexpr int columns_ring(int eights, bool lora) { return eights == 1 ? (lora ? 4 : 6) : (lora ? 3 : 4); }
constexpr int columns_slot_bytes(int eights, bool lora) { return 2048 + 1024 * eights + (lora ? 2048 : 0); }

template <int NB, int EIGHTS, bool LORA>
__device__ __forceinline__ void stream_columns(StreamParams const &S) {
  GemmParams const &P = S.g;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int W = 4, R = columns_ring(EIGHTS, LORA), SLOT = columns_slot_bytes(EIGHTS, LORA);
  constexpr int LOADS = 2 + EIGHTS + (LORA ? 2 : 0), LA_AT = 2048 + 1024 * EIGHTS;
  static_assert((R - 1) * LOADS < 64 && !(LORA && NB == 2), "loads in flight are counted in six bits");
  int const tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  int const g = lane / 16, c = lane % 16, l8 = lane / 8, ch8 = lane % 8;
  int const M = P.M, F = P.forloop_range, subs = P.KT / 64;
  constexpr int WIDE = 16 / NB;  // columns of a weight
  int const piece = blockIdx.x % (4 * NB);
  int const bx = blockIdx.x / (4 * NB), by = blockIdx.y, bz = blockIdx.z;
  // A wavefront's iterations are neighbours, and it starts at another one in each block: wavefronts on every
  // fourth iteration read 2 KB next to each other in columns 8 KB apart, all of them the same few memory channels
  // (4 rows x 28672 x 4096: 50.5 us, 39.9 this way).
  int const per = (F + W - 1) / W, first = wave * per;
  int const n_mine = F - first < per ? (F > first ? F - first : 0) : per, total = n_mine * subs;
  int const rot = n_mine > 1 ? (int)(blockIdx.x / (4 * NB) % (unsigned)n_mine) : 0;

  unsigned char *const mine = lds + wave * R * SLOT;
  uint32_t const mine_at = lane_lds_address(mine);
  auto swizzle = [](int row) { return (row >> 1) & 7; };
  uint32_t w_off[2], x_off[EIGHTS], la_off[2];
#pragma unroll
  for (int j = 0; j < 2; j++) {  // (rows 8 - 15 of the LDS tile: the columns behind, or the other weight's)
    int const ld = NB == 2 && j == 1 ? P.b1.d_cols : P.b0.d_cols;
    w_off[j] = 2u * (uint32_t)((NB == 2 ? l8 : 8 * j + l8) * ld + 8 * (ch8 ^ swizzle(8 * j + l8)));
  }
#pragma unroll
  for (int j = 0; j < 2; j++) {  // (lora A: 16 columns as well)
    la_off[j] = LORA ? 2u * (uint32_t)((8 * j + l8) * P.la.d_cols + 8 * (ch8 ^ swizzle(8 * j + l8))) : 0u;
  }
#pragma unroll
  for (int j = 0; j < EIGHTS; j++) {
    int const row = 8 * j + l8;
    x_off[j] = 2u * (uint32_t)((row < M ? row : M - 1) * P.a0.d_cols + 8 * (ch8 ^ swizzle(row)));
  }
  int i_it = rot, i_sub = 0, i_slot = 0, issued = 0;  // the next step to issue
  auto issue_next = [&]() {
    int const it = first + i_it;
    uint32_t const at = mine_at + (uint32_t)(i_slot * SLOT);
    auto weight = [&](GTile const &bt) {
      return static_cast<_Float16 const *>(bt.ptr) + gtile_offset(bt, bx, by, bz, it) + (long long)(WIDE * piece) * bt.d_cols + 64 * i_sub;
    };
    _Float16 const *x = static_cast<_Float16 const *>(P.a0.ptr) + gtile_offset(P.a0, bx, by, bz, it) + 64 * i_sub;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      lane_dma16(weight(NB == 2 && j == 1 ? P.b1 : P.b0), w_off[j], at + (uint32_t)(1024 * j));
    }
#pragma unroll
    for (int j = 0; j < EIGHTS; j++) {
      lane_dma16(x, x_off[j], at + (uint32_t)(2048 + 1024 * j));
    }
    if (LORA) {
      _Float16 const *la = static_cast<_Float16 const *>(P.la.ptr) + gtile_offset(P.la, bx, by, bz, it) + 64 * i_sub;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        lane_dma16(la, la_off[j], at + (uint32_t)(LA_AT + 1024 * j));
      }
    }
    issued++;
    i_slot = i_slot + 1 == R ? 0 : i_slot + 1;
    i_sub++;
    if (i_sub == subs) {
      i_sub = 0;
      i_it = i_it + 1 == n_mine ? 0 : i_it + 1;
    }
  };
  half4 lb_frag;  // lora B[4 g ..][16 piece + c], loop invariant
  if (LORA) {
    lb_frag = *reinterpret_cast<half4 const *>(static_cast<_Float16 const *>(P.lb.ptr) + gtile_offset(P.lb, bx, by, bz, 0) +
                                               (long long)(16 * piece + c) * P.lb.d_cols + 4 * g);
    stream_wait<0>();  // (before the counted loads begin)
    asm volatile("" : "+v"(lb_frag));
  }
  for (int s = 0; s < R && s < total; s++) {
    issue_next();
  }
  _Float16 *const all = reinterpret_cast<_Float16 *>(lds + S.results);  // [F][M][16]
  int slot = 0, step = 0;
  for (int i = 0; i < n_mine; i++) {
    float4v o = {0.0f, 0.0f, 0.0f, 0.0f}, d = o;
    for (int sub = 0; sub < subs; sub++, step++) {
      if (issued - step == R) {
        stream_wait<(R - 1) * LOADS>();
      } else {
        stream_wait<0>();
      }
      unsigned char const *const at = mine + slot * SLOT;
      int const xr = EIGHTS == 2 ? c : c % 8;
      half8 w[2], x[2], la[2];
#pragma unroll
      for (int s = 0; s < 2; s++) {
        w[s] = *reinterpret_cast<half8 const *>(at + 128 * c + 16 * ((4 * s + g) ^ swizzle(c)));
        x[s] = *reinterpret_cast<half8 const *>(at + 2048 + 128 * xr + 16 * ((4 * s + g) ^ swizzle(xr)));
        if (LORA) {
          la[s] = *reinterpret_cast<half8 const *>(at + LA_AT + 128 * c + 16 * ((4 * s + g) ^ swizzle(c)));
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (issued < total) {
        issue_next();
      }
      slot = slot + 1 == R ? 0 : slot + 1;
#pragma unroll
      for (int s = 0; s < 2; s++) {
        if (LORA) {
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(la[s], x[s], d, 0, 0, 0);
        }
        o = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[s], x[s], o, 0, 0, 0);
      }
    }
    if (LORA) {  // + [X.A] . B, as in stream_block
      half4 const df = {(_Float16)d[0], (_Float16)d[1], (_Float16)d[2], (_Float16)d[3]};
      o = __builtin_amdgcn_mfma_f32_16x16x16f16(lb_frag, df, o, 0, 0, 0);
    }
    int const j = i + rot, it = first + (j >= n_mine ? j - n_mine : j);
    if (c < M) {
      *reinterpret_cast<half4 *>(all + (it * M + c) * 16 + 4 * g) = __builtin_convertvector(o, half4);
    }
  }
  __syncthreads();
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  if (tid < 8 * M) {
    int const row = tid / 8, col = 2 * (tid % 8);
    half2v a = {(_Float16)0.0f, (_Float16)0.0f};
#pragma unroll 8
    for (int it = 0; it < F; it++) {  // (a packed fp16 add is the exact sum rounded once)
      a += *reinterpret_cast<half2v const *>(all + (it * M + row) * 16 + col);
    }
    bool const second = NB == 2 && col >= 8;
    GTile const &ot = second ? P.o1 : P.o0;
    _Float16 *const og = static_cast<_Float16 *>(const_cast<void *>(ot.ptr)) + gtile_offset(ot, bx, by, bz, 0);
    *reinterpret_cast<half2v *>(og + (long long)row * ot.d_cols + WIDE * piece + (second ? col - 8 : col)) = a;
    if (NB == 2 && P.gate != nullptr) {
      half2v const u = __builtin_bit_cast(half2v, __shfl_xor(__builtin_bit_cast(int, a), 4, 64));  // the other weight's columns
      if (!second) {
        *reinterpret_cast<half2v *>(P.gate + gtile_offset(P.o0, bx, by, bz, 0) + (long long)row * P.o0.d_cols + WIDE * piece + col) =
            half2v{gate_value(a[0], u[0]), gate_value(a[1], u[1])};
      }
    }
  }
}

template <int NB, int PRO, bool LORA, bool WCM, int MT>
__global__ __launch_bounds__(256) void gemm_stream_kernel(StreamParams const S) {
  fetch_kernel_arguments<sizeof(StreamParams), 2>();
  if constexpr (PRO == PRO_NONE && WCM && MT == 1) {
    if (S.strips) {
      if (S.g.M <= 8) {
        stream_columns<NB, 1, LORA>(S);
      } else {
        stream_columns<NB, 2, LORA>(S);
      }
      return;
    }
  }
  if (MT == 1 && S.g.M <= 8) {
    stream_block<NB, PRO, LORA, WCM, 0>(S);
  } else {
    stream_block<NB, PRO, LORA, WCM, MT>(S);
  }
}

// Both of two weights in a workgroup (a kernel of its own: with the forms above in one, its addresses do not fit the
// scalar registers).
template <bool WCM, int GROUPS>
__global__ __launch_bounds__(256) void gemm_stream_pairs_kernel(StreamParams const S) {
  fetch_kernel_arguments<sizeof(StreamParams), 2>();
  stream_block<2, PRO_NONE, false, WCM, GROUPS, 2>(S);
}

}  // namespace mi355
