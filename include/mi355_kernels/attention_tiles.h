// attn_tiles_kernel: the attention family of thread-block graphs at any tile size (query tiles of
// any number of rows, key tiles of any multiple of 16, head sizes 64 and 128, keys and values in
// either storage order).  The kernels of attention.h are built for whole tiles of 64 keys and 16
// rows; what they do not take runs here, register-resident as well, instead of statement by
// statement in the generic LDS interpreter.
//
// A workgroup owns 16 RPW query rows and walks the for-loop in rounds: wavefront ip of IP takes
// iteration r0 + ip by itself, K and V operands going from global memory into its registers (an
// MFMA operand of a column-major tile IS sixteen contiguous bytes per lane; a row-major tile takes
// one trip through a private strip of LDS and a transposing read), and leaves the iteration's fp16
// result in an LDS slot of its own.  After one barrier all threads add the round's slots to
// their registers in ITERATION order with one fp16 rounding per add, the sequence of roundings of
// the sequential loop (reference src/kernel/triton_code_gen.cc:223-232).  Slots are double
// buffered, so a round costs one barrier.
//
// What bounds it: the trip to memory at decode sizes (a wavefront issues all of an iteration's
// loads before it waits for the first), the conversions and exponentials beside the matrix
// instructions at prefill sizes.  Two row groups share every K and V operand where there are enough
// of them, which halves the L2 -> register traffic of a prefill.
// Keys of a pair of 16-key blocks are permuted as in attention.h (see cm_swizzle_key) so that a
// lane's eight values of P are consecutive keys; a lone last block keeps the plain order and takes
// the 16 x 16 x 16 instruction.
#pragma once

#include "attention.h"

namespace mi355 {

// CHB: 16-key blocks of K and V held in registers at a time.  A longer key tile is walked in chunks
// of CHB blocks; the form with the division needs the whole tile's row sum first, so its tile is
// one chunk (the host checks).  AttnParams as used here: rows = query rows of a block, stages =
// keys of a tile, lds_stage_bytes unused.
// Most iteration lanes of a workgroup: eight where 256 registers hold a wavefront's operands.
constexpr int attn_tiles_lanes(int D, int RPW, int CHB) { return RPW == 1 && CHB <= 4 && D == 64 ? 8 : 4; }

template <int D, bool HAS_DIV, bool CM, int RPW, int CHB>
__global__ __launch_bounds__(attn_tiles_lanes(D, RPW, CHB) * 64) void attn_tiles_kernel(AttnParams const) {
  AttnParams const P = load_kernel_arguments<AttnParams, 4>();  // (blockDim.x is read)
  constexpr int DV = D, DB = DV / 16, DK = D / 32, PAIRS = CHB / 2;
  constexpr int ROWS = 16 * RPW, LDO = DV + 8, SLOT = ROWS * LDO + ROWS;
  constexpr int CPR = DV / 8;                // 16-byte chunks of a result row
  constexpr int OWN = ROWS * CPR / 64;       // most chunks a thread adds up (one wavefront)
  constexpr int KLD = 40, VLD = DV + 8;      // row strides of the row-major staging strips
  static_assert(CHB % 2 == 0 && (D == 64 || D == 128), "pairs of key blocks, head size 64 or 128");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int const tid = threadIdx.x, NT = blockDim.x, IP = NT / 64;
  int const lane = tid % 64, ip = __builtin_amdgcn_readfirstlane(tid / 64);
  int const g = lane / 16, c = lane % 16, a4 = c >> 2, b4 = c & 3;
  int bx, by, bz, slice;
  decode_block(P, bx, by, bz, slice);
  int const row_base = slice * ROWS, m = P.rows, nb = P.stages / 16, F = P.forloop_range;
  int const nchunks = HAS_DIV ? 1 : (nb + CHB - 1) / CHB;
  _Float16 *const slots = reinterpret_cast<_Float16 *>(lds);  // [1 or 2][IP][SLOT]
  _Float16 *const k_strip = slots + (F > IP ? 2 : 1) * IP * SLOT + ip * (D * KLD + 32 * VLD);
  _Float16 *const v_strip = k_strip + D * KLD;

  // ---- loads -------------------------------------------------------------------------------
  // K of chunk `ch` of iteration `it`.  Column-major: the operands of S^T.  Row-major: the pair's
  // [D][32 keys] strip as 16-byte chunks, lane by lane (a lone block: [D][16 keys]).
  uint4v kr[CHB][DK];
  auto load_k = [&](int it, int ch) {
    int const ld = P.k.d_cols, nbc = (nb - ch * CHB) < CHB ? (nb - ch * CHB) : CHB;
    _Float16 const *kg = static_cast<_Float16 const *>(P.k.ptr) + tile_offset(P.k, bx, by, bz, it) +
                         (CM ? (long long)(16 * CHB * ch) * ld : (long long)(16 * CHB * ch));
#pragma unroll
    for (int p = 0; p < PAIRS; p++) {
      // (one path for pairs and lone blocks, offsets selected: the registers keep fixed places)
      bool const lone = 2 * p + 1 >= nbc;
      int const k_row = CM ? (lone ? c : 8 * a4 + b4) : (lone ? lane / 2 : lane / 4);
      int const k_pos = CM ? 8 * g : 8 * (lone ? lane % 2 : lane % 4);
#pragma unroll
      for (int i = 0; i < 2 * DK; i++) {
        if (2 * p + (i < DK ? 0 : 1) < nbc) {
          int const off = CM ? (32 * p + 4 * (i / DK) + k_row) * ld + 32 * (i % DK) + k_pos
                             : ((lone ? 32 * i : 16 * i) + k_row) * ld + 32 * p + k_pos;
          kr[2 * p + i / DK][i % DK] = *reinterpret_cast<uint4v const *>(kg + off);
        }
      }
    }
  };
  // V likewise: column-major V^T[16t + c][32p + 8g ..] (a lone block: keys 8 (g / 2) .., of which the
  // lane uses the half 4 (g % 2) ..), row-major the [32 keys][DV] strip
  uint4v vr[PAIRS][DB];
  auto load_v = [&](int it, int ch) {
    int const ld = P.v.d_cols, nbc = (nb - ch * CHB) < CHB ? (nb - ch * CHB) : CHB;
    _Float16 const *vg = static_cast<_Float16 const *>(P.v.ptr) + tile_offset(P.v, bx, by, bz, it) +
                         (CM ? (long long)(16 * CHB * ch) : (long long)(16 * CHB * ch) * ld);
#pragma unroll
    for (int p = 0; p < PAIRS; p++) {
      bool const lone = 2 * p + 1 >= nbc;
      int const v_pos = 8 * (lone ? g / 2 : g);
#pragma unroll
      for (int t = 0; t < DB; t++) {
        if (2 * p + (CM || t < DB / 2 ? 0 : 1) < nbc) {
          int const q = 64 * t + lane;
          int const off = CM ? (16 * t + c) * ld + 32 * p + v_pos : (32 * p + q / CPR) * ld + 8 * (q % CPR);
          vr[p][t] = *reinterpret_cast<uint4v const *>(vg + off);
        }
      }
    }
  };

  // Q fragments: Q[row c][32kk + 8g .. +7] (rows past the tile re-read its last one: every row is
  // worked on by itself and theirs are not stored)
  half8 qf[RPW][DK];
  {
    _Float16 const *q = static_cast<_Float16 const *>(P.q.ptr) + tile_offset(P.q, bx, by, bz, 0);
#pragma unroll
    for (int rp = 0; rp < RPW; rp++) {
      int const row = row_base + 16 * rp + c;
      _Float16 const *qr = q + (long long)(row < m ? row : m - 1) * P.q.d_cols + 8 * g;
#pragma unroll
      for (int kk = 0; kk < DK; kk++) {
        qf[rp][kk] = *reinterpret_cast<half8 const *>(qr + 32 * kk);
      }
    }
  }
  if (ip < F) {
    load_k(ip, 0);
  }
  half2v acc[OWN][4];  // this thread's chunks of the result (fp16 sums)
#pragma unroll
  for (int i = 0; i < OWN; i++) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      acc[i][e] = half2v{(_Float16)0.0f, (_Float16)0.0f};
    }
  }
  _Float16 racc = (_Float16)0.0f;  // row sum of row `tid`
  half2v const ones = {(_Float16)1.0f, (_Float16)1.0f};
  constexpr float LOG2E = 1.44269504088896340736f;

  int buf = 0;
  for (int r0 = 0; r0 < F; r0 += IP, buf ^= 1) {
    int const it = r0 + ip;
    _Float16 *const round = slots + buf * IP * SLOT;
    if (it < F) {
      float4v o[RPW][DB];
      float rs[RPW];
#pragma unroll
      for (int rp = 0; rp < RPW; rp++) {
        rs[rp] = 0.0f;
#pragma unroll
        for (int t = 0; t < DB; t++) {
          o[rp][t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
      for (int ch = 0; ch < nchunks; ch++) {
        int const nbc = (nb - ch * CHB) < CHB ? (nb - ch * CHB) : CHB;
        load_v(it, ch);
        // ---- S^T = K^T . Q^T, exp, row sums: S to fp16, exp in fp32, the result to fp16; the
        // row sum adds the rounded values in fp32
        uint32_t pk[RPW][PAIRS][4];
#pragma unroll
        for (int p = 0; p < PAIRS; p++) {
          if (2 * p < nbc) {
            bool const lone = 2 * p + 1 >= nbc;
            if (!CM) {
              if (!lone) {
#pragma unroll
                for (int i = 0; i < 2 * DK; i++) {
                  *reinterpret_cast<uint4v *>(k_strip + (16 * i + lane / 4) * KLD + 8 * (lane % 4)) = kr[2 * p + i / DK][i % DK];
                }
              } else {
#pragma unroll
                for (int i = 0; i < DK; i++) {
                  *reinterpret_cast<uint4v *>(k_strip + (32 * i + lane / 2) * KLD + 8 * (lane % 2)) = kr[2 * p][i];
                }
              }
              asm volatile("" ::: "memory");  // (a wavefront's LDS operations complete in order)
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
              if (j == 0 || !lone) {
                float4v s[RPW];
#pragma unroll
                for (int rp = 0; rp < RPW; rp++) {
                  s[rp] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
                }
#pragma unroll
                for (int kk = 0; kk < DK; kk++) {
                  half8 a;
                  if (CM) {
                    a = __builtin_bit_cast(half8, kr[2 * p + j][kk]);
                  } else {
                    _Float16 const *ka = k_strip + (32 * kk + 8 * g + a4) * KLD + 16 * j + 4 * b4;
                    half4 const lo = lds_read_tr16(ka), hi = lds_read_tr16(ka + 4 * KLD);
                    a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                  }
#pragma unroll
                  for (int rp = 0; rp < RPW; rp++) {
                    s[rp] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qf[rp][kk], s[rp], 0, 0, 0);
                  }
                }
#pragma unroll
                for (int rp = 0; rp < RPW; rp++) {
#pragma unroll
                  for (int h = 0; h < 2; h++) {
                    half2v const s2 = __builtin_convertvector(float2v{s[rp][2 * h], s[rp][2 * h + 1]}, half2v);
                    float2v const x2 = {__builtin_amdgcn_exp2f(__builtin_fmaf(static_cast<float>(s2[0]), LOG2E, 0.0f)),
                                        __builtin_amdgcn_exp2f(__builtin_fmaf(static_cast<float>(s2[1]), LOG2E, 0.0f))};
                    half2v const e2 = __builtin_convertvector(x2, half2v);
                    rs[rp] = __builtin_amdgcn_fdot2(e2, ones, rs[rp], false);
                    pk[rp][p][2 * j + h] = __builtin_bit_cast(uint32_t, e2);
                  }
                }
              }
            }
            asm volatile("" ::: "memory");
          }
        }
        // the next chunk's K (this iteration's or the next round's) flies under the rest
        if (ch + 1 < nchunks) {
          load_k(it, ch + 1);
        } else if (it + IP < F) {
          load_k(it + IP, 0);
        }
        if (ch == nchunks - 1) {
#pragma unroll
          for (int rp = 0; rp < RPW; rp++) {
            rs[rp] = sum_lane_groups(rs[rp]);
            if (HAS_DIV) {
              // E / sum, rounded to fp32 and then to fp16 as the division is: the reciprocal's product with one
              // correction is the nearest fp32 number.  (Without it quotients below 2^-14 came out one unit
              // off where they lie next to the middle of two fp16 numbers.  An infinite sum: 0, or no number
              // where E is infinite too; E is finite under a finite sum.)
              float const sum = static_cast<float>(static_cast<_Float16>(rs[rp])), inv = __builtin_amdgcn_rcpf(sum);
              float const by = __builtin_isinf(sum) ? 0.0f : -sum;
              auto quotient = [&](_Float16 e) {
                float q = __builtin_fmaf(static_cast<float>(e), inv, 0.0f);
                q = __builtin_fmaf(__builtin_fmaf(by, q, static_cast<float>(e)), inv, q);
                asm volatile("" : "+v"(q));  // (fused with the conversion the last step would round once)
                return static_cast<_Float16>(q);
              };
#pragma unroll
              for (int p = 0; p < PAIRS; p++) {
#pragma unroll
                for (int w = 0; w < 4; w++) {
                  // (slots of blocks that do not exist hold anything and are never multiplied)
                  half2v const e2 = __builtin_bit_cast(half2v, pk[rp][p][w]);
                  half2v const p2 = {quotient(e2[0]), quotient(e2[1])};
                  pk[rp][p][w] = __builtin_bit_cast(uint32_t, p2);
                }
              }
            }
          }
        }
        // ---- O += P . V, V^T first: o[rp][t][r] = O[row c][16t + 4g + r]
#pragma unroll
        for (int p = 0; p < PAIRS; p++) {
          if (2 * p + 1 < nbc) {
            if (!CM) {
#pragma unroll
              for (int t = 0; t < DB; t++) {
                int const q = 64 * t + lane;
                *reinterpret_cast<uint4v *>(v_strip + (q / CPR) * VLD + 8 * (q % CPR)) = vr[p][t];
              }
              asm volatile("" ::: "memory");
            }
#pragma unroll
            for (int t = 0; t < DB; t++) {
              half8 b;
              if (CM) {
                b = __builtin_bit_cast(half8, vr[p][t]);
              } else {
                _Float16 const *vb = v_strip + (4 * g + a4) * VLD + 16 * t + 4 * b4;
                half4 const lo = lds_read_tr16(vb), hi = lds_read_tr16(vb + 16 * VLD);
                b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
              }
#pragma unroll
              for (int rp = 0; rp < RPW; rp++) {
                uint4v const a = {pk[rp][p][0], pk[rp][p][1], pk[rp][p][2], pk[rp][p][3]};
                o[rp][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, __builtin_bit_cast(half8, a), o[rp][t], 0, 0, 0);
              }
            }
            asm volatile("" ::: "memory");
          } else if (2 * p < nbc) {
            if (!CM) {
#pragma unroll
              for (int t = 0; t < DB / 2; t++) {
                int const q = 64 * t + lane;
                *reinterpret_cast<uint4v *>(v_strip + (q / CPR) * VLD + 8 * (q % CPR)) = vr[p][t];
              }
              asm volatile("" ::: "memory");
            }
#pragma unroll
            for (int t = 0; t < DB; t++) {
              half4 b;
              if (CM) {
                b = __builtin_bit_cast(half4, (g & 1) ? uint2v{vr[p][t].z, vr[p][t].w} : uint2v{vr[p][t].x, vr[p][t].y});
              } else {
                b = lds_read_tr16(v_strip + (4 * g + a4) * VLD + 16 * t + 4 * b4);
              }
#pragma unroll
              for (int rp = 0; rp < RPW; rp++) {
                uint2v const a = {pk[rp][p][0], pk[rp][p][1]};
                o[rp][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(b, __builtin_bit_cast(half4, a), o[rp][t], 0, 0, 0);
              }
            }
            asm volatile("" ::: "memory");
          }
        }
      }
      // ---- this iteration's result, fp16, to its slot
      _Float16 *const slot = round + ip * SLOT;
#pragma unroll
      for (int rp = 0; rp < RPW; rp++) {
#pragma unroll
        for (int t = 0; t < DB; t++) {
          half2v const lo = __builtin_convertvector(float2v{o[rp][t][0], o[rp][t][1]}, half2v);
          half2v const hi = __builtin_convertvector(float2v{o[rp][t][2], o[rp][t][3]}, half2v);
          uint2v const w = {__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
          *reinterpret_cast<uint2v *>(slot + (16 * rp + c) * LDO + 16 * t + 4 * g) = w;
        }
        if (!HAS_DIV && g == 0) {
          slot[ROWS * LDO + 16 * rp + c] = static_cast<_Float16>(rs[rp]);
        }
      }
    }
    __syncthreads();
    // ---- the round's results in iteration order, one fp16 rounding per add (a packed fp16 add
    // is the exact sum rounded once)
    int const n = (F - r0) < IP ? (F - r0) : IP;
#pragma unroll
    for (int i = 0; i < OWN; i++) {
      int const e = tid + i * NT;
      if (e < ROWS * CPR) {
        _Float16 const *src = round + (e / CPR) * LDO + 8 * (e % CPR);
        for (int u = 0; u < n; u++) {
          uint4v const v = *reinterpret_cast<uint4v const *>(src + u * SLOT);
#pragma unroll
          for (int w = 0; w < 4; w++) {
            uint32_t const x = v[w];  // (a bit cast of a vector element itself would read element 0)
            acc[i][w] = acc[i][w] + __builtin_bit_cast(half2v, x);
          }
        }
      }
    }
    if (!HAS_DIV && tid < ROWS) {
      for (int u = 0; u < n; u++) {
        racc = racc + round[u * SLOT + ROWS * LDO + tid];
      }
    }
  }

  _Float16 *const og = static_cast<_Float16 *>(const_cast<void *>(P.o.ptr)) + tile_offset(P.o, bx, by, bz, 0);
#pragma unroll
  for (int i = 0; i < OWN; i++) {
    int const e = tid + i * NT, row = row_base + e / CPR;
    if (e < ROWS * CPR && row < m) {
      uint4v const w = {__builtin_bit_cast(uint32_t, acc[i][0]), __builtin_bit_cast(uint32_t, acc[i][1]),
                        __builtin_bit_cast(uint32_t, acc[i][2]), __builtin_bit_cast(uint32_t, acc[i][3])};
      *reinterpret_cast<uint4v *>(og + (long long)row * P.o.d_cols + 8 * (e % CPR)) = w;
    }
  }
  if (!HAS_DIV && tid < ROWS && row_base + tid < m) {
    _Float16 *const rg = static_cast<_Float16 *>(const_cast<void *>(P.r.ptr)) + tile_offset(P.r, bx, by, bz, 0);
    rg[(long long)(row_base + tid) * P.r.d_cols] = racc;
  }
}

}  // namespace mi355
