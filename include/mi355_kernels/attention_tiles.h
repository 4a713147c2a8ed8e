// attn_tiles_kernel: the attention family of thread-block graphs at any tile size (query tiles of
// any number of rows, key tiles of any multiple of 16, head sizes 64 and 128, keys and values in
// either storage order).  The kernels of attention.h are built for whole tiles of 64 keys and 16
// rows; what they do not take runs here, register-resident as well, instead of statement by
// statement in the generic LDS interpreter.
//
// A workgroup owns 16 RPW query rows and walks the for-loop in rounds: wavefront ip of IP takes
// iteration r0 + ip by itself and leaves its fp16 result in LDS.  After one barrier all threads add the
// round's results up in ITERATION order with one fp16 rounding per add, the sequence of roundings of the
// sequential loop (reference src/kernel/triton_code_gen.cc:223-232); after another the next round may write.
//
// K and V go pair by pair of 16-key blocks from memory into registers, in the order they have in memory, and
// from there through a strip of LDS of the wavefront's own (with a transposing read where the reduction index
// is not the contiguous one); the strip is also where the iteration's result ends.  An operand of a
// column-major tile IS sixteen contiguous bytes per lane, but sixteen lanes in a row are then sixteen rows,
// and a compute unit gets 16 bytes a cycle that way against 59 in memory order.
//
// What bounds it: the trip to memory at decode sizes, at prefill sizes latency and the conversions and
// exponentials beside the matrix instructions (so: four wavefronts of a SIMD have registers, which is why
// sums between rounds wait in LDS).  Two row groups share every K and V operand where there are enough of
// them, which halves the L2 -> register traffic of a prefill.  With operands straight from memory, a tile's keys
// in registers at once and workgroups of an XCD from anywhere, both launches of [12, 1040, 1040] in tiles
// of 80 took 24.6 us column-major and 35.5 row-major, now 18.8 and 19.3; head size 128, [16, 1024, 1008] in
// tiles of 128 x 48, 59.5 and 37.5; [64, 1, 16384] in tiles of 64 65.9 and 50.7.
#pragma once

#include <type_traits>

#include "attention.h"

namespace mi355 {

// Keys of a pair of 16-key blocks are permuted as in attention.h (see cm_swizzle_key) so that a lane's
// eight values of P are consecutive keys; a lone last block is a pair whose second half counts for nothing.
// AttnParams as used here: rows = query rows of a block, stages = keys of a tile, lds_stage_bytes unused.
// PAIRS: with the division, which needs the whole tile's row sum before P . V, the pairs of a tile, whose
// exponentials stay in registers (the host checks); 0 without it, the pairs then go through one by one.
// Most iteration lanes of a workgroup: eight where four wavefronts of a SIMD have registers.
constexpr int attn_tiles_lanes(int D, int PAIRS) { return D == 64 && PAIRS <= 2 ? 8 : 4; }
// Halfs of a wavefront's strip: 32 keys of K or V as rows of D elements (pitch D + 8) or of 32 keys (pitch
// 40), or an iteration's result: 16 RPW rows of the same pitch and their sums.
constexpr int attn_tiles_strip(int D, int RPW) {
  int const keys = D * 40 > 32 * (D + 8) ? D * 40 : 32 * (D + 8), result = 16 * RPW * (D + 8) + 16 * RPW;
  return keys > result ? keys : result;
}

// Bytes of LDS of a workgroup: the strips, and the sums between rounds.
constexpr int attn_tiles_lds(int D, int RPW, int ip, int rounds) {
  return 2 * (ip * attn_tiles_strip(D, RPW) + (rounds > 1 ? 16 * RPW * (D + 8) + 16 * RPW : 0));
}

// Everything in memory is named as global memory.  Addresses out of the parameter block are generic to the
// compiler, whose flat loads count with a wavefront's LDS operations as well: every read of the strip then waited
// for the loads ahead of their use, those after the last round too.  Us on the device, flat and global, one operator
// with the division: 2 groups of 33 rows, 9 blocks of 8 tiles of 16 keys, row-major, 3.95 and 3.59; 8 of 40, 4 of 16,
// 5.59 and 5.04; tiles of 80 keys, column-major, 10.87 and 9.72.  (Without strips, each
// load straight to its operand: 3.25, 4.20 and 14.42; a lone block is worked on here as half of a pair.)
typedef __attribute__((address_space(1))) uint4v global_chunk;

template <int D, bool HAS_DIV, bool CM, int RPW, int PAIRS, class Params = AttnParams>
__global__ __launch_bounds__(attn_tiles_lanes(D, PAIRS) * 64)
    __attribute__((amdgpu_waves_per_eu(attn_tiles_lanes(D, PAIRS) == 8 ? 4 : 1))) void attn_tiles_kernel(Params const) {
  AttnParams const P = load_kernel_arguments<AttnParams, 4, (int)sizeof(Params)>();  // (blockDim.x is read)
  constexpr int DB = D / 16, DK = D / 32, ROWS = 16 * RPW, LD = D + 8, KLD = 40;  // pitches of rows of D and of keys
  constexpr int CPR = D / 8;                // 16-byte chunks of a row
  constexpr int CHUNKS = D / 16, KEYS = 64 / CPR;  // chunks a lane holds of a pair; keys per chunk of a wavefront
  constexpr int STRIP = attn_tiles_strip(D, RPW);
  static_assert((D == 64 || D == 128) && HAS_DIV == (PAIRS > 0), "head size 64 or 128");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int const tid = threadIdx.x, NT = blockDim.x, IP = NT / 64;
  int const lane = tid % 64, ip = __builtin_amdgcn_readfirstlane(tid / 64);
  int const g = lane / 16, c = lane % 16, a4 = c >> 2, b4 = c & 3;
  int bx, by, bz, slice;
  decode_block(P, bx, by, bz, slice);
  int const row_base = slice * ROWS, m = P.rows, nb = P.stages / 16, F = P.forloop_range;
  int const pairs = HAS_DIV ? PAIRS : (nb + 1) / 2;
  bool const odd = nb % 2 != 0;  // the last pair is a lone block
  // a wavefront's LDS: its strip, and the result of its iteration once the strip is done with
  _Float16 *const all = reinterpret_cast<_Float16 *>(lds), *const strip = all + ip * STRIP;
  _Float16 *const sums = all + IP * STRIP;  // [ROWS][LD], the row sums: with more than one round

  // ---- loads and their way into the strip ----------------------------------------------------
  // 32 keys of K or V lie in memory as rows of D elements (`by_key`: K column-major, V row-major) or as D
  // rows of 32 keys; lane l takes the 16-byte chunk l of what follows each other.  Of a lone block the first
  // half is read twice: the loads are always the same number.
  // Of the operand that has 32 keys in a row two pairs are loaded together where registers allow (DEPTH): the
  // 64 bytes of a row that a pair is are half a line, and a line fetched in two halves at different times
  // costs memory twice ([64 groups, 16384 keys] 86 us instead of 61).
  constexpr int DEPTH = !HAS_DIV && RPW == 1 ? 2 : 1, KS = CM ? 1 : DEPTH, VS = CM ? DEPTH : 1;
  uint4v kr[KS][CHUNKS], vr[VS][CHUNKS];
  auto load = [&](bool by_key, _Float16 const *from, int ld, bool lone, uint4v (&to)[CHUNKS]) {
    char const *const at = reinterpret_cast<char const *>(from);
    int const row = by_key ? lane / CPR : lone ? lane / 2 : lane / 4, pos = by_key ? lane % CPR : lone ? lane % 2 : lane % 4;
    uint32_t const off = 2u * (uint32_t)(row * ld + 8 * pos);
    long long const step = 2LL * (by_key ? KEYS : lone ? 32 : 16) * ld;
#pragma unroll
    for (int i = 0; i < CHUNKS; i++) {
      to[i] = *(global_chunk const *)(at + (i < CHUNKS / 2 ? i : lone ? i - CHUNKS / 2 : i) * step + off);
    }
  };
  auto load_k = [&](int slot, int it, int p) {
    _Float16 const *const tile = static_cast<_Float16 const *>(P.k.ptr) + tile_offset(P.k, bx, by, bz, it);
    load(CM, tile + (CM ? (long long)(32 * p) * P.k.d_cols : 32 * p), P.k.d_cols, odd && p == pairs - 1, kr[slot]);
  };
  auto load_v = [&](int slot, int it, int p) {
    _Float16 const *const tile = static_cast<_Float16 const *>(P.v.ptr) + tile_offset(P.v, bx, by, bz, it);
    load(!CM, tile + (CM ? 32 * p : (long long)(32 * p) * P.v.d_cols), P.v.d_cols, odd && p == pairs - 1, vr[slot]);
  };
  // (Places in the strip are one number per lane plus constants.)  K by keys: key 8 a + 4 j + b at row
  // 16 j + 4 a + b, which makes a lane's eight scores consecutive keys.
  _Float16 *const key_at = strip + lane / CPR * LD + 8 * (lane % CPR);
  _Float16 *const turned_at = D == 64 ? strip + (16 * (lane / 32) + lane / 8 % 4) * LD + 8 * (lane % 8) : key_at;
  _Float16 *const pair_at = strip + lane / 4 * KLD + 8 * (lane % 4), *const lone_at = strip + lane / 2 * KLD + 8 * (lane % 2);
  auto stage_k = [&](int slot, bool lone) {
#pragma unroll
    for (int i = 0; i < CHUNKS; i++) {
      if (CM) {
        *reinterpret_cast<uint4v *>(turned_at + (D == 64 ? 4 * i : 16 * (i % 2) + 4 * (i / 2)) * LD) = kr[slot][i];
      } else if (!lone) {
        *reinterpret_cast<uint4v *>(pair_at + 16 * i * KLD) = kr[slot][i];
      } else if (i < CHUNKS / 2) {
        *reinterpret_cast<uint4v *>(lone_at + 32 * i * KLD) = kr[slot][i];
      }
    }
    asm volatile("" ::: "memory");  // (a wavefront's LDS operations complete in order)
  };
  auto stage_v = [&](int slot, bool lone) {  // (the half that a lone block does not have: zeros)
    uint4v const zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < CHUNKS; i++) {
      if (!CM) {
        *reinterpret_cast<uint4v *>(key_at + KEYS * i * LD) = lone && i >= CHUNKS / 2 ? zero : vr[slot][i];
      } else if (!lone) {
        *reinterpret_cast<uint4v *>(pair_at + 16 * i * KLD) = vr[slot][i];
      } else {
        *reinterpret_cast<uint4v *>(lone_at + 32 * (i % (CHUNKS / 2)) * KLD + (i < CHUNKS / 2 ? 0 : 16)) = i < CHUNKS / 2 ? vr[slot][i] : zero;
      }
    }
    asm volatile("" ::: "memory");
  };

  // The next DEPTH pairs of K or V: past an iteration's last one the wavefront's next iteration, past its last
  // iteration (or the for-loop's, which is read again and counts for nothing) that one once more.
  int const steps = (F + IP - 1) / IP * pairs;  // of every wavefront, the same number
  int k_it = ip < F ? ip : F - 1, k_pair = 0, v_it = k_it, v_pair = 0;
  auto advance = [&](int &it, int &pair) {
    pair++;
    if (pair == pairs) {
      pair = 0;
      it = it + IP < F ? it + IP : F - 1;
    }
  };
  auto load_ks = [&](int slots) {
#pragma unroll
    for (int slot = 0; slot < KS; slot++) {
      if (slot < slots) {
        load_k(slot, k_it, k_pair);
        advance(k_it, k_pair);
      }
    }
  };
  auto load_vs = [&](int slots) {
#pragma unroll
    for (int slot = 0; slot < VS; slot++) {
      if (slot < slots) {
        load_v(slot, v_it, v_pair);
        advance(v_it, v_pair);
      }
    }
  };

  // Q fragments: Q[row c][32kk + 8g .. +7] (rows past the tile re-read its last one: every row is
  // worked on by itself and theirs are not stored), through the strip as well
  half8 qf[RPW][DK];
  {
    _Float16 const *q = static_cast<_Float16 const *>(P.q.ptr) + tile_offset(P.q, bx, by, bz, 0);
    uint4v raw[RPW][CHUNKS / 2];
#pragma unroll
    for (int rp = 0; rp < RPW; rp++) {
#pragma unroll
      for (int i = 0; i < CHUNKS / 2; i++) {
        int const row = row_base + 16 * rp + KEYS * i + lane / CPR;
        raw[rp][i] = *(global_chunk const *)(q + (long long)(row < m ? row : m - 1) * P.q.d_cols + 8 * (lane % CPR));
      }
    }
    load_ks(steps < DEPTH ? 1 : DEPTH);
    load_vs(steps < DEPTH ? 1 : DEPTH);
#pragma unroll
    for (int rp = 0; rp < RPW; rp++) {
#pragma unroll
      for (int i = 0; i < CHUNKS / 2; i++) {
        *reinterpret_cast<uint4v *>(key_at + KEYS * i * LD) = raw[rp][i];
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int kk = 0; kk < DK; kk++) {
        qf[rp][kk] = *reinterpret_cast<half8 const *>(strip + c * LD + 32 * kk + 8 * g);
      }
      asm volatile("" ::: "memory");
    }
  }
  half2v const ones = {(_Float16)1.0f, (_Float16)1.0f};
  constexpr float LOG2E = 1.44269504088896340736f;
  float4v o[RPW][DB];
  float rs[RPW];

  // S^T = K^T . Q^T of a staged pair, exp, row sums: S to fp16, exp in fp32, the result to fp16; the row
  // sum adds the rounded values in fp32.  pk: the exponentials of keys 8 g .. + 7 of row c.
  auto scores = [&](bool lone, uint32_t (&pk)[RPW][4]) {
#pragma unroll
    for (int j = 0; j < 2; j++) {
      float4v s[RPW];
#pragma unroll
      for (int rp = 0; rp < RPW; rp++) {
        s[rp] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
      }
#pragma unroll
      for (int kk = 0; kk < DK; kk++) {
        half8 a;
        if (CM) {
          a = *reinterpret_cast<half8 const *>(strip + (16 * j + c) * LD + 32 * kk + 8 * g);
        } else {
          _Float16 const *ka = strip + (32 * kk + 8 * g + a4) * KLD + 8 * b4 + 4 * j;
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
          pk[rp][2 * j + h] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x2, half2v));
        }
      }
    }
#pragma unroll
    for (int rp = 0; rp < RPW; rp++) {
#pragma unroll
      for (int w = 0; w < 4; w++) {
        pk[rp][w] = lone && g >= 2 ? 0u : pk[rp][w];
        rs[rp] = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, pk[rp][w]), ones, rs[rp], false);
      }
    }
    asm volatile("" ::: "memory");
  };
  // O += P . V of a staged pair, V^T first: o[rp][t][r] = O[row c][16t + 4g + r]
  auto values = [&](uint32_t const (&pk)[RPW][4]) {
#pragma unroll
    for (int t = 0; t < DB; t++) {
      half8 b;
      if (CM) {
        b = *reinterpret_cast<half8 const *>(strip + (16 * t + c) * KLD + 8 * g);
      } else {
        _Float16 const *vb = strip + (8 * g + a4) * LD + 16 * t + 4 * b4;
        half4 const lo = lds_read_tr16(vb), hi = lds_read_tr16(vb + 4 * LD);
        b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int rp = 0; rp < RPW; rp++) {
        uint4v const a = {pk[rp][0], pk[rp][1], pk[rp][2], pk[rp][3]};
        o[rp][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, __builtin_bit_cast(half8, a), o[rp][t], 0, 0, 0);
      }
    }
    asm volatile("" ::: "memory");
  };

  auto start = [&]() {
#pragma unroll
    for (int rp = 0; rp < RPW; rp++) {
      rs[rp] = 0.0f;
#pragma unroll
      for (int t = 0; t < DB; t++) {
        o[rp][t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
  };
  // ---- the end of an iteration, of the wavefronts' iterations r0 .. r0 + IP - 1
  auto finish = [&](int r0) {
    // ---- this iteration's result, fp16, where the strip was
#pragma unroll
    for (int rp = 0; rp < RPW; rp++) {
#pragma unroll
      for (int t = 0; t < DB; t++) {
        half2v const lo = __builtin_convertvector(float2v{o[rp][t][0], o[rp][t][1]}, half2v);
        half2v const hi = __builtin_convertvector(float2v{o[rp][t][2], o[rp][t][3]}, half2v);
        uint2v const w = {__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
        *reinterpret_cast<uint2v *>(strip + (16 * rp + c) * LD + 16 * t + 4 * g) = w;
      }
      if (!HAS_DIV && g == 0) {
        strip[ROWS * LD + 16 * rp + c] = static_cast<_Float16>(rs[rp]);
      }
    }
    __syncthreads();
    // ---- the round's results in iteration order, one fp16 rounding per add (a packed fp16 add
    // is the exact sum rounded once).  Between rounds the sums wait in LDS, not in registers.
    int const n = (F - r0) < IP ? (F - r0) : IP;
    bool const first = r0 == 0, done = r0 + IP >= F;
    _Float16 *const og = static_cast<_Float16 *>(const_cast<void *>(P.o.ptr)) + tile_offset(P.o, bx, by, bz, 0);
    AttnFold const next = done ? next_fold<Params>() : AttnFold{};
    bool const shared = next.tickets != nullptr;
    auto total = [&](int r) {  // the row's sum, of this round's and those before
      _Float16 sum = first ? (_Float16)0.0f : sums[ROWS * LD + r];
      for (int u = 0; u < n; u++) {
        sum = sum + all[u * STRIP + ROWS * LD + r];
      }
      return sum;
    };
    for (int e = tid; e < ROWS * CPR; e += NT) {
      int const r = e / CPR, at = r * LD + 8 * (e % CPR), row = row_base + r;
      uint4v sum = {0, 0, 0, 0};
      if (!first) {
        sum = *reinterpret_cast<uint4v const *>(sums + at);
      }
      for (int u = 0; u < n; u++) {
        uint4v const v = *reinterpret_cast<uint4v const *>(all + u * STRIP + at);
#pragma unroll
        for (int w = 0; w < 4; w++) {
          uint32_t const x = v[w], y = sum[w];  // (a bit cast of a vector element itself would read element 0)
          sum[w] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, y) + __builtin_bit_cast(half2v, x));
        }
      }
      if (!done) {
        *reinterpret_cast<uint4v *>(sums + at) = sum;
      } else if (row < m) {
        store_result_16(og + (long long)row * P.o.d_cols + 8 * (e % CPR), sum, shared);
        fold_chunk<Params>(next, bx, by, bz, row, 8 * (e % CPR), sum, [&] { return total(r); });
      }
    }
    if (!HAS_DIV && tid < ROWS) {
      _Float16 const sum = total(tid);
      if (!done) {
        sums[ROWS * LD + tid] = sum;
      } else if (row_base + tid < m) {
        _Float16 *const rg = static_cast<_Float16 *>(const_cast<void *>(P.r.ptr)) + tile_offset(P.r, bx, by, bz, 0);
        store_result_2(rg + (long long)(row_base + tid) * P.r.d_cols, sum, shared);
      }
    }
    if (!done) {
      __syncthreads();  // (the results are read: their place is a strip again)
    }
  };

  if constexpr (HAS_DIV) {
    for (int r0 = 0; r0 < F; r0 += IP) {
      int const it = r0 + ip < F ? r0 + ip : F - 1, next = it + IP < F ? it + IP : F - 1;
      start();
      uint32_t pk[PAIRS][RPW][4];
#pragma unroll
      for (int p = 0; p < PAIRS; p++) {
        bool const lone = odd && p == PAIRS - 1;
        stage_k(0, lone);
        load_k(0, p == PAIRS - 1 ? next : it, p == PAIRS - 1 ? 0 : p + 1);
        scores(lone, pk[p]);
      }
#pragma unroll
      for (int rp = 0; rp < RPW; rp++) {
        // E / sum, rounded to fp32 and then to fp16 as the division is: the reciprocal's product with one
        // correction is the nearest fp32 number.  (Without it quotients below 2^-14 came out one unit
        // off where they lie next to the middle of two fp16 numbers.  An infinite sum: 0, or no number
        // where E is infinite too; E is finite under a finite sum.)
        float const sum = static_cast<float>(static_cast<_Float16>(sum_lane_groups(rs[rp]))), inv = __builtin_amdgcn_rcpf(sum);
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
            half2v const e2 = __builtin_bit_cast(half2v, pk[p][rp][w]);
            uint32_t const q2 = __builtin_bit_cast(uint32_t, half2v{quotient(e2[0]), quotient(e2[1])});
            // (a lone block's missing half stays zero, whatever the sum is)
            pk[p][rp][w] = odd && p == PAIRS - 1 && g >= 2 ? 0u : q2;
          }
        }
      }
#pragma unroll
      for (int p = 0; p < PAIRS; p++) {
        stage_v(0, odd && p == PAIRS - 1);
        load_v(0, p == PAIRS - 1 ? next : it, p == PAIRS - 1 ? 0 : p + 1);
        values(pk[p]);
      }
      finish(r0);
    }
  } else {
    int r0 = 0, p = 0;
    // more: another group of DEPTH steps follows.  An operand of one slot is loaded for the next step, one of
    // DEPTH in the last step of a group for the next group.
    auto step = [&](int slot, bool next, auto more) {
      bool const lone = odd && p == pairs - 1, group = decltype(more)::value && slot == DEPTH - 1;
      uint32_t pk[RPW][4];
      stage_k(slot % KS, lone);
      if (KS == 1 ? next : group) {
        load_ks(DEPTH);
      }
      scores(lone, pk);
      stage_v(slot % VS, lone);
      if (VS == 1 ? next : group) {
        load_vs(DEPTH);
      }
      values(pk);
      p++;
      if (p == pairs) {
#pragma unroll
        for (int rp = 0; rp < RPW; rp++) {
          rs[rp] = sum_lane_groups(rs[rp]);
        }
        finish(r0);
        start();
        p = 0;
        r0 += IP;
      }
    };
    start();
    int s = 0;
    // (RPW 2: the last step loads once more what it has; a copy of the loop's body without loads costs registers)
    for (; s + (RPW == 1 ? DEPTH : 0) < steps; s += DEPTH) {
#pragma unroll
      for (int slot = 0; slot < DEPTH; slot++) {
        step(slot, true, std::true_type{});
      }
    }
#pragma unroll
    for (int slot = 0; slot < (RPW == 1 ? DEPTH : 0); slot++) {
      if (slot == 0 || s + slot < steps) {
        step(slot, slot + 1 < DEPTH && s + slot + 1 < steps, std::false_type{});
      }
    }
  }
  fold_part<Params>(bx, by, bz, slice, row_base, m - row_base < ROWS ? m - row_base : ROWS, lds);
}

}  // namespace mi355
