// The next operator at the end of an attention kernel: where a plan of two outputs (numerators and row sums,
// perhaps one piece of each per split of the keys) is followed by the operator that folds the pieces and
// divides (combine.h), a row of that operator's result depends on the same row of the attention operator's
// results only.  A workgroup that has whole rows goes on with them; where the pieces of a row come from
// several workgroups, the last of them to finish does.  Both operators' tensors are written.
//
// What it saves is a launch: of the pair's time 3 - 4 us on the host, on the device the gap, the start and the
// argument block of a kernel that has next to nothing to do, and a trip of the results through memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "combine.h"

namespace mi355 {

struct AttnFold {
  _Float16 const *n, *d;  // rows of S pieces of X columns, of S row sums
  _Float16 *o;            // rows of X columns, o_cols apart
  int *tickets;           // one per row block, zero between launches; null: a workgroup has whole rows
  int lin[3];             // rows per step of bx, by, bz
  int ticket_lin[3];      // row blocks per step of bx, by, bz
  int arrivals;           // workgroups that have pieces of a row block
  int S, X, o_cols;
  uint32_t mxv;  // division magic of X / 4
  float after;   // -0, what leaves a quotient as it is, or +0, what a sum or a saver behind the division begins with
};

// Memory as global memory (a flat access counts as an LDS operation too).  A result that a workgroup on another
// XCD is to read goes past this XCD's L2: a relaxed atomic store of the device's scope is such a write and costs
// what a plain one does, where a release fence would write back the whole L2.
typedef __attribute__((address_space(1))) uint32_t fold_global_u32;
typedef __attribute__((address_space(1))) uint64_t fold_global_u64;
typedef uint32_t fold_uint4 __attribute__((ext_vector_type(4)));
typedef uint32_t fold_uint2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) fold_uint4 fold_global_uint4;
typedef __attribute__((address_space(1))) fold_uint2 fold_global_uint2;
typedef __attribute__((address_space(1))) uint16_t fold_global_u16;

__device__ __forceinline__ void store_result_16(_Float16 *p, fold_uint4 v, bool shared) {
  if (shared) {
    auto *q = (fold_global_u64 *)(uint64_t *)p;
    __hip_atomic_store(q, (uint64_t)v[0] | (uint64_t)v[1] << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q + 1, (uint64_t)v[2] | (uint64_t)v[3] << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    *(fold_global_uint4 *)(fold_uint4 *)p = v;
  }
}
__device__ __forceinline__ void store_result_8(_Float16 *p, fold_uint2 v, bool shared) {
  if (shared) {
    __hip_atomic_store((fold_global_u64 *)(uint64_t *)p, (uint64_t)v[0] | (uint64_t)v[1] << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    *(fold_global_uint2 *)(fold_uint2 *)p = v;
  }
}
__device__ __forceinline__ void store_result_4(_Float16 *p, uint32_t v, bool shared) {
  if (shared) {
    __hip_atomic_store((fold_global_u32 *)(uint32_t *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    *(fold_global_u32 *)(uint32_t *)p = v;
  }
}
__device__ __forceinline__ void store_result_2(_Float16 *p, _Float16 v, bool shared) {
  if (shared) {
    __hip_atomic_store((fold_global_u16 *)(uint16_t *)p, __builtin_bit_cast(uint16_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    *(fold_global_u16 *)(uint16_t *)p = __builtin_bit_cast(uint16_t, v);
  }
}

__device__ __forceinline__ long long fold_row(AttnFold const &F, int bx, int by, int bz, int row_base) {
  return (long long)bx * F.lin[0] + (long long)by * F.lin[1] + (long long)bz * F.lin[2] + row_base;
}
// combine_fused_kernel's arithmetic.  One piece a row, this workgroup's own: the quotient of a column that it stores and
// of the row's sum.  With one piece all its forms come to the same but for the sign of a zero (a negative number over
// an infinite sum, or a quotient past the smallest number): what divides before it sums adds the quotient to +0.
__device__ __forceinline__ _Float16 fold_own(AttnFold const &F, _Float16 n, _Float16 sum) {
  return static_cast<_Float16>((0.0f + static_cast<float>(n)) / (0.0f + static_cast<float>(sum))) + static_cast<_Float16>(F.after);
}
__device__ __forceinline__ void fold_own_chunk(AttnFold const &F, long long row, int x, fold_uint4 n, _Float16 sum) {
  typedef _Float16 half8v __attribute__((ext_vector_type(8)));
  half8v const v = __builtin_bit_cast(half8v, n);
  half8v out;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    out[j] = fold_own(F, v[j], sum);
  }
  store_result_16(F.o + row * F.o_cols + x, __builtin_bit_cast(fold_uint4, out), false);
}

// The same of S <= PIECES pieces a row, most of them other workgroups', summed before the division.  All of a thread's loads go out together:
// from the memory that all XCDs share a trip is a microsecond.  `lds`: room for rows x S row sums.
constexpr int kFoldPieces = 16;
template <int PIECES>
__device__ __forceinline__ void fold_shared_rows(AttnFold const &F, long long row0, int rows, _Float16 *lds) {
  typedef _Float16 half4v __attribute__((ext_vector_type(4)));
  int const xv = F.X / 4, items = rows * xv;
  auto row_sum = [&](int d) {
    auto const *const q = (fold_global_u16 const *)(uint16_t const *)(F.d + row0 * F.S + d);
    return __builtin_bit_cast(_Float16, (uint16_t)__hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  };
  int const all = rows * F.S, d0 = threadIdx.x;
  _Float16 const first_sum = row_sum(d0 < all ? d0 : all - 1);  // (ahead of the pieces: loads come back in order)
  for (int e0 = 0; e0 < items; e0 += blockDim.x) {  // (every thread as often: there is a barrier inside)
    int const e = e0 + (int)threadIdx.x < items ? e0 + (int)threadIdx.x : items - 1;
    int const r = F.mxv ? (int)__umulhi((uint32_t)e, F.mxv) : e, x = (e - r * xv) * 4;
    auto const *const first = (fold_global_u64 const *)(uint64_t const *)(F.n + (row0 + r) * F.S * F.X + x);
    uint64_t v[PIECES];
#pragma unroll
    for (int u = 0; u < PIECES; u++) {  // (places past the last piece re-read it and are not added)
      v[u] = __hip_atomic_load(first + (u < F.S ? u : F.S - 1) * (F.X / 4), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (e0 == 0) {
      if (d0 < all) {
        lds[d0] = first_sum;
      }
      for (int d = d0 + blockDim.x; d < all; d += blockDim.x) {
        lds[d] = row_sum(d);
      }
      __syncthreads();
    }
    uint32_t sums[PIECES];
#pragma unroll
    for (int u = 0; u < PIECES; u++) {
      sums[u] = __builtin_bit_cast(uint16_t, lds[r * F.S + (u < F.S ? u : F.S - 1)]);
    }
#pragma unroll
    for (int u = 0; u < PIECES; u++) {  // (read whether they are added or not: under the condition each is a trip of its own)
      asm volatile("" : "+v"(sums[u]), "+v"(v[u]));
    }
    float den = 0.0f, acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < PIECES; u++) {
      if (u < F.S) {
        half4v const piece = __builtin_bit_cast(half4v, v[u]);
        den += static_cast<float>(__builtin_bit_cast(_Float16, (uint16_t)sums[u]));
#pragma unroll
        for (int j = 0; j < 4; j++) {
          acc[j] += static_cast<float>(piece[j]);
        }
      }
    }
    float const den16 = static_cast<float>(static_cast<_Float16>(den));
    half4v out;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      out[j] = static_cast<_Float16>(static_cast<float>(static_cast<_Float16>(acc[j])) / den16);
    }
    if (e0 + (int)threadIdx.x < items) {
      store_result_8(F.o + (row0 + r) * F.o_cols + x, __builtin_bit_cast(fold_uint2, out), false);
    }
  }
}

// Called by a whole workgroup after its stores of rows row_base .. row_base + rows - 1 of block (bx, by, bz), which are row
// block `slice` of it; `lds`: 16 bytes and room for rows x S halfs that nothing else uses any more after a barrier.  (A
// workgroup that has whole rows has folded them where it stored its results: fold_own.)
// The last workgroup of a row block sees the others' results: each wavefront waits until its own stores are in the
// memory that all XCDs share (they are device-scope stores: see store_result_16) before the workgroup's
// ticket is drawn, and the loads are of the same scope.  Nobody waits for another workgroup.
__device__ __forceinline__ void attn_fold(AttnFold const &F, int bx, int by, int bz, int slice, int row_base, int rows, void *lds) {
  if (F.tickets == nullptr) {
    return;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int *const last = static_cast<int *>(lds);
  if (threadIdx.x == 0) {
    int *const ticket = F.tickets + bx * F.ticket_lin[0] + by * F.ticket_lin[1] + bz * F.ticket_lin[2] + slice;
    int const before = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *last = before == F.arrivals - 1;
    if (before == F.arrivals - 1) {
      __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
    }
  }
  __syncthreads();
  if (*last != 0) {
    long long const row0 = fold_row(F, bx, by, bz, row_base);
    _Float16 *const sums = static_cast<_Float16 *>(lds) + 8;
    if (F.S <= 8) {
      fold_shared_rows<8>(F, row0, rows, sums);
    } else {
      fold_shared_rows<kFoldPieces>(F, row0, rows, sums);
    }
  }
}

}  // namespace mi355
