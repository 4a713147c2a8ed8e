// The un-fused attention graph in one launch: S = Q . K, E = exp(S), R = row sums of E, P = E / R,
// O = P . V for a batch of matrices, every one of the five tensors written, with the roundings the
// operators have one by one (fp32 sums, one fp16 rounding per element of a tensor).
//
// A workgroup owns 16 query rows and all keys; its wavefronts take blocks of 32 keys by turns.
// S^T = K^T . Q^T leaves a lane with eight consecutive scores of one row: they are rounded, stored,
// exponentiated, stored, and the exponentials stay in registers (16 VGPRs at 1024 keys) until the row's
// sum is known; divided they are the operand of P . V, so neither product reads what the other operators
// wrote.  K and V go from memory through registers into a strip of LDS of the wavefront's own, in the order
// they have in memory, and leave it as MFMA operands; results leave the same way.  The wavefronts' sums are
// added up in LDS in wavefront order.
//
// What bounds it: at [8, 500, 1000], head size 64, the 24 MB of scores it stores (without those stores 8.9 us
// of 12.6) behind the chain Q, K - scores - sum - V - store; as three launches 20.2 us, 12.2 here.  Reading K
// and V straight in operand order (16 rows to 16 lanes, a quarter of the rate) it took 13.7 us, at head size
// 128 26 us instead of 12; one 64-bit address per load instead of 32-bit offsets cost 1 us more.
#include "common.h"
#include "f16_gemm.h"

#include <algorithm>

namespace mi355 {

namespace {

constexpr int kRows = 16;
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

struct RowsAttention {
  _Float16 const *q, *k, *v;
  _Float16 *s, *e, *r, *p, *o;
  int m, n, row_blocks;
  unsigned total;  // workgroups
};

__device__ __forceinline__ half4 strip_tr16(_Float16 const *p) {
  typedef short short4v __attribute__((ext_vector_type(4)));
  typedef short4v __attribute__((address_space(3))) *lds_p;
  return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_p)(__attribute__((address_space(3))) void *)p));
}

// A wavefront's own LDS: a block of 32 keys of K or V, as rows of 32 keys (pitch kKeyPitch halfs) or of D
// elements (pitch D + 8), and 16 rows of 32 scores on their way out.  Both pitches spread an operand read
// over all banks.
constexpr int kKeyPitch = 40;
template <int D>
constexpr int strip_halfs() {
  return D * kKeyPitch + kRows * kKeyPitch;
}
template <int D, int W>
constexpr int rows_attention_lds() {
  return std::max(W * strip_halfs<D>() * 2, W * kRows * (D + 4) * 4) + W * kRows * 4;
}

// CH: blocks of 32 keys a wavefront has.  KC: K and V column-major (their reduction index contiguous).
template <int D, bool KC, int W, int CH>
__global__ __launch_bounds__(64 * W) void f16_attention_rows_kernel(RowsAttention const A) {
  constexpr int DK = D / 32, T = D / 16, OPS = D / 16;  // 16-byte chunks a lane holds of 32 keys of K or V
  constexpr int AHEAD = CH < 2 ? CH : 2;  // blocks in flight
  constexpr int CPR = D / 8, DP = D + 8, OP = D + 4;  // chunks of a row of D; its pitch in a strip; pitch of a row of sums
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int const lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), g = lane / 16, c = lane % 16;
  _Float16 *const strip = reinterpret_cast<_Float16 *>(lds) + wave * strip_halfs<D>(), *const out = strip + D * kKeyPitch;
  float *const row_sums = reinterpret_cast<float *>(lds + rows_attention_lds<D, W>() - W * kRows * 4);  // [W][16]

  // an XCD (one L2) gets consecutive row blocks: they share K and V
  unsigned const xcd = blockIdx.x % 8, each = A.total / 8, more = A.total % 8;
  unsigned const id = xcd * each + (xcd < more ? xcd : more) + blockIdx.x / 8;
  int const batch = (int)(id / (unsigned)A.row_blocks), row0 = (int)(id % (unsigned)A.row_blocks) * kRows;
  int const m = A.m, n = A.n;
  // (rows past the matrix repeat its last one, bit for bit: they store what that one stores)
  int const row = row0 + c < m ? row0 + c : m - 1;
  _Float16 const *const kg = A.k + (size_t)batch * n * D, *const vg = A.v + (size_t)batch * n * D;

  // Block i of this wavefront: two blocks in a row are 64 consecutive keys, whole lines of a tensor.  A block
  // that would pass the end is the last 32 keys instead, the first `again` of them another block's: their
  // scores are stored once more, with the same bits, and count for nothing.
  auto own_key = [&](int i) { return 32 * ((i / 2) * 2 * W + (CH % 2 != 0 && i == CH - 1 ? wave : 2 * wave + i % 2)); };
  auto first_key = [&](int i) { return own_key(i) < n - 32 ? own_key(i) : n - 32; };
  auto again = [&](int i) { return own_key(i) - first_key(i); };
  // A block goes from memory into registers in the order it has there: rows of D elements (`by_key`) or,
  // for each of D elements, 32 keys.  (Read as the operands it becomes, sixteen rows to sixteen lanes, it
  // would come at a quarter of the rate: 16 bytes a cycle against 59.)
  half8 raw[AHEAD][OPS];
  uint32_t column[OPS];  // bytes of row 16 x + lane / 4 of a matrix with n columns
#pragma unroll
  for (int x = 0; x < OPS; x++) {
    column[x] = 2u * ((uint32_t)(16 * x + lane / 4) * (uint32_t)n + 8u * (uint32_t)(lane % 4));
  }
  auto load = [&](bool by_key, _Float16 const *from, int key0, half8 (&to)[OPS]) {
    char const *const at = reinterpret_cast<char const *>(by_key ? from + (size_t)key0 * D : from + key0);
#pragma unroll
    for (int x = 0; x < OPS; x++) {
      if (by_key) {
        to[x] = *reinterpret_cast<half8 const *>(at + 16u * (uint32_t)(64 * x + lane));
      } else {
        to[x] = *reinterpret_cast<half8_any const *>(at + column[x]);
      }
    }
  };
  // ... and from there to the strip.  `turn`: key 8 a + 4 j + b at row 16 j + 4 a + b, the order of the operands
  // of S^T.  `drop`: the first keys of a block become zeros.
  auto stage = [&](bool by_key, bool turn, int drop, half8 const (&from)[OPS]) {
#pragma unroll
    for (int x = 0; x < OPS; x++) {
      int const at = 64 * x + lane, k = at / CPR, r = turn ? 16 * (k >> 2 & 1) + 4 * (k >> 3) + (k & 3) : k;
      half8 v = from[x];
      if (drop > 0) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
          v[u] = (by_key ? k : 8 * (at % 4) + u) < drop ? (_Float16)0.0f : v[u];
        }
      }
      *reinterpret_cast<half8 *>(by_key ? strip + r * DP + 8 * (at % CPR) : strip + at / 4 * kKeyPitch + 8 * (at % 4)) = v;
    }
    asm volatile("" ::: "memory");  // (a wavefront's LDS operations complete in order)
  };
  // 16 rows of 32 results, eight of a row per lane, to memory as 64-byte pieces of rows
  uint32_t const out_lane = 2u * ((uint32_t)(row0 + lane / 4 < m ? lane / 4 : m - 1 - row0) * (uint32_t)n + 8u * (uint32_t)(lane % 4));
  size_t const at_out = ((size_t)batch * m + row0) * (size_t)n;
  auto put = [&](_Float16 *tensor, half8 v, int key0) {
    asm volatile("" ::: "memory");
    *reinterpret_cast<half8 *>(out + c * kKeyPitch + 8 * g) = v;
    asm volatile("" ::: "memory");
    half8 const w = *reinterpret_cast<half8 const *>(out + lane / 4 * kKeyPitch + 8 * (lane % 4));
    *reinterpret_cast<half8_any *>(reinterpret_cast<char *>(tensor + at_out + key0) + out_lane) = w;
  };
  half8 qf[DK];
  {
    _Float16 const *const q = A.q + ((size_t)batch * m + row) * D + 8 * g;
#pragma unroll
    for (int kk = 0; kk < DK; kk++) {
      qf[kk] = *reinterpret_cast<half8 const *>(q + 32 * kk);
    }
  }
#pragma unroll
  for (int i = 0; i < AHEAD; i++) {
    load(KC, kg, first_key(i), raw[i]);
  }
  half8 e[CH];
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < CH; i++) {
    int const key0 = first_key(i), skip = again(i);
    stage(KC, true, 0, raw[i % AHEAD]);
    if (i + AHEAD < CH) {
      load(KC, kg, first_key(i + AHEAD), raw[i % AHEAD]);
    } else {
      load(!KC, vg, first_key(i + AHEAD - CH), raw[i % AHEAD]);
    }
    half8 sv;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      float4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kk = 0; kk < DK; kk++) {
        half8 op;
        if (KC) {
          op = *reinterpret_cast<half8 const *>(strip + (16 * j + c) * DP + 32 * kk + 8 * g);
        } else {
          _Float16 const *const at = strip + (32 * kk + 8 * g + (c >> 2)) * kKeyPitch + 8 * (c & 3) + 4 * j;
          half4 const lo = strip_tr16(at), hi = strip_tr16(at + 4 * kKeyPitch);
          op = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(op, qf[kk], acc, 0, 0, 0);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        sv[4 * j + u] = static_cast<_Float16>(acc[u]);
      }
    }
    // (lane (g, c): scores of row c and keys 8 g ..)
#pragma unroll
    for (int u = 0; u < 8; u++) {
      e[i][u] = static_cast<_Float16>(f16_unary_value(true, static_cast<float>(sv[u])));
    }
    half8 count = e[i];
    if (skip > 0) {
#pragma unroll
      for (int u = 0; u < 8; u++) {
        count[u] = 8 * g + u < skip ? (_Float16)0.0f : count[u];
      }
    }
#pragma unroll
    for (int u = 0; u < 8; u += 2) {
      sum = __builtin_amdgcn_fdot2(half2v{count[u], count[u + 1]}, half2v{(_Float16)1.0f, (_Float16)1.0f}, sum, false);
    }
    put(A.s, sv, key0);
    put(A.e, e[i], key0);
  }
  // ---- the rows' sums: over the four lanes of a row, then over the wavefronts
  sum += __shfl_xor(sum, 16, 64);
  sum += __shfl_xor(sum, 32, 64);
  if (g == 0) {
    row_sums[wave * kRows + c] = sum;
  }
  __syncthreads();
  sum = 0.0f;
#pragma unroll
  for (int w = 0; w < W; w++) {
    sum += row_sums[w * kRows + c];
  }
  _Float16 const total = static_cast<_Float16>(sum);
  if (wave == 0 && g == 0) {
    A.r[(size_t)batch * m + row] = total;
  }
  // E / total, rounded to fp32 and then to fp16 as the division is: the reciprocal's product with one
  // correction is the nearest fp32 number (an infinite sum: 0, or no number where E is infinite too)
  float const all = static_cast<float>(total), inv = __builtin_amdgcn_rcpf(all);
  float const by = __builtin_isinf(all) ? 0.0f : -all;
  float4v o[T];
#pragma unroll
  for (int t = 0; t < T; t++) {
    o[t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
  }
#pragma unroll
  for (int i = 0; i < CH; i++) {
    int const key0 = first_key(i), skip = again(i), slot = (CH + i) % AHEAD;
    stage(!KC, false, skip, raw[slot]);
    if (i + AHEAD < CH) {
      load(!KC, vg, first_key(i + AHEAD), raw[slot]);
    }
    half8 p;
#pragma unroll
    for (int u = 0; u < 8; u++) {
      float const x = static_cast<float>(e[i][u]);
      float y = __builtin_fmaf(x, inv, 0.0f);
      y = __builtin_fmaf(__builtin_fmaf(by, y, x), inv, y);
      asm volatile("" : "+v"(y));  // (fused with the conversion the last step would round once)
      p[u] = static_cast<_Float16>(y);
    }
    put(A.p, p, key0);
    if (skip > 0) {  // (and whatever the quotient of a key that is another block's, it meets a zero)
#pragma unroll
      for (int u = 0; u < 8; u++) {
        p[u] = 8 * g + u < skip ? (_Float16)0.0f : p[u];
      }
    }
    // V^T first: o[t][r] = O[row c][16 t + 4 g + r]
#pragma unroll
    for (int t = 0; t < T; t++) {
      half8 op;
      if (KC) {
        op = *reinterpret_cast<half8 const *>(strip + (16 * t + c) * kKeyPitch + 8 * g);
      } else {
        _Float16 const *const at = strip + (8 * g + (c >> 2)) * DP + 16 * t + 4 * (c & 3);
        half4 const lo = strip_tr16(at), hi = strip_tr16(at + 4 * DP);
        op = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op, p, o[t], 0, 0, 0);
    }
    asm volatile("" ::: "memory");
  }
  // ---- the wavefronts' sums, in wavefront order
  __syncthreads();  // (the strips are done with)
  float *const sums = reinterpret_cast<float *>(lds);  // [W][16][OP]
#pragma unroll
  for (int t = 0; t < T; t++) {
    *reinterpret_cast<float4v *>(sums + (wave * kRows + c) * OP + 16 * t + 4 * g) = o[t];
  }
  __syncthreads();
  for (int x = threadIdx.x; x < kRows * D / 4; x += 64 * W) {
    int const r = x / (D / 4), col = 4 * (x % (D / 4));
    float4v all_waves = *reinterpret_cast<float4v const *>(sums + r * OP + col);
#pragma unroll
    for (int w = 1; w < W; w++) {
      float4v const v = *reinterpret_cast<float4v const *>(sums + (w * kRows + r) * OP + col);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        all_waves[u] += v[u];
      }
    }
    if (row0 + r < m) {
      *reinterpret_cast<half4 *>(A.o + ((size_t)batch * m + row0 + r) * D + col) = __builtin_convertvector(all_waves, half4);
    }
  }
}

template <int D, bool KC, int W, int CH>
int launch_rows(RowsAttention const &A) {
  auto *fn = f16_attention_rows_kernel<D, KC, W, CH>;
  constexpr int lds = rows_attention_lds<D, W>();
  MI355_GRANT_LDS(fn, lds);
  MI355_HIP(launch_kernel(fn, A.total, 64 * W, lds, state().stream(), A));
  return MI355_OK;
}

// A wavefront's blocks: as few as hold the row.  Eight wavefronts leave room for two workgroups on a compute
// unit up to 768 keys ([28, 146, 828]: 280 workgroups, 19.6 us with sixteen wavefronts, 16.7 with eight).  At
// head size 128 twelve, with fewer blocks each, were slower: [1, 30, 700] 10.1 us, with eight 9.2, [16, 250, 1500]
// 23.6 and 21.2 (and of five blocks or more their registers spill).
template <bool KC>
int launch_rows_of(RowsAttention const &A, int d) {
  int const blocks = (A.n + 31) / 32, eights = (blocks + 7) / 8;
  if (d == 64) {
    switch (eights) {
      case 1: return launch_rows<64, KC, 8, 1>(A);
      case 2: return launch_rows<64, KC, 8, 2>(A);
      case 3: return launch_rows<64, KC, 8, 3>(A);
      case 4: return launch_rows<64, KC, 8, 4>(A);
      case 5:
      case 6: return launch_rows<64, KC, 16, 3>(A);
      default: return launch_rows<64, KC, 16, 4>(A);
    }
  }
  switch (eights) {
    case 1: return launch_rows<128, KC, 8, 1>(A);
    case 2: return launch_rows<128, KC, 8, 2>(A);
    case 3: return launch_rows<128, KC, 8, 3>(A);
    case 4: return launch_rows<128, KC, 8, 4>(A);
    case 5:
    case 6: return launch_rows<128, KC, 8, 6>(A);
    default: return launch_rows<128, KC, 8, 8>(A);
  }
}

// Where one launch is the faster of the two (against a matmul, the softmax of its rows and a matmul; 68
// graphs): where its workgroups run in about one round, and at head size 64 also where a row is short,
// because every 16 rows read all of K and V.  [heads, rows, keys]: head size 64, [8, 500, 1000] 20.2 and
// 12.2 us, [8, 800, 1024] 23.5 and 15.8, [32, 1000, 500] 51.4 and 43.0, but [32, 512, 1024] 42.1 and 50.2;
// [8, 640, 2000] 33.5 and 29.9, but [16, 512, 2000] 50.3 and 55.3.  Head size 128, [2, 1200, 600] 16.5 and
// 11.7, but [8, 640, 600] 20.4 and 21.7; [8, 300, 1500] 25.0 and 20.0, but few workgroups with a long row
// each leave most of the chip idle: [4, 300, 1500] 19.7 and 21.5, [1, 1, 2048] 11.4 and 16.3, [4, 30, 800] 10.7
// and 11.3, [2, 19, 869] 12.8 and 13.3, but [8, 128, 800] 12.7 and 11.9, [1, 30, 700] 11.5 and 9.2.
bool rows_pay(int d, int n, long long workgroups) {
  if (d == 64) {
    return n <= 512 || (n <= 1024 && workgroups <= 768) || (n <= 2048 && workgroups <= 400);
  }
  int const fewest = n <= 768 ? 1 : (n <= 1024 ? 64 : 128);
  return (n <= 256 && workgroups <= 400) || (n <= 2048 && workgroups >= fewest && workgroups <= 256);
}

}  // namespace
}  // namespace mi355

using namespace mi355;

extern "C" int mi355_f16_attention_rows(void const *Q, void const *K, void const *V, void *S, void *E, void *R, void *P, void *O,
                                        int batch, int m, int n, int d, int dv, int kv_column_major, int *taken) {
  MI355_REQUIRE_INIT();
  if (taken == nullptr) {
    return fail(MI355_ERR_INVALID, "no place for the answer");
  }
  *taken = 0;
  if (batch < 0 || m < 0 || n < 0 || d < 0 || dv < 0) {
    return fail(MI355_ERR_INVALID, "negative attention extent");
  }
  // (rows of d and dv elements are read as aligned 16-byte chunks; a row of keys may start anywhere)
  uintptr_t const rows = reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(O) |
                         (kv_column_major ? reinterpret_cast<uintptr_t>(K) : reinterpret_cast<uintptr_t>(V));
  long long const blocks = (long long)batch * ((m + kRows - 1) / kRows);
  if (d != dv || (d != 64 && d != 128) || m < 1 || n < 32 || n > 2048 || (rows & 15) != 0 || blocks < 1 ||
      blocks > 2147483647LL || !rows_pay(d, n, blocks) || state().f16_matmul_route == 1) {
    return MI355_OK;
  }
  RowsAttention A{};
  A.q = static_cast<_Float16 const *>(Q);
  A.k = static_cast<_Float16 const *>(K);
  A.v = static_cast<_Float16 const *>(V);
  A.s = static_cast<_Float16 *>(S);
  A.e = static_cast<_Float16 *>(E);
  A.r = static_cast<_Float16 *>(R);
  A.p = static_cast<_Float16 *>(P);
  A.o = static_cast<_Float16 *>(O);
  A.m = m;
  A.n = n;
  A.row_blocks = (m + kRows - 1) / kRows;
  A.total = (unsigned)blocks;
  *taken = 1;
  return kv_column_major ? launch_rows_of<true>(A, d) : launch_rows_of<false>(A, d);
}
