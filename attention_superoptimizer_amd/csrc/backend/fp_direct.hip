// Fingerprint matmul C = A . B over Z_227 x Z_113 in one launch, for products too small to repay the
// launch and the passes over memory that splitting their operands into residue planes costs
// (fp_mfma.hip): a workgroup reduces its own tiles to bytes on the way into LDS.
//
// Four wavefronts own 16 RG rows and 64 columns of C; RG of them a 16-row group each, KW = 4 / RG
// sharing a group and taking every KW-th chunk of 64 k.  A step stages KW chunks: 4 consecutive k of a
// row of A are one dword per residue, a 4 x 4 patch of B is turned into four; the next step's raw
// values are in flight meanwhile.  B^T is the first matrix operand: a lane ends up with 16
// consecutive columns of one row.
//
// What bounds it: for one chunk of k the vector instructions that recombine (eight an output) and the
// store, for many the chain of a step, load - reduce - LDS - multiply.  As split planes and a product
// these took, and take here: [32, 256, 64] . [32, 64, 1024] 17.5 and 10.9 us, [32, 256, 1024] .
// [32, 1024, 64] 19.7 and 11.9, [256, 512] . [512, 512] 10.1 and 6.7; rows that are not whole 8-byte
// groups (the vector kernel before), [3, 70, 96] . [3, 96, 130] 10.7 and 7.2.
#include "common.h"
#include "fp_direct.h"

#include <algorithm>
#include <type_traits>

namespace mi355 {

namespace {

constexpr int kThreads = 256, kPitch = 80;  // bytes of an LDS row of 64 residues: free of bank conflicts
typedef int v4i __attribute__((ext_vector_type(4)));

struct DirectJob {
  uint16_t const *A, *B;
  uint16_t *C;
  int m, n, k, tiles_m, tiles_n;
  unsigned first_block;
};
constexpr int kMaxJobs = 48;
struct DirectMany {
  DirectJob job[kMaxJobs];
  int count;
  unsigned total;
};
static_assert(sizeof(DirectMany) <= 4096, "kernel arguments are limited to 4 KB");

template <int KW, bool VEC>  // VEC: rows of A, B and C start on 8 bytes and hold whole groups of 4
__global__ __launch_bounds__(kThreads) void fp_direct_kernel(DirectMany const D) {
  constexpr int RG = 4 / KW, A_BYTES = 16 * RG * kPitch, B_BYTES = 64 * kPitch, CHUNK = 2 * (A_BYTES + B_BYTES);
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];  // [KW][A mod 227, A mod 113, B^T mod 227, B^T mod 113]
  int const tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), g = lane / 16, c = lane % 16;
  int const kw = wave % KW, rg = wave / KW;

  // an XCD (one L2) gets consecutive tiles: they share rows of A
  unsigned const xcd = blockIdx.x % 8, each = D.total / 8, more = D.total % 8;
  unsigned const w = xcd * each + (xcd < more ? xcd : more) + blockIdx.x / 8;
  int j = 0;
  while (j + 1 < D.count && w >= D.job[j + 1].first_block) {
    j++;
  }
  DirectJob const &J = D.job[j];
  int const m = J.m, n = J.n, k = J.k;
  int const tile = (int)(w - J.first_block), per_batch = J.tiles_m * J.tiles_n;
  int const b = tile / per_batch, t = tile % per_batch;
  int const row0 = t / J.tiles_n * (16 * RG), col0 = t % J.tiles_n * 64;
  uint16_t const *const A = J.A + (size_t)b * m * k, *const B = J.B + (size_t)b * k * n;

  // staging: thread = patch (hi, lo): of A, row `hi` of a 16-row group and 4 k from 4 lo; of B, 4 k
  // from 4 hi and 4 columns from 4 lo
  int const hi = tid / 16, lo = tid % 16;
  uint2 ra[KW][RG], rb[KW][4];
  auto four = [&](uint16_t const *p, int left) {  // up to four values, zeros after `left` of them
    uint2 v = {0, 0};
    v.x = (left > 0 ? p[0] : 0u) | (left > 1 ? (uint32_t)p[1] << 16 : 0u);
    v.y = (left > 2 ? p[2] : 0u) | (left > 3 ? (uint32_t)p[3] << 16 : 0u);
    return v;
  };
  // Beyond k the values of A have to be zeros (those of B then count for nothing), rows and columns
  // outside of C are not stored: with whole groups of 4 every load is in bounds after a clamp.
  auto fetch = [&](int step) {
#pragma unroll
    for (int u = 0; u < KW; u++) {
      int const ka = (step * KW + u) * 64 + 4 * lo, kb = (step * KW + u) * 64 + 4 * hi;
#pragma unroll
      for (int r = 0; r < RG; r++) {
        uint16_t const *const p = A + (size_t)min(row0 + 16 * r + hi, m - 1) * k;
        if (VEC) {
          ra[u][r] = *reinterpret_cast<uint2 const *>(p + (ka < k ? ka : 0));
        } else {
          ra[u][r] = four(p + ka, k - ka);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (VEC) {
          rb[u][i] = *reinterpret_cast<uint2 const *>(B + (size_t)min(kb + i, k - 1) * n + min(col0 + 4 * lo, n - 4));
        } else {
          rb[u][i] = four(B + (size_t)(kb + i) * n + col0 + 4 * lo, kb + i < k ? n - col0 - 4 * lo : 0);
        }
      }
    }
  };
  auto put = [&](int step) {
#pragma unroll
    for (int u = 0; u < KW; u++) {
      unsigned char *const ap = lds + u * CHUNK, *const aq = ap + A_BYTES, *const bp = aq + A_BYTES, *const bq = bp + B_BYTES;
#pragma unroll
      for (int r = 0; r < RG; r++) {
        int const at = (16 * r + hi) * kPitch + 4 * lo;
        uint2 x = ra[u][r];
        if (VEC && (step * KW + u) * 64 + 4 * lo >= k) {
          x = uint2{0, 0};
        }
        residues_row(x, *reinterpret_cast<uint32_t *>(ap + at), *reinterpret_cast<uint32_t *>(aq + at));
      }
      uint32_t p[4], q[4];
      residues_patch(rb[u], p, q);
#pragma unroll
      for (int v = 0; v < 4; v++) {
        // column 4 lo + v is row lo of matrix tile v: the lanes of a write differ in their banks
        int const at = (16 * v + lo) * kPitch + 4 * hi;
        *reinterpret_cast<uint32_t *>(bp + at) = p[v];
        *reinterpret_cast<uint32_t *>(bq + at) = q[v];
      }
    }
  };
  auto stage = [&](int step) {
    put(step);
    if (fp_past_residues(fp_bits(ra) | fp_bits(rb))) {  // (looked at last: the first values are not kept waiting)
      fp_into_ring(ra);
      fp_into_ring(rb);
      put(step);
    }
  };

  bool const few = k <= 128;
  v4i acc[2][4];
#pragma unroll
  for (int f = 0; f < 2; f++) {
    int const base = kw != 0 ? 0 : f == 0 ? (few ? kSumBaseFewP : kSumBaseP) : (few ? kSumBaseFewQ : kSumBaseQ);
#pragma unroll
    for (int x = 0; x < 4; x++) {
      acc[f][x] = v4i{base, base, base, base};
    }
  }
  int const chunks = (k + 63) / 64, steps = (chunks + KW - 1) / KW;
  fetch(0);
  for (int s = 0; s < steps; s++) {
    __syncthreads();
    stage(s);
    __syncthreads();
    if (s + 1 < steps) {
      fetch(s + 1);
    }
    if (s * KW + kw < chunks) {
#pragma unroll
      for (int f = 0; f < 2; f++) {
        unsigned char const *const at = lds + kw * CHUNK + f * A_BYTES, *const bt = lds + kw * CHUNK + 2 * A_BYTES + f * B_BYTES;
        v4i const a = *reinterpret_cast<v4i const *>(at + (16 * rg + c) * kPitch + 16 * g);
#pragma unroll
        for (int x = 0; x < 4; x++) {
          v4i const bb = *reinterpret_cast<v4i const *>(bt + (16 * x + c) * kPitch + 16 * g);
          acc[f][x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bb, a, acc[f][x], 0, 0, 0);
        }
      }
    }
  }
  if (KW > 1) {  // the wavefronts' k together
    int *const part = reinterpret_cast<int *>(lds);  // [KW - 1][RG][32][64]
    __syncthreads();
    if (kw > 0) {
#pragma unroll
      for (int x = 0; x < 32; x++) {
        part[(((kw - 1) * RG + rg) * 32 + x) * 64 + lane] = acc[x / 16][x / 4 % 4][x % 4];
      }
    }
    __syncthreads();
    if (kw > 0) {
      return;
    }
#pragma unroll
    for (int u = 0; u < KW - 1; u++) {
#pragma unroll
      for (int x = 0; x < 32; x++) {
        acc[x / 16][x / 4 % 4][x % 4] += part[((u * RG + rg) * 32 + x) * 64 + lane];
      }
    }
  }
  int const row = row0 + 16 * rg + c;
  if (row >= m) {
    return;
  }
  uint16_t *const out = J.C + (size_t)b * m * n + (size_t)row * n;
  auto store = [&](auto is_few) {
#pragma unroll
    for (int h = 0; h < 2; h++) {  // a lane's columns are 16 g .. + 15: 4 e + x from tile x
      int const col = col0 + 16 * g + 8 * h;
      uint32_t z[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        int const x = u % 4, e = 2 * h + u / 4;
        z[u] = fp_from_based_sums<decltype(is_few)::value>((uint32_t)acc[0][x][e], (uint32_t)acc[1][x][e]);
      }
      uint32_t const w[4] = {z[0] | (z[1] << 16), z[2] | (z[3] << 16), z[4] | (z[5] << 16), z[6] | (z[7] << 16)};
      if (VEC && col + 8 <= n) {
        __builtin_memcpy(__builtin_assume_aligned(out + col, 8), w, 16);
      } else if (VEC && col < n) {
        __builtin_memcpy(__builtin_assume_aligned(out + col, 8), w, 8);
      } else if (!VEC) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
          if (col + u < n) {
            out[col + u] = static_cast<uint16_t>(z[u]);
          }
        }
      }
    }
  };
  few ? store(std::true_type{}) : store(std::false_type{});
}

template <int KW>
constexpr int direct_lds() {
  constexpr int tiles = KW * 2 * (16 * (4 / KW) + 64) * kPitch, part = (KW - 1) * (4 / KW) * 32 * 64 * 4;
  return tiles > part ? tiles : part;
}

template <bool VEC>
hipError_t launch_direct(int kw, DirectMany const &D) {
  hipStream_t const st = state().stream();
  switch (kw) {
    case 1: return launch_kernel(fp_direct_kernel<1, VEC>, D.total, kThreads, direct_lds<1>(), st, D);
    case 2: return launch_kernel(fp_direct_kernel<2, VEC>, D.total, kThreads, direct_lds<2>(), st, D);
    default: return launch_kernel(fp_direct_kernel<4, VEC>, D.total, kThreads, direct_lds<4>(), st, D);
  }
}

}  // namespace

// Up to 2048 tile steps of 64 x 64 x 64: from there on the planes, split once, repay their launch because
// this kernel reduces an operand again for every tile that reads it ([1024, 1024] . [1024, 1024], 4096
// steps: 14.3 us on planes, 14.9 here; [2048, 512] . [512, 2048], 8192: 18.6 and 18.9).  A long k over few
// tiles is a chain of steps here, parts of k on other compute units there ([256, 4096] . [4096, 256]: 15.7
// and 30.3).
bool fp_direct_pays(int batch, int m, int n, int k) {
  if (state().fp_vector_dot_only || batch <= 0 || m <= 0 || n <= 0 || k <= 0) {
    return false;
  }
  long long const tiles = (long long)batch * ((m + 63) / 64) * ((n + 63) / 64);
  return k <= 1024 && tiles * ((k + 63) / 64) <= 2048;
}

int launch_fp_direct(uint16_t const *const *A, uint16_t const *const *B, uint16_t *const *C, int const *batch, int const *m,
                     int const *n, int const *k, int count) {
  for (int done = 0; done < count; done += kMaxJobs) {
    int const jobs = std::min(count - done, kMaxJobs);
    // Wavefronts to a row group: as few as leave a workgroup for every compute unit, no more than
    // there are chunks of k.
    int kw = 1;
    for (; kw < 4; kw *= 2) {
      long long blocks = 0, deep = 0;
      for (int e = done; e < done + jobs; e++) {
        int const rows = 64 / kw;
        blocks += (long long)batch[e] * ((m[e] + rows - 1) / rows) * ((n[e] + 63) / 64);
        deep = std::max<long long>(deep, (k[e] + 63) / 64);
      }
      if (blocks >= 256 || deep < 2 * kw) {
        break;
      }
    }
    DirectMany D{};
    long long total = 0;
    bool vec = true;
    for (int e = 0; e < jobs; e++) {
      DirectJob &J = D.job[e];
      int const i = done + e, rows = 64 / kw;
      J.A = A[i];
      J.B = B[i];
      J.C = C[i];
      J.m = m[i];
      J.n = n[i];
      J.k = k[i];
      J.tiles_m = (m[i] + rows - 1) / rows;
      J.tiles_n = (n[i] + 63) / 64;
      vec = vec && k[i] % 4 == 0 && n[i] % 4 == 0 &&
              ((reinterpret_cast<uintptr_t>(A[i]) | reinterpret_cast<uintptr_t>(B[i]) | reinterpret_cast<uintptr_t>(C[i])) & 7) == 0;
      J.first_block = (unsigned)total;
      total += (long long)batch[i] * J.tiles_m * J.tiles_n;
    }
    if (total > 2147483647LL) {
      return fail(MI355_ERR_UNSUPPORTED, "matmuls have too many output tiles");
    }
    D.count = jobs;
    D.total = (unsigned)total;
    if (vec) {
      MI355_HIP(launch_direct<true>(kw, D));
    } else {
      MI355_HIP(launch_direct<false>(kw, D));
    }
  }
  return MI355_OK;
}

}  // namespace mi355
