// The customized-op interpreters: one workgroup per logical thread block walks
// the thread-block graph once per for-loop iteration with every tile in LDS.
//
//   fp_interp_kernel   uint16 over Z_25651, integer only
//                      (reference compute_customizedop_fingerprint,
//                       src/kernel/cuda/customized_kernel.cu:307-603)
//   f16_interp_kernel  fp16 tiles, fp32 math, matmul on the matrix cores
//                      (reference customized_kernel_function, :39-305, with the
//                       arithmetic the reference's generated programs define,
//                       src/kernel/triton_code_gen.cc:223-333)
#include "common.h"
#include "mi355_kernels/kernarg.h"
#include "tb_program.h"
#include <atomic>
#include <memory>
#include <type_traits>

#include <algorithm>
#include <string>
#include <vector>
#include <cstring>

namespace mi355 {

constexpr int kInterpThreads = 256;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

struct TileOrigin {
  long long base;  // element offset of the batch slice
  int row0, col0;
};

// (Every operand is the same in all lanes.  When the program record sits in LDS the compiler
// cannot know that, so they are made scalar here: the sums of products then run on the scalar
// unit instead of as quarter-rate vector integer multiplies.)
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ TileOrigin tile_origin(DevOp const &op, int it, int bx, int by, int bz) {
  TileOrigin o;
  bx = uniform(bx);
  by = uniform(by);
  bz = uniform(bz);
  it = uniform(it);
  o.row0 = bx * uniform(op.row_bs[0]) + by * uniform(op.row_bs[1]) + bz * uniform(op.row_bs[2]) +
           it * uniform(op.row_fs);
  o.col0 = bx * uniform(op.col_bs[0]) + by * uniform(op.col_bs[1]) + bz * uniform(op.col_bs[2]) +
           it * uniform(op.col_fs);
  o.base = (long long)bx * uniform(op.g_bs[0]) + (long long)by * uniform(op.g_bs[1]) +
           (long long)bz * uniform(op.g_bs[2]) + (long long)it * uniform(op.g_fs);
  return o;
}
__device__ __forceinline__ TileOrigin tile_origin(DevOp const &op, int it, int bx) {
  return tile_origin(op, it, bx, blockIdx.y, blockIdx.z);
}

// ===========================================================================
// uint16 interpreter
// ===========================================================================
// LDS table block: [0,113) exp premultiplied by the CRT lift, [128,355) div_p,
// [384,497) div_q
__device__ __forceinline__ uint32_t lds_exp(uint16_t const *tbl, uint32_t x) {
  return tbl[residue_q(x)];
}
__device__ __forceinline__ uint32_t lds_div(uint16_t const *tbl, uint32_t x, uint32_t y) {
  return fp_from_residues(residue_p(__umul24(residue_p(x), tbl[128 + residue_p(y)])),
                          __umul24(residue_q(x), tbl[384 + residue_q(y)]));
}
__device__ __forceinline__ uint32_t lds_silu(uint16_t const *tbl, uint32_t x) {
  uint32_t neg = mod_pq(FP_PQ - x);
  uint32_t den = mod_pq(1u + lds_exp(tbl, neg));
  return lds_div(tbl, x, den);
}

// Tile index arithmetic without integer division: q = e / d for e * d < 2^32 is one
// multiply-high with magic = ceil(2^32 / d) (0 stands for d == 1), computed on the host.
__device__ __forceinline__ int fdiv(int e, uint32_t magic) {
  return magic ? (int)__umulhi((uint32_t)e, magic) : e;
}

// C[m][n] = A[m][k] . B[k][n] over Z_25651 without a modulus in the inner loop:
// every operand is split into its residues modulo 227 and 113 (both fit a byte), four
// consecutive k are packed into one dword per field, and the packed 4 x 8-bit dot
// instruction accumulates in each field; one CRT recombination per output and k chunk
// (reference multipliers, include/mirage/type.h:26-36).  The sum of products modulo
// 25651 is fixed by its two residues, so the value equals the reference's
// `(r + a*b) % 25651` chain (matmul.h:773-804) bit for bit.  m, n, k, kc multiples of 4.
// scratch: Ap[2][kc/4][m + 4] then Bp[2][kc/4][n] dwords; thread tiles are 4 x 4.
__device__ void fp_matmul_packed(uint16_t const *A, uint16_t const *B, uint16_t *C, int m, int n,
                                 int k, DevOp const &op, uint32_t *scratch, int tid) {
  int const kc = op.mm_kc, kq = kc / 4, lda = m + 4;
  uint32_t *Ap = scratch, *Bp = scratch + 2 * kq * lda;
  int const n2 = n / 2, n4 = n / 4, tiles = (m / 4) * n4;
  for (int k0 = 0; k0 < k; k0 += kc) {
    if (k0 > 0) {
      __syncthreads();  // the previous chunk's residues are still being read
    }
    for (int e = tid; e < m * kq; e += kInterpThreads) {
      int const row = fdiv(e, op.mg0), q = e - row * kq;
      uint2 v = *reinterpret_cast<uint2 const *>(A + row * k + k0 + 4 * q);
      uint32_t v0 = v.x & 0xffffu, v1 = v.x >> 16, v2 = v.y & 0xffffu, v3 = v.y >> 16;
      Ap[q * lda + row] = residues_p4(v0, v1, v2, v3);
      Ap[(kq + q) * lda + row] = residues_q4(v0, v1, v2, v3);
    }
    for (int e = tid; e < kq * n2; e += kInterpThreads) {
      int const q = fdiv(e, op.mg1), c2 = (e - q * n2) * 2;
      uint16_t const *bp = B + (k0 + 4 * q) * n + c2;
      uint32_t w0 = *reinterpret_cast<uint32_t const *>(bp);
      uint32_t w1 = *reinterpret_cast<uint32_t const *>(bp + n);
      uint32_t w2 = *reinterpret_cast<uint32_t const *>(bp + 2 * n);
      uint32_t w3 = *reinterpret_cast<uint32_t const *>(bp + 3 * n);
      uint2 pp, qq;
      pp.x = residues_p4(w0 & 0xffffu, w1 & 0xffffu, w2 & 0xffffu, w3 & 0xffffu);
      pp.y = residues_p4(w0 >> 16, w1 >> 16, w2 >> 16, w3 >> 16);
      qq.x = residues_q4(w0 & 0xffffu, w1 & 0xffffu, w2 & 0xffffu, w3 & 0xffffu);
      qq.y = residues_q4(w0 >> 16, w1 >> 16, w2 >> 16, w3 >> 16);
      *reinterpret_cast<uint2 *>(Bp + q * n + c2) = pp;
      *reinterpret_cast<uint2 *>(Bp + (kq + q) * n + c2) = qq;
    }
    __syncthreads();
    for (int t = tid; t < tiles; t += kInterpThreads) {
      int const tr = fdiv(t, op.mg2), r0 = tr * 4, c0 = (t - tr * n4) * 4;
      uint32_t accp[4][4], accq[4][4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
          accp[i][j] = 0;
          accq[i][j] = 0;
        }
      }
      uint32_t const *ap = Ap + r0, *bp = Bp + c0;
      for (int q = 0; q < kq; q++) {
        uint4v a_p = *reinterpret_cast<uint4v const *>(ap + q * lda);
        uint4v a_q = *reinterpret_cast<uint4v const *>(ap + (kq + q) * lda);
        uint4v b_p = *reinterpret_cast<uint4v const *>(bp + q * n);
        uint4v b_q = *reinterpret_cast<uint4v const *>(bp + (kq + q) * n);
#pragma unroll
        for (int i = 0; i < 4; i++) {
#pragma unroll
          for (int j = 0; j < 4; j++) {
            accp[i][j] = __builtin_amdgcn_udot4(a_p[i], b_p[j], accp[i][j], false);
            accq[i][j] = __builtin_amdgcn_udot4(a_q[i], b_q[j], accq[i][j], false);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        uint16_t *cp = C + (r0 + i) * n + c0;
        uint32_t z[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          z[j] = fp_from_residues(mod_p(accp[i][j]), mod_q(accq[i][j]));
        }
        if (k0 > 0) {
          uint2 old = *reinterpret_cast<uint2 const *>(cp);
          z[0] = mod_pq(z[0] + (old.x & 0xffffu));
          z[1] = mod_pq(z[1] + (old.x >> 16));
          z[2] = mod_pq(z[2] + (old.y & 0xffffu));
          z[3] = mod_pq(z[3] + (old.y >> 16));
        }
        uint2 out;
        out.x = z[0] | (z[1] << 16);
        out.y = z[2] | (z[3] << 16);
        *reinterpret_cast<uint2 *>(cp) = out;
      }
    }
  }
}

// The same product on the int8 matrix cores, for tiles whose m and n are multiples of 16
// and a k chunk that is a multiple of 64.  Residues are packed as signed bytes (mod 227
// recentred to [-113, 113], mod 113 as it is), A as Ab[field][m][kc], B transposed as
// Bb[field][n][kc]; kc is a power of two and the 16-byte chunks of a row are XOR-swizzled by
// a key of the row so that the 16 rows a 16-lane group reads fall on all banks without any
// padding (the scratch is no larger than the dot4 path's); a wavefront owns 32 x 32 outputs at a time and issues
// v_mfma_i32_16x16x64_i8 per field; B^T is the first operand, so a lane ends up with four
// consecutive columns of one row of C.  One CRT recombination per output and k chunk.
typedef int v4i __attribute__((ext_vector_type(4)));

__device__ void fp_matmul_mfma(uint16_t const *A, uint16_t const *B, uint16_t *C, int m, int n, int k,
                               DevOp const &op, unsigned char *scratch, int tid) {
  // A is packed `mb` rows at a time (op.mm_mb, a multiple of 16 that divides m; the whole
  // tile when the scratch allows), B^T once per k chunk
  int const kc = op.mm_kc, kq = kc / 4, pitch = kc, mb = op.mm_mb;
  unsigned char *Ab = scratch, *Bb = scratch + 2 * mb * pitch;
  // chunk c of row `row` lives at chunk c ^ key(row): rows that share a 256-byte bank line
  // (4 rows of 64 bytes, 2 of 128) and rows a multiple of that apart get different keys
  int const key_shift = kc >= 256 ? 0 : (kc == 128 ? 1 : 2);
  int const key_mask = (kc / 16 < 16 ? kc / 16 : 16) - 1;
  auto swz = [&](int row, int byte) {  // byte offset within the row -> swizzled byte offset
    return (((byte >> 4) ^ ((row >> key_shift) & key_mask)) << 4) | (byte & 15);
  };
  int const n2 = n / 2;
  // residue fields this product needs (compile_plan): a field that nobody reads, or that is zero
  // because an operand's is, is neither packed nor multiplied
  bool const do_p = (uniform(op.mm_fields) & 1) != 0, do_q = (uniform(op.mm_fields) & 2) != 0;
  int const wave = tid / 64, lane = tid % 64, r = lane % 16, g = lane / 16;
  int const mt_n = (n + 31) / 32, mt = ((mb + 31) / 32) * mt_n;  // 32 x 32 pieces of a row block
  for (int k0 = 0; k0 < k; k0 += kc) {
    if (k0 > 0) {
      __syncthreads();  // the previous chunk's residues are still being read
    }
    for (int e = tid; e < kq * n2; e += kInterpThreads) {
      int const q = fdiv(e, op.mg1), c2 = (e - q * n2) * 2;
      uint16_t const *bp = B + (k0 + 4 * q) * n + c2;
      uint32_t w0 = *reinterpret_cast<uint32_t const *>(bp);
      uint32_t w1 = *reinterpret_cast<uint32_t const *>(bp + n);
      uint32_t w2 = *reinterpret_cast<uint32_t const *>(bp + 2 * n);
      uint32_t w3 = *reinterpret_cast<uint32_t const *>(bp + 3 * n);
      int const at0 = c2 * pitch + swz(c2, 4 * q), at1 = (c2 + 1) * pitch + swz(c2 + 1, 4 * q);
      if (do_p) {
        *reinterpret_cast<uint32_t *>(Bb + at0) =
            residues_p4_signed(w0 & 0xffffu, w1 & 0xffffu, w2 & 0xffffu, w3 & 0xffffu);
        *reinterpret_cast<uint32_t *>(Bb + at1) = residues_p4_signed(w0 >> 16, w1 >> 16, w2 >> 16, w3 >> 16);
      }
      if (do_q) {
        *reinterpret_cast<uint32_t *>(Bb + n * pitch + at0) =
            residues_q4(w0 & 0xffffu, w1 & 0xffffu, w2 & 0xffffu, w3 & 0xffffu);
        *reinterpret_cast<uint32_t *>(Bb + n * pitch + at1) = residues_q4(w0 >> 16, w1 >> 16, w2 >> 16, w3 >> 16);
      }
    }
    for (int m0 = 0; m0 < m; m0 += mb) {
      if (m0 > 0) {
        __syncthreads();  // the previous row block's residues are still being read
      }
      for (int e = tid; e < mb * kq; e += kInterpThreads) {
        int const row = fdiv(e, op.mg0), q = e - row * kq;
        uint2 v = *reinterpret_cast<uint2 const *>(A + (m0 + row) * k + k0 + 4 * q);
        uint32_t v0 = v.x & 0xffffu, v1 = v.x >> 16, v2 = v.y & 0xffffu, v3 = v.y >> 16;
        int const at = row * pitch + swz(row, 4 * q);
        if (do_p) {
          *reinterpret_cast<uint32_t *>(Ab + at) = residues_p4_signed(v0, v1, v2, v3);
        }
        if (do_q) {
          *reinterpret_cast<uint32_t *>(Ab + mb * pitch + at) = residues_q4(v0, v1, v2, v3);
        }
      }
      __syncthreads();
      for (int t = wave; t < mt; t += kInterpThreads / 64) {
        int const row_m = (t / mt_n) * 32, col_n = (t - (t / mt_n) * mt_n) * 32;
        int const i1 = row_m + 16 < mb ? 1 : 0, j1 = col_n + 16 < n ? 1 : 0;
        unsigned char const *a_at[2], *b_at[2];
        int a_key[2], b_key[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          int const ar = row_m + 16 * (i ? i1 : 0) + r, br = col_n + 16 * (i ? j1 : 0) + r;
          a_at[i] = Ab + ar * pitch;
          b_at[i] = Bb + br * pitch;
          a_key[i] = (ar >> key_shift) & key_mask;
          b_key[i] = (br >> key_shift) & key_mask;
        }
        v4i acc[2][2][2];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          acc[e / 4][(e / 2) % 2][e % 2] = v4i{0, 0, 0, 0};
        }
        for (int ks = 0; ks < kc; ks += 64) {
#pragma unroll
          for (int f = 0; f < 2; f++) {
            if (f ? !do_q : !do_p) {
              continue;
            }
            v4i a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
              int const ca = (((ks >> 4) + g) ^ a_key[i]) << 4, cb = (((ks >> 4) + g) ^ b_key[i]) << 4;
              a[i] = *reinterpret_cast<v4i const *>(a_at[i] + f * mb * pitch + ca);
              b[i] = *reinterpret_cast<v4i const *>(b_at[i] + f * n * pitch + cb);
            }
#pragma unroll
            for (int i = 0; i < 2; i++) {
#pragma unroll
              for (int jn = 0; jn < 2; jn++) {
                acc[f][i][jn] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[jn], a[i], acc[f][i][jn], 0, 0, 0);
              }
            }
          }
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
#pragma unroll
          for (int jn = 0; jn < 2; jn++) {
            if (i > i1 || jn > j1) {
              continue;
            }
            uint16_t *cp = C + (m0 + row_m + 16 * i + r) * n + col_n + 16 * jn + 4 * g;
            uint32_t z[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
              z[e] = fp_from_residue_sums(acc[0][i][jn][e], acc[1][i][jn][e]);
            }
            if (k0 > 0) {
              uint2 old = *reinterpret_cast<uint2 const *>(cp);
              z[0] = mod_pq(z[0] + (old.x & 0xffffu));
              z[1] = mod_pq(z[1] + (old.x >> 16));
              z[2] = mod_pq(z[2] + (old.y & 0xffffu));
              z[3] = mod_pq(z[3] + (old.y >> 16));
            }
            uint2 out;
            out.x = z[0] | (z[1] << 16);
            out.y = z[2] | (z[3] << 16);
            *reinterpret_cast<uint2 *>(cp) = out;
          }
        }
      }
    }
  }
}

__device__ __forceinline__ uint32_t add_mod_pair(uint32_t a, uint32_t b) {
  // two uint16 lanes: (a + b) mod 25651 in each
  uint32_t lo = mod_pq((a & 0xffffu) + (b & 0xffffu));
  uint32_t hi = mod_pq((a >> 16) + (b >> 16));
  return lo | (hi << 16);
}

// One workgroup of the uint16 interpreter: logical block (bx, by, bz) of program P, part
// `split` of its for-loop.  The lookup tables are already in LDS.
__device__ __forceinline__ void fp_interp_block(DevProgram const &P, unsigned char *lds, int bx,
                                                int by, int bz, int split) {
  uint16_t *tbl = reinterpret_cast<uint16_t *>(lds);
  int const tid = threadIdx.x;
  int const F = P.forloop_range;
  // a split for-loop: this workgroup covers iterations [it_begin, it_end) of block bx
  // (32-bit: a for-loop is cut into at most 64 parts, and 64 F is far below 2^32)
  unsigned const parts = (unsigned)P.splits;
  int const it_begin = parts == 1 ? 0 : (int)((unsigned)F * (unsigned)split / parts);
  int const it_end = parts == 1 ? F : (int)((unsigned)F * (unsigned)(split + 1) / parts);
  int const num_ops = uniform(P.num_ops);
  for (int it = it_begin; it < it_end; it++) {
    for (int o = 0; o < num_ops; o++) {
      DevOp const &op = P.ops[o];
      switch (uniform(op.kind)) {
        case DOP_LOAD: {
          if (uniform(op.hoist) && it > it_begin) {
            break;
          }
          DevTensor const &t = P.t[uniform(op.dst)];
          uint16_t *s = reinterpret_cast<uint16_t *>(lds + uniform(t.off));
          TileOrigin org = tile_origin(op, it, bx, by, bz);
          int const d_cols = uniform(op.d_cols);
          uint16_t const *g = static_cast<uint16_t const *>(P.in[uniform(op.io)]) + org.base +
                              (long long)org.row0 * d_cols + org.col0;
          if (uniform(op.vec8)) {
            int const cpr = uniform(t.cols) / 8, n = uniform(t.rows) * cpr;
            int const cols = uniform(t.cols);
            uint32_t const mcpr = (uint32_t)uniform((int)t.mcpr);
            for (int e = tid; e < n; e += kInterpThreads) {
              int const r = fdiv(e, mcpr), c = (e - r * cpr) * 8;
              uint4v v = *reinterpret_cast<uint4v const *>(g + (long long)r * d_cols + c);
              *reinterpret_cast<uint4v *>(s + r * cols + c) = v;
            }
          } else {
            int const cols = uniform(t.cols), n = uniform(t.rows) * cols;
            uint32_t const mcols = (uint32_t)uniform((int)t.mcols);
            for (int e = tid; e < n; e += kInterpThreads) {
              int const r = fdiv(e, mcols), c = e - r * cols;
              s[e] = g[(long long)r * d_cols + c];
            }
          }
          break;
        }
        case DOP_MATMUL: {
          // reference matmul.h:773-804
          DevTensor const &ta = P.t[op.src0], &tb = P.t[op.src1], &tc = P.t[op.dst];
          uint16_t const *A = reinterpret_cast<uint16_t const *>(lds + ta.off);
          uint16_t const *B = reinterpret_cast<uint16_t const *>(lds + tb.off);
          uint16_t *C = reinterpret_cast<uint16_t *>(lds + tc.off);
          int const m = ta.rows, k = ta.cols, n = tb.cols;
          if (op.mm_kc > 0 && op.sub == 1) {
            fp_matmul_mfma(A, B, C, m, n, k, op, lds + P.mm_off, tid);
          } else if (op.mm_kc > 0) {
            fp_matmul_packed(A, B, C, m, n, k, op, reinterpret_cast<uint32_t *>(lds + P.mm_off),
                             tid);
          } else {
            // shapes the packed path does not take; the modulus is applied every 4
            // products (4 * 25650^2 + 25650 < 2^32), same ring value as reducing each step
            int const total = m * n;
            for (int e = tid; e < total; e += kInterpThreads) {
              int const row = fdiv(e, tb.mcols), col = e - row * n;
              uint32_t acc = 0;
              int kk = 0;
              for (; kk + 4 <= k; kk += 4) {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                  acc += (uint32_t)A[row * k + kk + u] * B[(kk + u) * n + col];
                }
                acc %= FP_PQ;
              }
              for (; kk < k; kk++) {
                acc = (acc + (uint32_t)A[row * k + kk] * B[kk * n + col]) % FP_PQ;
              }
              C[e] = static_cast<uint16_t>(acc);
            }
          }
          break;
        }
        case DOP_UNARY: {
          DevTensor const &t = P.t[op.dst];
          uint16_t *p = reinterpret_cast<uint16_t *>(lds + t.off);
          int const n = t.rows * t.cols;
          // (16 bytes at a time; every tile starts on a 16-byte boundary)
          bool const exp = uniform(op.sub) == TB_EXP_OP;
          for (int e = tid; e < n / 8; e += kInterpThreads) {
            uint4v w = reinterpret_cast<uint4v const *>(p)[e];
#pragma unroll
            for (int j = 0; j < 4; j++) {
              uint32_t const lo = w[j] & 0xffffu, hi = w[j] >> 16;
              w[j] = exp ? lds_exp(tbl, lo) | (lds_exp(tbl, hi) << 16) : lds_silu(tbl, lo) | (lds_silu(tbl, hi) << 16);
            }
            reinterpret_cast<uint4v *>(p)[e] = w;
          }
          for (int e = n / 8 * 8 + tid; e < n; e += kInterpThreads) {
            p[e] = static_cast<uint16_t>(exp ? lds_exp(tbl, p[e]) : lds_silu(tbl, p[e]));
          }
          break;
        }
        case DOP_BINARY: {
          // reference element_binary.h:86-105; an operand dim is the output's or 1, so the
          // reference's `% dim` broadcast index is the output index or 0
          DevTensor const &t1 = P.t[op.src0], &t2 = P.t[op.src1], &to = P.t[op.dst];
          uint16_t const *x1 = reinterpret_cast<uint16_t const *>(lds + t1.off);
          uint16_t const *x2 = reinterpret_cast<uint16_t const *>(lds + t2.off);
          uint16_t *y = reinterpret_cast<uint16_t *>(lds + to.off);
          int const n = to.rows * to.cols;
          int const r1 = t1.rows == to.rows ? t1.cols : 0, c1 = t1.cols == to.cols ? 1 : 0;
          int const r2 = t2.rows == to.rows ? t2.cols : 0, c2 = t2.cols == to.cols ? 1 : 0;
          int const cols = uniform(to.cols);
          if (cols % 8 == 0) {
            // eight neighbours of a row at a time: an operand that has the row holds them in 16 bytes,
            // one that has a single column is the same for all
            int const cpr = cols / 8;
            auto eight = [&](uint16_t const *x, int at, int step) {
              if (step) {
                return *reinterpret_cast<uint4v const *>(x + at);
              }
              uint32_t const y = x[at] * 0x10001u;
              return uint4v{y, y, y, y};
            };
            for (int e = tid; e < n / 8; e += kInterpThreads) {
              int const r = fdiv(e, to.mcpr), c = (e - r * cpr) * 8;
              uint4v const a = eight(x1, r * r1 + c * c1, c1), b = eight(x2, r * r2 + c * c2, c2);
              uint4v z;
#pragma unroll
              for (int j = 0; j < 4; j++) {
                uint32_t const al = a[j] & 0xffffu, ah = a[j] >> 16, bl = b[j] & 0xffffu, bh = b[j] >> 16;
                z[j] = op.sub == TB_DIV_OP   ? lds_div(tbl, al, bl) | (lds_div(tbl, ah, bh) << 16)
                       : op.sub == TB_ADD_OP ? mod_pq(al + bl) | (mod_pq(ah + bh) << 16)
                                             : mod_pq(al * bl) | (mod_pq(ah * bh) << 16);
              }
              *reinterpret_cast<uint4v *>(y + e * 8) = z;
            }
            break;
          }
          for (int e = tid; e < n; e += kInterpThreads) {
            int const r = fdiv(e, to.mcols), c = e - r * to.cols;
            uint32_t a = x1[r * r1 + c * c1];
            uint32_t b = x2[r * r2 + c * c2];
            uint32_t z;
            if (op.sub == TB_DIV_OP) {
              z = lds_div(tbl, a, b);
            } else if (op.sub == TB_ADD_OP) {
              z = mod_pq(a + b);
            } else {
              z = mod_pq(a * b);
            }
            y[e] = static_cast<uint16_t>(z);
          }
          break;
        }
        case DOP_REDUCE: {
          // reference reduction.h:147-156; uint16 terms are summed unreduced in
          // 32 bits and folded every 32768 terms
          DevTensor const &ti = P.t[op.src0], &to = P.t[op.dst];
          uint16_t const *x = reinterpret_cast<uint16_t const *>(lds + ti.off);
          uint16_t *y = reinterpret_cast<uint16_t *>(lds + to.off);
          int const n = to.rows * to.cols, deg = op.red_deg, inner = op.red_inner;
          if (inner == 1 && deg >= 64) {
            // one output per 16 lanes: each lane strides the row, then the lanes fold
            int const lane16 = tid & 15;
            for (int e = tid >> 4; e < n; e += kInterpThreads / 16) {
              uint16_t const *row = x + e * deg;
              uint32_t r = 0;  // (an LDS tile is far too small to overflow 32 bits here)
              if (deg % 8 == 0) {
                for (int kk = lane16; kk < deg / 8; kk += 16) {
                  uint4v const w = reinterpret_cast<uint4v const *>(row)[kk];
#pragma unroll
                  for (int j = 0; j < 4; j++) {
                    r += (w[j] & 0xffffu) + (w[j] >> 16);
                  }
                }
              } else {
                for (int kk = lane16; kk < deg; kk += 16) {
                  r += row[kk];
                }
              }
              r %= FP_PQ;
              r += __shfl_xor(r, 8, 16);
              r += __shfl_xor(r, 4, 16);
              r += __shfl_xor(r, 2, 16);
              r += __shfl_xor(r, 1, 16);
              if (lane16 == 0) {
                y[e] = static_cast<uint16_t>(r % FP_PQ);
              }
            }
          } else {
            for (int e = tid; e < n; e += kInterpThreads) {
              int const outer = fdiv(e, op.mg0);
              int pos = outer * (inner * deg) + (e - outer * inner);
              uint32_t r = 0;
              for (int kk = 0; kk < deg; kk++, pos += inner) {
                r += x[pos];
                if ((kk & 32767) == 32767) {
                  r %= FP_PQ;
                }
              }
              y[e] = static_cast<uint16_t>(r % FP_PQ);
            }
          }
          break;
        }
        case DOP_CONCAT: {
          // reference concat.h:90-101
          DevTensor const &to = P.t[op.dst];
          uint16_t const *A = reinterpret_cast<uint16_t const *>(lds + P.t[op.src0].off);
          uint16_t const *B = reinterpret_cast<uint16_t const *>(lds + P.t[op.src1].off);
          uint16_t *y = reinterpret_cast<uint16_t *>(lds + to.off);
          int const n = to.rows * to.cols, a = op.cat_a, b = op.cat_b, inner = op.cat_inner;
          for (int e = tid; e < n; e += kInterpThreads) {
            int const ei = fdiv(e, op.mg0), in_i = e - ei * inner;
            int const outer = fdiv(ei, op.mg1), cd = ei - outer * (a + b);
            y[e] = cd < a ? A[in_i + cd * inner + outer * inner * a]
                          : B[in_i + (cd - a) * inner + outer * inner * b];
          }
          break;
        }
        case DOP_OUTPUT: {
          // reference output_saver.h:373-401 (accumulate) and :418-447 (store)
          DevTensor const &ti = P.t[uniform(op.src0)], &ta = P.t[uniform(op.dst)];
          uint16_t const *x = reinterpret_cast<uint16_t const *>(lds + uniform(ti.off));
          uint16_t *acc = reinterpret_cast<uint16_t *>(lds + uniform(ta.off));
          int const ta_rows = uniform(ta.rows), ta_cols = uniform(ta.cols), n = ta_rows * ta_cols;
          bool const last = (it == it_end - 1), first = (it == it_begin);
          TileOrigin org = tile_origin(op, 0, bx, by, bz);
          int const d_cols = uniform(op.d_cols), io = uniform(op.io);
          uint16_t *g = (P.splits > 1 ? P.part[io] + (long long)split * P.part_stride[io]
                                      : static_cast<uint16_t *>(P.out[io])) +
                        org.base + (long long)org.row0 * d_cols + org.col0;
          if (uniform(op.vec8)) {
            int const cpr = ta_cols / 8, n8 = ta_rows * cpr;
            uint32_t const mcpr = (uint32_t)uniform((int)ta.mcpr);
            for (int e = tid; e < n8; e += kInterpThreads) {
              uint4v v = *reinterpret_cast<uint4v const *>(x + e * 8);
              if (!first) {
                uint4v w = *reinterpret_cast<uint4v const *>(acc + e * 8);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                  v[j] = add_mod_pair(v[j], w[j]);
                }
              }
              if (last) {
                int const r = fdiv(e, mcpr), c = (e - r * cpr) * 8;
                *reinterpret_cast<uint4v *>(g + (long long)r * d_cols + c) = v;
              } else {
                *reinterpret_cast<uint4v *>(acc + e * 8) = v;
              }
            }
          } else {
            for (int e = tid; e < n; e += kInterpThreads) {
              uint32_t v = x[e];
              if (!first) {
                v = mod_pq(v + acc[e]);
              }
              if (last) {
                int const r = fdiv(e, ta.mcols), c = e - r * ta_cols;
                g[(long long)r * d_cols + c] = static_cast<uint16_t>(v);
              } else {
                acc[e] = static_cast<uint16_t>(v);
              }
            }
          }
          break;
        }
        default:
          break;
      }
      __syncthreads();
    }
  }
}


__device__ __forceinline__ void fp_load_tables(unsigned char *lds, uint16_t const *__restrict__ g_exp,
                                               uint16_t const *__restrict__ g_divp,
                                               uint16_t const *__restrict__ g_divq) {
  uint16_t *tbl = reinterpret_cast<uint16_t *>(lds);
  int const tid = threadIdx.x;
  for (int i = tid; i < (int)FP_Q; i += kInterpThreads) {
    tbl[i] = static_cast<uint16_t>(fp_from_residues(g_exp[i], 0u));
    tbl[384 + i] = g_divq[i];
  }
  for (int i = tid; i < (int)FP_P; i += kInterpThreads) {
    tbl[128 + i] = g_divp[i];
  }
}

__global__ __launch_bounds__(kInterpThreads) void fp_interp_kernel(
    DevProgram const P, uint16_t const *__restrict__ g_exp, uint16_t const *__restrict__ g_divp,
    uint16_t const *__restrict__ g_divq) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  // (the program record is an argument of 3 KB that the block walks operator by operator: all
  // of its lines in one trip)
  fetch_kernel_arguments_large<sizeof(DevProgram)>();
  fp_load_tables(lds, g_exp, g_divp, g_divq);
  __syncthreads();
  fp_interp_block(P, lds, blockIdx.x % P.grid[0], blockIdx.y, blockIdx.z, blockIdx.x / P.grid[0]);
}

// Many programs in one launch (a 1-D grid): workgroup w belongs to the program i with
// first_block[i] <= w < first_block[i + 1] and is workgroup w - first_block[i] of that
// program's own (grid.x * splits, grid.y, grid.z) grid.  The program record is copied from
// global memory to LDS (above every program's tiles, at `program_lds_offset`) once, so the
// interpreter reads it as it reads a kernel argument.
__global__ __launch_bounds__(kInterpThreads) void fp_interp_multi_kernel(
    DevProgram const *__restrict__ progs, int const *__restrict__ first_block, int n,
    int program_lds_offset, uint16_t const *__restrict__ g_exp,
    uint16_t const *__restrict__ g_divp, uint16_t const *__restrict__ g_divq) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int lo = 0, hi = n;
  int const w = blockIdx.x;
  while (hi - lo > 1) {
    int const mid = (lo + hi) / 2;
    if (first_block[mid] <= w) {
      lo = mid;
    } else {
      hi = mid;
    }
  }
  static_assert(sizeof(DevProgram) % 16 == 0, "the program record is copied in 16-byte words");
  uint4v const *src = reinterpret_cast<uint4v const *>(progs + lo);
  uint4v *dst = reinterpret_cast<uint4v *>(lds + program_lds_offset);
  for (int i = threadIdx.x; i < (int)(sizeof(DevProgram) / 16); i += kInterpThreads) {
    dst[i] = src[i];
  }
  fp_load_tables(lds, g_exp, g_divp, g_divq);
  __syncthreads();
  DevProgram const &P = *reinterpret_cast<DevProgram const *>(lds + program_lds_offset);
  int v = w - first_block[lo];
  int const gx = P.grid[0] * P.splits;
  int const x = v % gx;
  v /= gx;
  fp_interp_block(P, lds, x % P.grid[0], v % P.grid[1], v / P.grid[1], x / P.grid[0]);
}

// ===========================================================================
// fp16 interpreter
// ===========================================================================
__device__ __forceinline__ _Float16 *tile_ptr(unsigned char *lds, DevTensor const &t) {
  return reinterpret_cast<_Float16 *>(lds + t.off);
}

// C[m][n] = A[m][k] . B[k][n] on the matrix cores.  A is k-contiguous per row (cs == 1).
// B is either k-contiguous per column (rs == 1: one 16-byte LDS read per operand) or, the
// default, row-major as it was loaded (cs == 1): its operand is then gathered with
// transposing LDS reads (two 8-byte reads per operand, four k of sixteen columns each), so
// no tile is ever transposed while it is staged.  Row strides are multiples of 8 halfs.
// Wavefronts take output tiles round-robin.  Rows and columns past the end are clamped on
// read and masked on write.
// Transposing read: within 16 lanes, lane 4a + b names four halfs T[row0 + a][col0 + 4b ..]
// and lane i receives T[row0 + 0..3][col0 + i].
__device__ __forceinline__ half4 lds_tr16(_Float16 const *p) {
  typedef short short4v __attribute__((ext_vector_type(4)));
  short4v const v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (short4v __attribute__((address_space(3))) *)(__attribute__((address_space(3))) void *)(p));
  return __builtin_bit_cast(half4, v);
}
// B[krow .. krow + 7][col0 + lane % 16] for the 16 lanes of a group: `bp` is this lane's
// address inside rows krow .. krow + 3 (see b_tr_lane), rows + 4 are `rs` * 4 halfs further
__device__ __forceinline__ half8 b_frag_tr(_Float16 const *bp, int rs) {
  half4 const lo = lds_tr16(bp), hi = lds_tr16(bp + 4 * rs);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// this lane's address for the reads above: row (lane % 16) / 4, columns col0 + 4 * (lane % 4),
// kept inside the row when the tile has fewer than col0 + 16 columns (those output columns
// are masked)
__device__ __forceinline__ int b_tr_lane(int lane, int col0, int n, int rs) {
  int const a = (lane % 16) / 4;
  int col = col0 + 4 * (lane % 4);
  int const last = ((n + 3) / 4) * 4 - 4;
  col = col < last ? col : last;
  return a * rs + col;
}
template <int TILE>
__device__ __forceinline__ void mfma_matmul(unsigned char *lds, DevTensor const &ta,
                                            DevTensor const &tb, DevTensor const &tc, int wave,
                                            int lane, int num_waves) {
  _Float16 const *A = tile_ptr(lds, ta);
  _Float16 const *B = tile_ptr(lds, tb);
  _Float16 *C = tile_ptr(lds, tc);
  int const m = ta.rows, k = ta.cols, n = tb.cols;
  int const tiles_m = (m + TILE - 1) / TILE, tiles_n = (n + TILE - 1) / TILE;
  for (int tile = wave; tile < tiles_m * tiles_n; tile += num_waves) {
    int const tm = tile / tiles_n, tn = tile % tiles_n;
    if constexpr (TILE == 32) {
      int arow = tm * 32 + lane % 32;
      arow = arow < m ? arow : m - 1;
      _Float16 const *ap = A + arow * ta.rs + 8 * (lane / 32);
      bool const b_rows = tb.cs == 1;  // row-major B: transposing reads
      _Float16 const *bp = b_rows ? B + (8 * (lane / 32)) * tb.rs +
                                        b_tr_lane(lane, tn * 32 + 16 * ((lane / 16) % 2), n, tb.rs)
                                  : B + (tn * 32 + lane % 32) * tb.cs + 8 * (lane / 32);
      float16v acc;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        acc[i] = 0.0f;
      }
      for (int k0 = 0; k0 < k; k0 += 16) {
        half8 a = *reinterpret_cast<half8 const *>(ap + k0);
        half8 b = b_rows ? b_frag_tr(bp + k0 * tb.rs, tb.rs) : *reinterpret_cast<half8 const *>(bp + k0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; r++) {
        int row = tm * 32 + (r / 4) * 8 + (lane / 32) * 4 + (r % 4);
        int col = tn * 32 + lane % 32;
        if (row < m) {
          C[row * tc.rs + col * tc.cs] = static_cast<_Float16>(acc[r]);
        }
      }
    } else {
      int arow = tm * 16 + lane % 16;
      arow = arow < m ? arow : m - 1;
      _Float16 const *ap = A + arow * ta.rs;
      bool const b_rows = tb.cs == 1;  // row-major B: transposing reads
      int bcol = tn * 16 + lane % 16;
      bcol = bcol < n ? bcol : n - 1;
      _Float16 const *bp = b_rows ? B + b_tr_lane(lane, tn * 16, n, tb.rs) : B + bcol * tb.cs;
      float4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
      int k0 = 0;
      for (; k0 + 32 <= k; k0 += 32) {
        half8 a = *reinterpret_cast<half8 const *>(ap + k0 + 8 * (lane / 16));
        half8 b = b_rows ? b_frag_tr(bp + (k0 + 8 * (lane / 16)) * tb.rs, tb.rs)
                         : *reinterpret_cast<half8 const *>(bp + k0 + 8 * (lane / 16));
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc, 0, 0, 0);
      }
      for (; k0 + 16 <= k; k0 += 16) {
        half4 a = *reinterpret_cast<half4 const *>(ap + k0 + 4 * (lane / 16));
        half4 b = b_rows ? lds_tr16(bp + (k0 + 4 * (lane / 16)) * tb.rs)
                         : *reinterpret_cast<half4 const *>(bp + k0 + 4 * (lane / 16));
        acc = __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        int row = tm * 16 + (lane / 16) * 4 + r;
        int col = tn * 16 + lane % 16;
        if (row < m && col < n) {
          C[row * tc.rs + col * tc.cs] = static_cast<_Float16>(acc[r]);
        }
      }
    }
  }
}

// rows of 16-byte pieces: element-wise statements then move eight halfs per LDS access
__device__ __forceinline__ bool vec_tile(DevTensor const &t) {
  return t.cs == 1 && t.rs % 8 == 0 && t.cols % 8 == 0;
}
__device__ __forceinline__ half8 splat8(_Float16 x) {
  half8 v = {x, x, x, x, x, x, x, x};
  return v;
}

// `trace` (null unless the phase trace option is on): the first workgroup's first thread
// stamps the 100 MHz clock at its start and after every statement's barrier; trace[0] counts
// the stamps that follow it.
__global__ __launch_bounds__(kInterpThreads) void f16_interp_kernel(DevProgram const P,
                                                                    unsigned long long *trace) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  fetch_kernel_arguments_large<sizeof(DevProgram)>();  // (the program record, walked operator by operator)
  int const tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  int const F = P.forloop_range;
  bool const tracing = trace != nullptr && tid == 0 && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0;
  unsigned long long stamps = 0;
  if (tracing) {
    trace[++stamps] = __builtin_amdgcn_s_memrealtime();
  }
  for (int it = 0; it < F; it++) {
    for (int o = 0; o < P.num_ops; o++) {
      DevOp const &op = P.ops[o];
      switch (op.kind) {
        case DOP_LOAD: {
          if (op.hoist && it > 0) {
            break;
          }
          DevTensor const &t = P.t[op.dst];
          _Float16 *s = tile_ptr(lds, t);
          TileOrigin org = tile_origin(op, it, blockIdx.x);
          _Float16 const *g = static_cast<_Float16 const *>(P.in[op.io]) + org.base;
          // A column-major device tensor (element (r, c) at c * d_rows + r) is walked as the
          // row-major matrix of its transpose: rows and columns, origins and the tile's LDS
          // strides swap roles, and the 16-byte pieces run down the tile's columns.
          bool const cm = op.sub == 1;
          int const vrows = cm ? t.cols : t.rows, vcols = cm ? t.rows : t.cols;
          int const ld = cm ? op.d_rows : op.d_cols;
          int const r0 = cm ? org.col0 : org.row0, c0 = cm ? org.row0 : org.col0;
          int const srs = cm ? t.cs : t.rs, scs = cm ? t.rs : t.cs;
          if (op.vec8) {
            int const cpr = vcols / 8, n = vrows * cpr;
            uint32_t const magic = cm ? op.mg1 : t.mcpr;
            for (int e = tid; e < n; e += kInterpThreads) {
              int const r = fdiv(e, magic), c = (e - r * cpr) * 8;
              half8 v = *reinterpret_cast<half8 const *>(g + (long long)(r0 + r) * ld + c0 + c);
              if (op.vec8 == 1) {
                *reinterpret_cast<half8 *>(s + r * srs + c) = v;
              } else {
#pragma unroll
                for (int j = 0; j < 8; j++) {
                  s[r * srs + (c + j) * scs] = v[j];
                }
              }
            }
          } else {
            int const n = vrows * vcols;
            uint32_t const magic = cm ? op.mg0 : t.mcols;
            for (int e = tid; e < n; e += kInterpThreads) {
              int const r = fdiv(e, magic), c = e - r * vcols;
              s[r * srs + c * scs] = g[(long long)(r0 + r) * ld + c0 + c];
            }
          }
          break;
        }
        case DOP_MATMUL: {
          DevTensor const &ta = P.t[op.src0], &tb = P.t[op.src1], &tc = P.t[op.dst];
          int const m = ta.rows, k = ta.cols, n = tb.cols;
          // (any m and n: rows and columns past the end are clamped on read, masked on write)
          bool const fast = ta.cs == 1 && ta.rs % 8 == 0 && k % 16 == 0 &&
                            ((tb.rs == 1 && tb.cs % 8 == 0) || (tb.cs == 1 && tb.rs % 4 == 0 && n >= 4));
          if (fast && m % 32 == 0 && n % 32 == 0) {
            mfma_matmul<32>(lds, ta, tb, tc, wave, lane, kInterpThreads / 64);
          } else if (fast) {
            mfma_matmul<16>(lds, ta, tb, tc, wave, lane, kInterpThreads / 64);
          } else {
            _Float16 const *A = tile_ptr(lds, ta);
            _Float16 const *B = tile_ptr(lds, tb);
            _Float16 *C = tile_ptr(lds, tc);
            for (int e = tid; e < m * n; e += kInterpThreads) {
              int const row = fdiv(e, tb.mcols), col = e - row * n;
              float acc = 0.0f;
              for (int kk = 0; kk < k; kk++) {
                acc = __builtin_fmaf(static_cast<float>(A[row * ta.rs + kk * ta.cs]),
                                     static_cast<float>(B[kk * tb.rs + col * tb.cs]), acc);
              }
              // rounded to fp32 first and to fp16 second: the fence keeps the last multiply-add
              // and the conversion from merging into one instruction that rounds once
              asm volatile("" : "+v"(acc));
              C[row * tc.rs + col * tc.cs] = static_cast<_Float16>(acc);
            }
          }
          break;
        }
        case DOP_UNARY: {
          DevTensor const &t = P.t[op.dst];
          _Float16 *p = tile_ptr(lds, t);
          int const n = t.rows * t.cols;
          bool const is_exp = op.sub == TB_EXP_OP;
          if (vec_tile(t)) {
            int const cpr = t.cols / 8;
            for (int e = tid; e < n / 8; e += kInterpThreads) {
              int const r = fdiv(e, t.mcpr), c = (e - r * cpr) * 8;
              half8 *q = reinterpret_cast<half8 *>(p + r * t.rs + c);
              half8 v = *q;
#pragma unroll
              for (int j = 0; j < 8; j++) {
                float const x = static_cast<float>(v[j]);
                v[j] = static_cast<_Float16>(is_exp ? __expf(x) : x / (1.0f + __expf(-x)));
              }
              *q = v;
            }
            break;
          }
          for (int e = tid; e < n; e += kInterpThreads) {
            int const r = fdiv(e, t.mcols), c = e - r * t.cols;
            _Float16 *q = p + r * t.rs + c * t.cs;
            float x = static_cast<float>(*q);
            float y = is_exp ? __expf(x) : x / (1.0f + __expf(-x));
            *q = static_cast<_Float16>(y);
          }
          break;
        }
        case DOP_BINARY: {
          DevTensor const &t1 = P.t[op.src0], &t2 = P.t[op.src1], &to = P.t[op.dst];
          _Float16 const *x1 = tile_ptr(lds, t1);
          _Float16 const *x2 = tile_ptr(lds, t2);
          _Float16 *y = tile_ptr(lds, to);
          int const n = to.rows * to.cols;
          // an operand dim is either the output's or 1 (checked by the lowering): broadcast = index 0
          bool const r1 = t1.rows > 1, c1 = t1.cols > 1, r2 = t2.rows > 1, c2 = t2.cols > 1;
          // an operand with columns is read eight at a time, one without is one value per row
          bool const v1 = !c1 || (t1.cs == 1 && (t1.rs % 8 == 0 || !r1));
          bool const v2 = !c2 || (t2.cs == 1 && (t2.rs % 8 == 0 || !r2));
          if (vec_tile(to) && v1 && v2) {
            int const cpr = to.cols / 8;
            for (int e = tid; e < n / 8; e += kInterpThreads) {
              int const r = fdiv(e, to.mcpr), c = (e - r * cpr) * 8;
              _Float16 const *p1 = x1 + (r1 ? r : 0) * t1.rs, *p2 = x2 + (r2 ? r : 0) * t2.rs;
              half8 const a8 = c1 ? *reinterpret_cast<half8 const *>(p1 + c) : splat8(*p1);
              half8 const b8 = c2 ? *reinterpret_cast<half8 const *>(p2 + c) : splat8(*p2);
              half8 z8;
#pragma unroll
              for (int j = 0; j < 8; j++) {
                float const a = static_cast<float>(a8[j]), b = static_cast<float>(b8[j]);
                float const z = (op.sub == TB_DIV_OP) ? a / b : (op.sub == TB_ADD_OP) ? a + b : a * b;
                z8[j] = static_cast<_Float16>(z);
              }
              *reinterpret_cast<half8 *>(y + r * to.rs + c) = z8;
            }
            break;
          }
          for (int e = tid; e < n; e += kInterpThreads) {
            int const r = fdiv(e, to.mcols), c = e - r * to.cols;
            float a = static_cast<float>(x1[(r1 ? r : 0) * t1.rs + (c1 ? c : 0) * t1.cs]);
            float b = static_cast<float>(x2[(r2 ? r : 0) * t2.rs + (c2 ? c : 0) * t2.cs]);
            float z = (op.sub == TB_DIV_OP) ? a / b : (op.sub == TB_ADD_OP) ? a + b : a * b;
            y[r * to.rs + c * to.cs] = static_cast<_Float16>(z);
          }
          break;
        }
        case DOP_REDUCE: {
          DevTensor const &ti = P.t[op.src0], &to = P.t[op.dst];
          _Float16 const *x = tile_ptr(lds, ti);
          _Float16 *y = tile_ptr(lds, to);
          int const n = to.rows * to.cols, deg = op.red_deg, inner = op.red_inner;
          // Along the columns of a row (output (r, c) = sum over j of x[r][c + j inner]) or along
          // the rows (output (r, c) = sum over j of x[r + j to.rows][c]): no division in the sum.
          // Long sums are shared by 16 lanes (fp32 parts, added across the lanes at the end).
          bool const along_cols = to.rows == ti.rows;
          int const lanes = (deg >= 64 && n * 16 <= 4 * kInterpThreads) ? 16 : 1;
          int const step = along_cols ? inner * ti.cs : to.rows * ti.rs;
          if (along_cols && inner == 1 && ti.cs == 1 && ti.rs % 8 == 0 && deg % 8 == 0) {
            // a run of consecutive elements: each lane adds pieces of eight, one after the
            // other in element order (with one lane this is the plain order)
            for (int e0 = 0; e0 < n; e0 += kInterpThreads / lanes) {
              int const e = e0 + tid / lanes, part = tid % lanes;
              float r = 0.0f;
              if (e < n) {
                int const orow = fdiv(e, to.mcols), ocol = e - orow * to.cols;
                _Float16 const *src = x + orow * ti.rs + ocol;
                for (int kk = 8 * part; kk < deg; kk += 8 * lanes) {
                  half8 const v = *reinterpret_cast<half8 const *>(src + kk);
#pragma unroll
                  for (int j = 0; j < 8; j++) {
                    r += static_cast<float>(v[j]);
                  }
                }
              }
              if (lanes == 16) {
                r += __shfl_xor(r, 1, 64);
                r += __shfl_xor(r, 2, 64);
                r += __shfl_xor(r, 4, 64);
                r += __shfl_xor(r, 8, 64);
              }
              if (e < n && part == 0) {
                int const orow = fdiv(e, to.mcols), ocol = e - orow * to.cols;
                y[orow * to.rs + ocol * to.cs] = static_cast<_Float16>(r);
              }
            }
            break;
          }
          if (vec_tile(to) && ti.cs == 1 && ti.rs % 8 == 0 && (!along_cols || inner % 8 == 0)) {
            // eight neighbouring outputs per lane, each with the element order of the plain loop
            int const cpr = to.cols / 8;
            for (int e0 = 0; e0 < n / 8; e0 += kInterpThreads / lanes) {
              int const e = e0 + tid / lanes, part = tid % lanes;
              float r[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
              int const orow = fdiv(e, to.mcpr), ocol = (e - orow * cpr) * 8;
              if (e < n / 8) {
                _Float16 const *src = x + orow * ti.rs + ocol + part * step;
                for (int kk = part; kk < deg; kk += lanes, src += lanes * step) {
                  half8 const v = *reinterpret_cast<half8 const *>(src);
#pragma unroll
                  for (int j = 0; j < 8; j++) {
                    r[j] += static_cast<float>(v[j]);
                  }
                }
              }
              if (lanes == 16) {
#pragma unroll
                for (int j = 0; j < 8; j++) {
                  r[j] += __shfl_xor(r[j], 1, 64);
                  r[j] += __shfl_xor(r[j], 2, 64);
                  r[j] += __shfl_xor(r[j], 4, 64);
                  r[j] += __shfl_xor(r[j], 8, 64);
                }
              }
              if (e < n / 8 && part == 0) {
                half8 h;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                  h[j] = static_cast<_Float16>(r[j]);
                }
                *reinterpret_cast<half8 *>(y + orow * to.rs + ocol) = h;
              }
            }
            break;
          }
          for (int e0 = 0; e0 < n; e0 += kInterpThreads / lanes) {
            int const e = e0 + tid / lanes, part = tid % lanes;
            float r = 0.0f;
            if (e < n) {
              int const orow = fdiv(e, to.mcols), ocol = e - orow * to.cols;
              _Float16 const *src = x + orow * ti.rs + ocol * ti.cs + part * step;
              for (int kk = part; kk < deg; kk += lanes, src += lanes * step) {
                r += static_cast<float>(*src);
              }
            }
            if (lanes == 16) {
              r += __shfl_xor(r, 1, 64);
              r += __shfl_xor(r, 2, 64);
              r += __shfl_xor(r, 4, 64);
              r += __shfl_xor(r, 8, 64);
            }
            if (e < n && part == 0) {
              int const orow = fdiv(e, to.mcols), ocol = e - orow * to.cols;
              y[orow * to.rs + ocol * to.cs] = static_cast<_Float16>(r);
            }
          }
          break;
        }
        case DOP_CONCAT: {
          DevTensor const &t1 = P.t[op.src0], &t2 = P.t[op.src1], &to = P.t[op.dst];
          _Float16 const *A = tile_ptr(lds, t1);
          _Float16 const *B = tile_ptr(lds, t2);
          _Float16 *y = tile_ptr(lds, to);
          int const n = to.rows * to.cols;
          bool const along_cols = (op.cat_inner == 1 && t1.rows == to.rows);
          for (int e = tid; e < n; e += kInterpThreads) {
            int const r = fdiv(e, to.mcols), c = e - r * to.cols;
            _Float16 v;
            if (along_cols) {
              v = c < t1.cols ? A[r * t1.rs + c * t1.cs] : B[r * t2.rs + (c - t1.cols) * t2.cs];
            } else {
              v = r < t1.rows ? A[r * t1.rs + c * t1.cs] : B[(r - t1.rows) * t2.rs + c * t2.cs];
            }
            y[r * to.rs + c * to.cs] = v;
          }
          break;
        }
        case DOP_OUTPUT: {
          // accumulators start at zero and take `acc + x`, rounded to fp16 every
          // iteration (triton_code_gen.cc:223-232); stored once after the loop
          DevTensor const &ti = P.t[op.src0], &ta = P.t[op.dst];
          _Float16 const *x = tile_ptr(lds, ti);
          _Float16 *acc = tile_ptr(lds, ta);
          int const n = ta.rows * ta.cols;
          bool const last = (it == F - 1);
          TileOrigin org = tile_origin(op, 0, blockIdx.x);
          _Float16 *g = static_cast<_Float16 *>(P.out[op.io]) + org.base;
          if (op.vec8 && vec_tile(ti)) {
            int const cpr = ta.cols / 8;
            for (int e = tid; e < n / 8; e += kInterpThreads) {
              int const r = fdiv(e, ta.mcpr), c = (e - r * cpr) * 8;
              half8 v = *reinterpret_cast<half8 const *>(x + r * ti.rs + c);
              if (it > 0) {
                half8 const a = *reinterpret_cast<half8 const *>(acc + r * ta.rs + c);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                  v[j] = static_cast<_Float16>(static_cast<float>(v[j]) + static_cast<float>(a[j]));
                }
              }
              if (last) {
                *reinterpret_cast<half8 *>(g + (long long)(org.row0 + r) * op.d_cols + org.col0 + c) = v;
              } else {
                *reinterpret_cast<half8 *>(acc + r * ta.rs + c) = v;
              }
            }
            break;
          }
          for (int e = tid; e < n; e += kInterpThreads) {
            int const r = fdiv(e, ta.mcols), c = e - r * ta.cols;
            float v = static_cast<float>(x[r * ti.rs + c * ti.cs]);
            if (it > 0) {
              v += static_cast<float>(acc[r * ta.rs + c * ta.cs]);
            }
            _Float16 h = static_cast<_Float16>(v);
            if (last) {
              // (op.sub == 1: a column-major device tensor, element (r, c) at c * d_rows + r)
              g[op.sub == 1 ? (long long)(org.col0 + c) * op.d_rows + org.row0 + r
                            : (long long)(org.row0 + r) * op.d_cols + org.col0 + c] = h;
            } else {
              acc[r * ta.rs + c * ta.cs] = h;
            }
          }
          break;
        }
        default:
          break;
      }
      __syncthreads();
      if (tracing && stamps < 4000) {
        trace[++stamps] = __builtin_amdgcn_s_memrealtime();
      }
    }
  }
  if (tracing) {
    trace[0] = stamps;
  }
}

// ===========================================================================
// launchers
// ===========================================================================
// out[e] = sum over splits of part[split * n + e] (mod 25651)
__global__ void fp_combine_splits_kernel(uint16_t const *__restrict__ part,
                                         uint16_t *__restrict__ out, long long n,
                                         long long stride_elems, int splits) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  long long const stride = (long long)gridDim.x * blockDim.x;
  for (; i < n; i += stride) {
    uint32_t v = 0;
    for (int s = 0; s < splits; s++) {
      v += part[(long long)s * stride_elems + i];  // splits <= 64: far from 2^32
    }
    out[i] = static_cast<uint16_t>(v % FP_PQ);
  }
}

// pinned host buffer -> device buffer, 16 bytes per lane
__global__ void stage_records_kernel(uint4v const *__restrict__ src, uint4v *__restrict__ dst, int n16) {
  int const i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n16) {
    dst[i] = src[i];
  }
}

// The same for many (partials, output) pairs in one launch; job j owns workgroups
// [first_block[j], first_block[j + 1]).
struct CombineJob {
  uint16_t const *part;
  uint16_t *out;
  long long n, stride_elems;
  int splits, pad;
};
__global__ void fp_combine_splits_multi_kernel(CombineJob const *__restrict__ jobs,
                                               int const *__restrict__ first_block, int n_jobs) {
  int lo = 0, hi = n_jobs;
  int const w = blockIdx.x;
  while (hi - lo > 1) {
    int const mid = (lo + hi) / 2;
    if (first_block[mid] <= w) {
      lo = mid;
    } else {
      hi = mid;
    }
  }
  CombineJob const J = jobs[lo];
  long long const blocks = first_block[lo + 1] - first_block[lo];
  long long i = (long long)(w - first_block[lo]) * blockDim.x + threadIdx.x;
  long long const stride = blocks * blockDim.x;
  for (; i < J.n; i += stride) {
    uint32_t v = 0;
    for (int s = 0; s < J.splits; s++) {
      v += J.part[(long long)s * J.stride_elems + i];
    }
    J.out[i] = static_cast<uint16_t>(v % FP_PQ);
  }
}

// How many workgroups share one logical block's for-loop in the uint16 interpreter.
// The accumulating saver is a sum over iterations in a ring, so any split of the
// iteration range gives the same value; small grids are split until the device is full.
// `wanted` splits at most, fewer if the partial sums do not fit what is left of this queue's
// scratch after `used` bytes; the partials are placed there and `used` advances.
static void set_splits(DevProgram &prog, PlanExtents const &ext, int num_outputs, int wanted,
                       size_t &used) {
  State &s = state();
  prog.splits = 1;
  if (wanted < 2 || s.scratch() == nullptr) {
    return;
  }
  long long elems = 0;
  for (int i = 0; i < num_outputs; i++) {
    elems += (ext.out_elems[i] + 7) / 8 * 8;
  }
  int splits = wanted;
  while (splits > 1 && used + (size_t)(elems * splits * 2) > s.scratch_bytes) {
    splits--;
  }
  if (splits < 2) {
    return;
  }
  prog.splits = splits;
  uint16_t *p = reinterpret_cast<uint16_t *>(static_cast<char *>(s.scratch()) + used);
  for (int i = 0; i < num_outputs; i++) {
    prog.part[i] = p;
    prog.part_elems[i] = ext.out_elems[i];
    prog.part_stride[i] = (ext.out_elems[i] + 7) / 8 * 8;
    p += prog.part_stride[i] * splits;
  }
  used += (size_t)(elems * splits * 2);
}

static void choose_splits(DevProgram &prog, PlanExtents const &ext, int num_outputs) {
  prog.splits = 1;
  int const blocks = (int)fp_program_blocks(prog);
  int const F = prog.forloop_range;
  if (F < 2 || blocks >= 192 || prog.fused == 5) {
    return;
  }
  size_t used = 0;
  set_splits(prog, ext, num_outputs, std::min(std::min(F, 64), (256 + blocks - 1) / blocks), used);
}

// `ext_out` set: the caller decides about split for-loops itself (batched launches).
// `interpreter`: lower for the generic interpreter whatever kernel would recognise the plan.
static int prepare(mi355_plan const *plan, void const *const *inputs, void *const *outputs,
                   bool f16, DevProgram &prog, PlanExtents *ext_out = nullptr, bool interpreter = false) {
  if (plan == nullptr || inputs == nullptr || outputs == nullptr) {
    return fail(MI355_ERR_INVALID, "null argument");
  }
  PlanExtents ext;
  std::string err;
  bool const try_fused = f16 && !state().force_interpreter && !interpreter;
  // a fused kernel keeps tiles in registers, so the interpreter's LDS need does not
  // bound it: lower without the limit first, and again with it if no fused kernel fits
  bool const declared = f16 && state().plan_smem_layout != 0;
  // (only a load-load-matmul-save plan can take the fused fingerprint kernel: everything
  // else is lowered once, with the limit)
  // (load, load, [exp / silu]*, matmul, [exp / silu], save)
  bool try_fused_fp = !f16 && !state().force_interpreter && plan->num_operators >= 4 &&
                      plan->num_operators <= 7 && plan->operator_types[0] == TB_INPUT_OP &&
                      plan->operator_types[1] == TB_INPUT_OP &&
                      plan->operator_types[plan->num_operators - 1] == TB_OUTPUT_OP;
  int matmuls = 0;
  for (int o = 2; try_fused_fp && o < plan->num_operators - 1; o++) {
    int const t = plan->operator_types[o];
    matmuls += t == TB_MATMUL_OP ? 1 : 0;
    try_fused_fp = t == TB_MATMUL_OP || t == TB_EXP_OP || t == TB_SILU_OP;
  }
  try_fused_fp = try_fused_fp && matmuls == 1;
  // (three loaders, two matmuls, one exponential)
  int kinds[3] = {0, 0, 0};
  for (int o = 0; o < plan->num_operators; o++) {
    int const t = plan->operator_types[o];
    kinds[0] += t == TB_INPUT_OP ? 1 : 0;
    kinds[1] += t == TB_MATMUL_OP ? 1 : 0;
    kinds[2] += t == TB_EXP_OP ? 1 : 0;
  }
  bool const try_fp_attention = !f16 && !state().force_interpreter && state().fp_vector_dot_only == 0 && kinds[0] == 3 && kinds[1] == 2 && kinds[2] == 1;
  int rc = compile_plan(*plan, f16, (try_fused || try_fused_fp || try_fp_attention) ? (1 << 30) : state().max_lds, prog, ext,
                        err, declared);
  if (rc != MI355_OK) {
    return fail(rc, "%s", err.c_str());
  }
  if (try_fp_attention) {
    for (int i = 0; i < plan->num_dmem_inputs; i++) {
      prog.in[i] = inputs[i];
    }
    for (int i = 0; i < plan->num_dmem_outputs; i++) {
      prog.out[i] = outputs[i];
    }
    if (!fp_attn_applicable(prog)) {
      rc = compile_plan(*plan, false, state().max_lds, prog, ext, err);
      if (rc != MI355_OK) {
        return fail(rc, "%s", err.c_str());
      }
    }
  }
  if (try_fused_fp) {
    // the fused fingerprint matmul keeps no tile in LDS either: same two-step lowering
    for (int i = 0; i < plan->num_dmem_inputs; i++) {
      prog.in[i] = inputs[i];
    }
    for (int i = 0; i < plan->num_dmem_outputs; i++) {
      prog.out[i] = outputs[i];
    }
    // a plan with an operand prologue can only run on the matrix-core route: it must fit
    size_t need = 0;
    bool fused = fp_gemm_applicable(prog);
    if (fused && fp_needs_matrix_cores(prog) &&
        !(fp_mfma_gemm_fits(prog, ext, &need) && need <= state().planes_bytes)) {
      fused = false;
    }
    if (!fused) {
      rc = compile_plan(*plan, false, state().max_lds, prog, ext, err);
      if (rc != MI355_OK) {
        return fail(rc, "%s", err.c_str());
      }
    }
  }
  auto bind = [&]() {
    for (int i = 0; i < plan->num_dmem_inputs; i++) {
      prog.in[i] = inputs[i];
    }
    for (int i = 0; i < plan->num_dmem_outputs; i++) {
      prog.out[i] = outputs[i];
    }
  };
  if (try_fused) {
    bind();
    if (attention_applicable(prog)) {
      prog.fused = 1;
    } else if (gemm_applicable(prog)) {
      prog.fused = 2;
    } else if (combine_applicable(prog)) {
      prog.fused = 3;
    } else {
      rc = compile_plan(*plan, f16, state().max_lds, prog, ext, err, declared);
      if (rc != MI355_OK) {
        return fail(rc, "%s", err.c_str());
      }
    }
  }
  for (int i = 0; i < plan->num_dmem_inputs; i++) {
    if (inputs[i] == nullptr) {
      return fail(MI355_ERR_INVALID, "input %d is null", i);
    }
    prog.in[i] = inputs[i];
  }
  for (int i = 0; i < plan->num_dmem_outputs; i++) {
    if (outputs[i] == nullptr) {
      return fail(MI355_ERR_INVALID, "output %d is null", i);
    }
    prog.out[i] = outputs[i];
  }
  // a fused matmul plan launched by itself takes the matrix cores when its operand tensors'
  // residue planes fit this queue's plane memory (a batch places the planes of its members)
  if (!f16 && prog.fused == 4 && ext_out == nullptr) {
    size_t need = 0;
    if (fp_mfma_gemm_fits(prog, ext, &need) && need <= state().planes_bytes) {
      fp_mfma_gemm_bind(prog, state().planes(), 256);
    }
  }
  if (ext_out != nullptr) {
    *ext_out = ext;
    prog.splits = 1;
  } else if (!f16) {
    choose_splits(prog, ext, plan->num_dmem_outputs);
  }
  // 16-byte global accesses also need 16-byte aligned base pointers
  for (int o = 0; o < prog.num_ops; o++) {
    DevOp &d = prog.ops[o];
    if (d.kind == DOP_LOAD && d.vec8 && (reinterpret_cast<uintptr_t>(prog.in[d.io]) & 15) != 0) {
      d.vec8 = 0;
    }
  }
  return MI355_OK;
}

static int fold_splits(DevProgram const &prog) {
  State &s = state();
  for (int o = 0; o < MI355_MAX_DMEM_OUTPUTS; o++) {
    if (prog.out[o] == nullptr || prog.part_elems[o] <= 0) {
      continue;
    }
    long long const n = prog.part_elems[o];
    int const blocks = (int)std::min<long long>((n + 255) / 256, 2048);
    MI355_HIP(launch_kernel(fp_combine_splits_kernel, blocks, 256, 0, s.stream(), prog.part[o],
                            static_cast<uint16_t *>(prog.out[o]), n, prog.part_stride[o], prog.splits));
  }
  return MI355_OK;
}

// What launch() returns when the fused kernel a program was recognised for does not take its
// addresses (tile origins beyond 31 bits, say): the program runs on the interpreter instead.
constexpr int kDeclined = 1;

static int launch(DevProgram const &prog, bool f16) {
  State &s = state();
  if (!f16 && prog.fused == 4) {
    if (!prog.fg[5] && fp_needs_matrix_cores(prog)) {
      return fail(MI355_ERR_UNSUPPORTED, "operand prologue without the matrix-core route");
    }
    if (int rc = prog.fg[5] ? launch_fp_mfma_gemm(prog, s.stream()) : launch_fp_gemm(prog, s.stream())) {
      return rc;
    }
    if (prog.splits > 1) {
      if (int rc = fold_splits(prog)) {
        return rc;
      }
    }
    s.last().kernel_id = MI355_KERNEL_FP_GEMM;
    s.last().workgroups = (int)fp_program_blocks(prog);
    s.last().threads = kInterpThreads;
    s.last().lds_bytes = prog.lds_bytes;
    s.last().row_split = prog.splits;
    return MI355_OK;
  }
  if (!f16 && prog.fused == 5) {
    if (int rc = launch_fp_attn(prog, s.stream())) {
      return rc;
    }
    s.last().kernel_id = MI355_KERNEL_FP_ATTENTION;
    s.last().workgroups = (int)fp_program_blocks(prog);
    s.last().threads = kInterpThreads;
    s.last().lds_bytes = prog.lds_bytes;
    s.last().row_split = 1;
    return MI355_OK;
  }
  if (prog.fused != 0) {
    int rc = prog.fused == 1   ? try_launch_attention(prog)
             : prog.fused == 2 ? try_launch_gemm(prog)
                               : try_launch_combine(prog);
    return rc == 1 ? MI355_OK : (rc < 0 ? rc : kDeclined);
  }
  dim3 grid(prog.grid[0] * (f16 ? 1 : prog.splits), prog.grid[1], prog.grid[2]);
  if (int const rc = f16 ? 0 : try_launch_fp_combine(prog)) {
    return rc == 1 ? MI355_OK : rc;
  }
  if (f16) {
    MI355_GRANT_LDS(f16_interp_kernel, prog.lds_bytes);
    MI355_HIP(launch_kernel(f16_interp_kernel, grid, kInterpThreads, prog.lds_bytes, s.stream(), prog, s.phase_trace));
  } else {
    MI355_GRANT_LDS(fp_interp_kernel, prog.lds_bytes);
    MI355_HIP(launch_kernel(fp_interp_kernel, grid, kInterpThreads, prog.lds_bytes, s.stream(), prog, s.exp_tbl, s.div_p,
                            s.div_q));
    if (prog.splits > 1) {
      if (int rc = fold_splits(prog)) {
        return rc;
      }
    }
  }
  s.last().kernel_id = f16 ? MI355_KERNEL_F16_INTERP : MI355_KERNEL_FP_INTERP;
  s.last().workgroups = (int)(grid.x * grid.y * grid.z);
  s.last().threads = kInterpThreads;
  s.last().lds_bytes = prog.lds_bytes;
  s.last().row_split = 1;
  return MI355_OK;
}

// One call of a customized operator: lowered and launched (or, under a recorder, recorded).  `prog` is what
// prepare() made of the same plan and tensors.
static int launch_plan(mi355_plan const *plan, void const *const *inputs, void *const *outputs, bool f16, DevProgram &prog) {
  int rc = launch(prog, f16);
  if (rc == kDeclined) {
    if ((rc = prepare(plan, inputs, outputs, f16, prog, nullptr, true)) == MI355_OK) {
      rc = launch(prog, f16);
    }
  }
  return rc;
}
static int run_plan(mi355_plan const *plan, void const *const *inputs, void *const *outputs, bool f16) {
  DevProgram prog;
  int const rc = prepare(plan, inputs, outputs, f16, prog);
  return rc != MI355_OK ? rc : launch_plan(plan, inputs, outputs, f16, prog);
}

}  // namespace mi355

using namespace mi355;

extern "C" int mi355_plan_extents(mi355_plan const *plan, long long *in_elems,
                                  long long *out_elems, int *lds_bytes_fp, int *lds_bytes_f16) {
  if (plan == nullptr) {
    return fail(MI355_ERR_INVALID, "null plan");
  }
  DevProgram prog;
  PlanExtents ext;
  std::string err;
  int rc = compile_plan(*plan, false, 1 << 30, prog, ext, err);
  if (rc != MI355_OK) {
    return fail(rc, "%s", err.c_str());
  }
  for (int i = 0; i < MI355_MAX_DMEM_INPUTS; i++) {
    if (in_elems != nullptr) {
      in_elems[i] = ext.in_elems[i];
    }
    if (out_elems != nullptr) {
      out_elems[i] = ext.out_elems[i];
    }
  }
  if (lds_bytes_fp != nullptr) {
    *lds_bytes_fp = prog.lds_bytes;
  }
  if (lds_bytes_f16 != nullptr) {
    rc = compile_plan(*plan, true, 1 << 30, prog, ext, err);
    if (rc != MI355_OK) {
      return fail(rc, "%s", err.c_str());
    }
    *lds_bytes_f16 = prog.lds_bytes;
  }
  return MI355_OK;
}

extern "C" int mi355_customized_fp(mi355_plan const *plan, void const *const *inputs,
                                   void *const *outputs) {
  MI355_REQUIRE_INIT();
  return run_plan(plan, inputs, outputs, false);
}

// ---- the entry point that allocates nothing ----------------------------------------------
// The partial sums of a split for-loop normally go to a scratch slab that mi355_init takes
// from the device allocator.  For callers that cannot have the library allocate or touch
// allocator-owned memory on their behalf, the same two kernels run with the partial sums in
// a file-scope device array instead.  `scratch` names the array on the host side only as a
// symbol: its device address is looked up once per device (static_scratch_setup, from
// mi355_init, with that device current) and only that address is ever handed to a kernel.
static __device__ __align__(256) unsigned char scratch[MI355_STATIC_SCRATCH_BYTES];
constexpr int kMaxDevices = 16;
static void *g_static_scratch[kMaxDevices] = {};

namespace mi355 {
int static_scratch_setup(int device) {
  if (device < 0 || device >= kMaxDevices) {
    return fail(MI355_ERR_INVALID, "device %d out of range", device);
  }
  void *ptr = nullptr;
  MI355_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  if (ptr == nullptr) {
    return fail(MI355_ERR_HIP, "hipGetSymbolAddress returned a null address for the static scratch");
  }
  g_static_scratch[device] = ptr;
  // raised here, not lazily at the first large launch: the entry point itself then makes no
  // call besides its two kernel launches
  MI355_HIP(hipFuncSetAttribute(reinterpret_cast<void const *>(fp_interp_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, state().max_lds));
  return MI355_OK;
}
}  // namespace mi355

extern "C" int mi355_customized_fp_static(mi355_plan const *plan, void const *const *inputs,
                                          void *const *outputs) {
  MI355_REQUIRE_INIT();
  State &s = state();
  if (plan == nullptr || inputs == nullptr || outputs == nullptr) {
    return fail(MI355_ERR_INVALID, "null argument");
  }
  void *const base = g_static_scratch[s.device];
  if (base == nullptr) {
    return fail(MI355_ERR_NOT_INITIALISED, "static scratch of device %d was not set up", s.device);
  }
  DevProgram prog;
  PlanExtents ext;
  std::string err;
  int rc = compile_plan(*plan, false, s.max_lds, prog, ext, err);
  if (rc != MI355_OK) {
    return fail(rc, "%s", err.c_str());
  }
  for (int i = 0; i < plan->num_dmem_inputs; i++) {
    if (inputs[i] == nullptr) {
      return fail(MI355_ERR_INVALID, "input %d is null", i);
    }
    prog.in[i] = inputs[i];
  }
  for (int i = 0; i < plan->num_dmem_outputs; i++) {
    if (outputs[i] == nullptr) {
      return fail(MI355_ERR_INVALID, "output %d is null", i);
    }
    prog.out[i] = outputs[i];
  }
  for (int o = 0; o < prog.num_ops; o++) {
    DevOp &d = prog.ops[o];
    if (d.kind == DOP_LOAD && d.vec8 && (reinterpret_cast<uintptr_t>(prog.in[d.io]) & 15) != 0) {
      d.vec8 = 0;
    }
  }
  // The split rule of mi355_customized_fp (set_splits): as many ranges as it would take, fewer
  // while their partial sums do not fit the array (any split gives the same ring sum).  A
  // for-loop it would split but of which not even two ranges fit is refused rather than run
  // unsplit on a fraction of the device.
  prog.splits = 1;
  long long const blocks = (long long)prog.grid[0] * prog.grid[1] * prog.grid[2];
  int const F = prog.forloop_range;
  if (F >= 2 && blocks < 192) {
    int splits = (int)std::min<long long>(std::min(F, 64), (256 + blocks - 1) / blocks);
    long long elems = 0;
    for (int i = 0; i < plan->num_dmem_outputs; i++) {
      elems += (ext.out_elems[i] + 7) / 8 * 8;
    }
    while (splits > 2 && elems * splits * 2 > (long long)MI355_STATIC_SCRATCH_BYTES) {
      splits--;
    }
    if (splits >= 2 && elems * splits * 2 > (long long)MI355_STATIC_SCRATCH_BYTES) {
      return fail(MI355_ERR_UNSUPPORTED,
                  "plan needs %lld bytes of partial sums for two ranges of its for-loop; the static "
                  "scratch holds %d", elems * splits * 2, (int)MI355_STATIC_SCRATCH_BYTES);
    }
    if (splits >= 2) {
      prog.splits = splits;
      uint16_t *p = static_cast<uint16_t *>(base);
      for (int i = 0; i < plan->num_dmem_outputs; i++) {
        prog.part[i] = p;
        prog.part_elems[i] = ext.out_elems[i];
        prog.part_stride[i] = (ext.out_elems[i] + 7) / 8 * 8;
        p += prog.part_stride[i] * splits;
      }
    }
  }
  if ((long long)prog.grid[0] * prog.splits > 2147483647LL) {
    return fail(MI355_ERR_UNSUPPORTED, "grid too large");
  }
  dim3 grid(prog.grid[0] * prog.splits, prog.grid[1], prog.grid[2]);
  fp_interp_kernel<<<grid, kInterpThreads, prog.lds_bytes, s.stream()>>>(prog, s.exp_tbl, s.div_p,
                                                                        s.div_q);
  MI355_HIP(hipGetLastError());
  if (prog.splits > 1) {
    // every (range, block) workgroup overwrites its whole tile of the slab before this launch
    // reads it, so nothing needs clearing between calls
    if (int rc2 = fold_splits(prog)) {
      return rc2;
    }
  }
  s.last().kernel_id = MI355_KERNEL_FP_INTERP;
  s.last().workgroups = (int)(grid.x * grid.y * grid.z);
  s.last().threads = kInterpThreads;
  s.last().lds_bytes = prog.lds_bytes;
  s.last().row_split = prog.splits;
  return MI355_OK;
}

// The residue planes of one operand of a fused matmul plan: what identifies them (operand
// tensor, side, prologue, geometry) and where they are.
struct SplitOperand {
  void const *src;
  int which, unary, slabs, rows, cols;
  char *planes;
};

static SplitOperand const *find_split_operand(std::vector<SplitOperand> const &split, DevProgram const &P,
                                              int which) {
  DevOp const &op = P.ops[P.fg[which]];
  for (SplitOperand const &o : split) {
    if (o.src == P.in[op.io] && o.which == which && o.unary == P.fp_unary[which] &&
        o.slabs == P.pl_geo[3 * which] && o.rows == op.d_rows && o.cols == op.d_cols) {
      return &o;
    }
  }
  return nullptr;
}

// One chunk of a batch: every program in one multi-program launch per LDS class, then one
// launch that folds the partial sums of all split for-loops.  A program whose tiles leave
// no room in LDS for its own record is launched by itself.
static int launch_fp_chunk(std::vector<DevProgram> &progs, std::vector<PlanExtents> const &exts,
                           std::vector<int> const &num_outputs) {
  State &s = state();
  int const n = (int)progs.size();
  // fused matmul plans take the matrix cores while the residue planes of their operand
  // tensors fit what is left of this queue's plane memory
  // Members that multiply the same operand tensor (the candidates of one problem read one copy
  // of their common inputs) share its planes: the first one splits it, the others point at
  // the result.
  std::vector<SplitOperand> split;
  std::vector<DevProgram const *> on_matrix_cores;
  size_t planes_used = 0;
  for (int i = 0; i < n; i++) {
    size_t need = 0;
    if (progs[i].fused == 4 && fp_mfma_gemm_fits(progs[i], exts[i], &need)) {
      DevProgram &P = progs[i];
      size_t bytes[2];
      fp_mfma_plane_bytes(P, &bytes[0], &bytes[1]);
      char *place[2] = {nullptr, nullptr};
      int shared = 0;
      size_t fresh = 0;
      for (int which = 0; which < 2; which++) {
        if (SplitOperand const *o = find_split_operand(split, P, which)) {
          place[which] = o->planes;
          shared |= 1 << which;
        }
        if (place[which] == nullptr) {
          fresh += (bytes[which] + 255) / 256 * 256;
        }
      }
      if (planes_used + fresh <= s.planes_bytes) {
        for (int which = 0; which < 2; which++) {
          if (place[which] == nullptr) {
            DevOp const &op = P.ops[P.fg[which]];
            place[which] = s.planes() + planes_used;
            planes_used += (bytes[which] + 255) / 256 * 256;
            split.push_back(SplitOperand{P.in[op.io], which, P.fp_unary[which], P.pl_geo[3 * which],
                                         op.d_rows, op.d_cols, place[which]});
          }
        }
        fp_mfma_gemm_bind(P, place[0], place[1], shared, n >= 8 ? 16 : 256);
        on_matrix_cores.push_back(&progs[i]);
        continue;
      }
    }
    if (progs[i].fused == 4 && fp_needs_matrix_cores(progs[i])) {
      // (the caller cuts chunks so that the planes of their members fit together)
      return fail(MI355_ERR_UNSUPPORTED, "operand prologue without the matrix-core route");
    }
  }
  // split for-loops until the chunk as a whole offers the device a few workgroups per CU
  long long total = 0;
  for (DevProgram &p : progs) {
    p.splits = 1;
    total += fp_program_blocks(p);
  }
  int const scale = (int)std::min<long long>(64, (1024 + total - 1) / total);
  size_t used = 0;
  for (int i = 0; i < n; i++) {
    if (progs[i].fused != 5) {
      set_splits(progs[i], exts[i], num_outputs[i], std::min(progs[i].forloop_range, scale), used);
    }
  }
  int const record = (int)sizeof(DevProgram);
  // Launch classes.  Interpreter programs by LDS need (a launch requests the largest need of
  // its members, which bounds how many workgroups share a compute unit); fused matmul
  // programs by register tiles per thread (a template argument of their kernel), those on
  // the matrix cores in a class of their own, and the attention family in another.
  constexpr int kClasses = 8;
  int const bounds[3] = {24 * 1024, 64 * 1024, s.max_lds - record - 16};
  // (with fewer than three interpreter workgroups per compute unit in the whole chunk nobody's
  // occupancy is at stake, and one launch is a third of the latency of three in a row)
  long long interp_blocks = 0;
  for (DevProgram const &p : progs) {
    if (p.fused == 0 && p.lds_bytes <= bounds[2]) {
      interp_blocks += (long long)p.grid[0] * p.splits * p.grid[1] * p.grid[2];
    }
  }
  bool const one_interp_class = interp_blocks <= 768;
  auto class_of = [&](DevProgram const &p) {
    if (p.fused == 4) {
      return p.fg[5] ? 6 : (p.fg[3] == 1 ? 3 : (p.fg[3] == 2 ? 4 : 5));
    }
    if (p.fused == 5) {
      return 7;
    }
    for (int c = 0; c < 3; c++) {
      if (p.lds_bytes <= bounds[c]) {
        return one_interp_class ? 2 : c;
      }
    }
    return -1;  // no room for the record above its tiles: launched by itself
  };
  std::vector<int> order;
  int class_begin[kClasses + 1] = {};
  for (int c = 0; c < kClasses; c++) {
    for (int i = 0; i < n; i++) {
      if (class_of(progs[i]) == c) {
        order.push_back(i);
      }
    }
    class_begin[c + 1] = (int)order.size();
  }
  int const members = (int)order.size();
  std::vector<CombineJob> jobs;
  std::vector<int> job_first(1, 0);
  for (int i : order) {
    DevProgram const &p = progs[i];
    if (p.splits < 2) {
      continue;
    }
    for (int o = 0; o < MI355_MAX_DMEM_OUTPUTS; o++) {
      if (p.out[o] == nullptr || p.part_elems[o] <= 0) {
        continue;
      }
      CombineJob j;
      j.part = p.part[o];
      j.out = static_cast<uint16_t *>(p.out[o]);
      j.n = p.part_elems[o];
      j.stride_elems = p.part_stride[o];
      j.splits = p.splits;
      j.pad = 0;
      jobs.push_back(j);
      job_first.push_back(job_first.back() + (int)std::min<long long>((j.n + 255) / 256, 256));
    }
  }
  int launched = 0;
  if (members > 0) {
    // staging layout: programs | first_block per class (members + kClasses ints) | jobs | job_first
    size_t const off_first = sizeof(DevProgram) * (size_t)members;
    size_t const off_jobs = (off_first + sizeof(int) * (size_t)(members + kClasses) + 15) / 16 * 16;
    size_t const off_jfirst = off_jobs + sizeof(CombineJob) * jobs.size();
    size_t const bytes = (off_jfirst + sizeof(int) * job_first.size() + 15) / 16 * 16;
    if (bytes > State::kBatchSlotBytes) {
      return fail(MI355_ERR_UNSUPPORTED, "batch chunk does not fit its staging buffer");
    }
    State::BatchSlot &slot = s.batch[tls_queue][s.batch_next[tls_queue]];
    s.batch_next[tls_queue] = (s.batch_next[tls_queue] + 1) % State::kBatchSlots;
    MI355_HIP(hipEventSynchronize(slot.copied));  // the copy that last read this buffer is done
    DevProgram *hp = reinterpret_cast<DevProgram *>(slot.host);
    int *hf = reinterpret_cast<int *>(slot.host + off_first);
    int fpos = 0;
    int first_off[kClasses], first_cnt[kClasses];
    for (int c = 0; c < kClasses; c++) {
      first_off[c] = fpos;
      first_cnt[c] = class_begin[c + 1] - class_begin[c];
      int acc = 0;
      for (int k = class_begin[c]; k < class_begin[c + 1]; k++) {
        DevProgram const &p = progs[order[k]];
        hp[k] = p;
        hf[fpos++] = acc;
        acc += (int)fp_program_blocks(p);
      }
      hf[fpos++] = acc;  // total of the class
    }
    if (!jobs.empty()) {
      memcpy(slot.host + off_jobs, jobs.data(), sizeof(CombineJob) * jobs.size());
      memcpy(slot.host + off_jfirst, job_first.data(), sizeof(int) * job_first.size());
    }
    // the records travel by a copy kernel that reads the pinned buffer over the bus: a
    // stream-ordered hipMemcpyAsync of this size costs the host ~100 us per call here
    stage_records_kernel<<<(int)((bytes / 16 + 255) / 256), 256, 0, s.stream()>>>(
        reinterpret_cast<uint4v const *>(slot.host), reinterpret_cast<uint4v *>(slot.dev),
        (int)(bytes / 16));
    MI355_HIP(hipEventRecord(slot.copied, s.stream()));
    if (!on_matrix_cores.empty()) {
      if (int rc = fp_mfma_split_programs(on_matrix_cores.data(), (int)on_matrix_cores.size(), s.stream())) {
        return rc;
      }
    }
    static std::atomic<bool> lds_raised{false};
    DevProgram const *dp = reinterpret_cast<DevProgram const *>(slot.dev);
    int const *df = reinterpret_cast<int const *>(slot.dev + off_first);
    for (int c = 0; c < kClasses; c++) {
      if (first_cnt[c] == 0) {
        continue;
      }
      int lds = 0;
      for (int k = class_begin[c]; k < class_begin[c + 1]; k++) {
        lds = std::max(lds, progs[order[k]].lds_bytes);
      }
      if (c == 7) {
        int const blocks = hf[first_off[c] + first_cnt[c]];
        if (int rc = launch_fp_attn_multi(dp + class_begin[c], df + first_off[c], first_cnt[c], blocks, lds, s.stream())) {
          return rc;
        }
        launched += blocks;
        continue;
      }
      if (c == 6) {
        int const blocks = hf[first_off[c] + first_cnt[c]];
        if (int rc = launch_fp_mfma_gemm_multi(dp + class_begin[c], df + first_off[c], first_cnt[c], blocks,
                                               s.stream())) {
          return rc;
        }
        launched += blocks;
        continue;
      }
      if (c >= 3) {
        int const blocks = hf[first_off[c] + first_cnt[c]];
        if (int rc = launch_fp_gemm_multi(dp + class_begin[c], df + first_off[c], first_cnt[c], blocks,
                                          c == 3 ? 1 : (c == 4 ? 2 : 4), lds, s.stream())) {
          return rc;
        }
        launched += blocks;
        continue;
      }
      int const program_off = (lds + 15) / 16 * 16;
      int const lds_total = program_off + record;
      if (lds_total > 65536 && !lds_raised) {
        MI355_HIP(hipFuncSetAttribute(reinterpret_cast<void const *>(fp_interp_multi_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, s.max_lds));
        lds_raised = true;
      }
      int const blocks = hf[first_off[c] + first_cnt[c]];
      fp_interp_multi_kernel<<<blocks, kInterpThreads, lds_total, s.stream()>>>(
          dp + class_begin[c], df + first_off[c], first_cnt[c], program_off, s.exp_tbl, s.div_p,
          s.div_q);
      launched += blocks;
    }
    if (!jobs.empty()) {
      fp_combine_splits_multi_kernel<<<job_first.back(), 256, 0, s.stream()>>>(
          reinterpret_cast<CombineJob const *>(slot.dev + off_jobs),
          reinterpret_cast<int const *>(slot.dev + off_jfirst), (int)jobs.size());
    }
    MI355_HIP(hipGetLastError());
  }
  // programs too large to share LDS with their own record: one launch each (launch() also
  // folds their split for-loops)
  for (int i = 0; i < n; i++) {
    if (class_of(progs[i]) < 0) {
      int rc = launch(progs[i], false);
      if (rc != MI355_OK) {
        return rc;
      }
      launched += s.last().workgroups;
    }
  }
  s.last().kernel_id = MI355_KERNEL_FP_INTERP;
  s.last().workgroups = launched;
  s.last().threads = kInterpThreads;
  s.last().lds_bytes = 0;
  s.last().row_split = 1;
  return MI355_OK;
}

extern "C" int mi355_customized_fp_batch(mi355_plan const *plans, int n,
                                         void const *const *inputs, void *const *outputs) {
  return mi355_customized_fp_batch_within(plans, n, inputs, outputs, nullptr, nullptr);
}

extern "C" int mi355_customized_fp_batch_within(mi355_plan const *plans, int n, void const *const *inputs,
                                                void *const *outputs, long long const *in_elems,
                                                long long const *out_elems) {
  MI355_REQUIRE_INIT();
  if (n < 0 || (n > 0 && (plans == nullptr || inputs == nullptr || outputs == nullptr))) {
    return fail(MI355_ERR_INVALID, "bad batch (n = %d)", n);
  }
  // independent operators: a handful of launches for all of them, on the caller's queue.  A
  // chunk ends after 64 operators, or where the residue planes of its fused matmul plans
  // would no longer fit this queue's plane memory together.
  int const chunk_max = 64;
  std::vector<DevProgram> progs;
  std::vector<PlanExtents> exts;
  std::vector<int> nout;
  size_t planes_wanted = 0;
  std::vector<SplitOperand> wanted;  // operands whose planes the chunk already counts
  auto flush = [&]() {
    int rc = progs.empty() ? MI355_OK : launch_fp_chunk(progs, exts, nout);
    progs.clear();
    exts.clear();
    nout.clear();
    planes_wanted = 0;
    wanted.clear();
    return rc;
  };
  for (int i = 0; i < n; i++) {
    DevProgram prog;
    PlanExtents ext;
    int rc = prepare(&plans[i], inputs + (size_t)i * MI355_MAX_DMEM_INPUTS,
                     outputs + (size_t)i * MI355_MAX_DMEM_OUTPUTS, false, prog, &ext);
    if (rc != MI355_OK) {
      return rc;
    }
    for (int j = 0; in_elems != nullptr && j < plans[i].num_dmem_inputs; j++) {
      if (ext.in_elems[j] > in_elems[(size_t)i * MI355_MAX_DMEM_INPUTS + j]) {
        return fail(MI355_ERR_INVALID, "operator %d: input loader would read past its tensor", i);
      }
    }
    for (int j = 0; out_elems != nullptr && j < plans[i].num_dmem_outputs; j++) {
      if (ext.out_elems[j] > out_elems[(size_t)i * MI355_MAX_DMEM_OUTPUTS + j]) {
        return fail(MI355_ERR_INVALID, "operator %d: output saver would write past its tensor", i);
      }
    }
    size_t need = 0;
    if (prog.fused == 4 && fp_mfma_gemm_fits(prog, ext, &need)) {
      size_t bytes[2];
      fp_mfma_plane_bytes(prog, &bytes[0], &bytes[1]);
      auto fresh = [&]() {
        size_t f = 0;
        for (int which = 0; which < 2; which++) {
          if (find_split_operand(wanted, prog, which) == nullptr) {
            f += (bytes[which] + 255) / 256 * 256;
          }
        }
        return f;
      };
      if (planes_wanted + fresh() > state().planes_bytes) {
        if (int rc2 = flush()) {
          return rc2;
        }
      }
      planes_wanted += fresh();
      for (int which = 0; which < 2; which++) {
        if (find_split_operand(wanted, prog, which) == nullptr) {
          DevOp const &op = prog.ops[prog.fg[which]];
          wanted.push_back(SplitOperand{prog.in[op.io], which, prog.fp_unary[which], prog.pl_geo[3 * which],
                                        op.d_rows, op.d_cols, nullptr});
        }
      }
    }
    progs.push_back(prog);
    exts.push_back(ext);
    nout.push_back(plans[i].num_dmem_outputs);
    if ((int)progs.size() == chunk_max) {
      if (int rc2 = flush()) {
        return rc2;
      }
    }
  }
  return flush();
}

extern "C" int mi355_customized_run(mi355_plan const *plan, void const *const *inputs,
                                    void *const *outputs) {
  MI355_REQUIRE_INIT();
  return run_plan(plan, inputs, outputs, true);
}

// ---- prepared operators ------------------------------------------------------------------------
// The kernel launches of one customized operator, or of two that follow each other, recorded once and
// repeated: see launch.h.  They hold for the queue (its scratch memory is in the arguments) and the options
// they were recorded under; a run from another queue or after mi355_set_option records them again.
struct PreparedPlan {
  mi355_plan plan;
  void const *inputs[MI355_MAX_DMEM_INPUTS];
  void *outputs[MI355_MAX_DMEM_OUTPUTS];
};
struct mi355_prepared {
  PreparedPlan op[2];
  int ops;
  bool fp16;
  int queue;
  unsigned generation;
  LaunchList list;
  mi355_launch_info info;
  int *tickets = nullptr;  // of `queue`
  int num_tickets = 0;
  unsigned tickets_life = 0;
  void drop_tickets() {
    if (tickets != nullptr) {
      give_tickets(queue, tickets, num_tickets, tickets_life);
      tickets = nullptr;
    }
  }
  ~mi355_prepared() { drop_tickets(); }
};

// Two fp16 operators that share work: 1 recorded, 0 not such a pair, < 0 an error.
static int record_pair(mi355_prepared &p, DevProgram const &first, DevProgram const &second) {
  FoldRequest fold;
  if (first.fused == 1 && second.fused == 3 && combine_as_rows(second, fold.rows)) {
    fold.tickets = [&](int count) {
      p.drop_tickets();
      p.tickets = take_tickets(p.queue, count, p.tickets_life);
      p.num_tickets = count;
      return p.tickets;
    };
    return try_launch_attention(first, &fold);
  }
  GateRequest gate;
  if (first.fused == 2 && second.fused == 2 && gate_pair(first, second, gate)) {
    // (in the queue's memory for operand copies: work of one queue is ordered)
    if (state().planes() == nullptr || gate.elements * 2 > state().planes_bytes) {
      return 0;
    }
    gate.h = state().planes();
    int rc = try_launch_gemm(first, &gate, false);
    rc = rc == 1 ? try_launch_gemm(second, &gate, true) : rc;
    if (rc == 0) {
      p.list.launches.clear();  // (what one of them recorded is not repeated)
    }
    return rc;
  }
  return 0;
}

static int record_prepared(mi355_prepared &p) {
  p.list.launches.clear();
  p.drop_tickets();
  p.queue = tls_queue;
  p.generation = options_generation();
  launch_recorder() = &p.list;
  // (what a pair's plans are compiled to serves the two operators as well where they share nothing: the host's part of a
  // split-KV decode's first pass 7.7 us, with both compiled again 8.6)
  DevProgram prog[2];
  int rc = MI355_OK;
  for (int i = 0; i < p.ops && rc == MI355_OK; i++) {
    rc = prepare(&p.op[i].plan, p.op[i].inputs, p.op[i].outputs, p.fp16, prog[i]);
  }
  int const pair = rc == MI355_OK && p.ops == 2 && p.fp16 ? record_pair(p, prog[0], prog[1]) : 0;
  if (pair < 0) {
    rc = pair;
  } else if (pair == 0) {
    p.drop_tickets();
    for (int i = 0; i < p.ops && rc == MI355_OK; i++) {
      rc = launch_plan(&p.op[i].plan, p.op[i].inputs, p.op[i].outputs, p.fp16, prog[i]);
    }
  }
  launch_recorder() = nullptr;
  p.info = state().last();
  if (rc != MI355_OK) {
    p.generation = 0;  // (nothing to repeat: recorded again on the next run)
  }
  return rc;
}

static int prepare_operators(mi355_plan const *const *plans, void const *const *const *inputs, void *const *const *outputs, int ops,
                             int fingerprint, mi355_prepared **prepared) {
  if (prepared == nullptr) {
    return fail(MI355_ERR_INVALID, "bad argument");
  }
  std::unique_ptr<mi355_prepared> p(new mi355_prepared{});
  p->ops = ops;
  p->fp16 = fingerprint == 0;
  for (int i = 0; i < ops; i++) {
    if (plans[i] == nullptr || inputs[i] == nullptr || outputs[i] == nullptr || plans[i]->num_dmem_inputs > MI355_MAX_DMEM_INPUTS ||
        plans[i]->num_dmem_outputs > MI355_MAX_DMEM_OUTPUTS) {
      return fail(MI355_ERR_INVALID, "bad argument");
    }
    p->op[i].plan = *plans[i];
    std::copy(inputs[i], inputs[i] + plans[i]->num_dmem_inputs, p->op[i].inputs);
    std::copy(outputs[i], outputs[i] + plans[i]->num_dmem_outputs, p->op[i].outputs);
  }
  if (int rc = record_prepared(*p)) {
    return rc;
  }
  *prepared = p.release();
  return MI355_OK;
}

extern "C" int mi355_prepare(mi355_plan const *plan, void const *const *inputs, void *const *outputs, int fingerprint,
                             mi355_prepared **prepared) {
  MI355_REQUIRE_INIT();
  return prepare_operators(&plan, &inputs, &outputs, 1, fingerprint, prepared);
}

extern "C" int mi355_prepare_two(mi355_plan const *first, void const *const *first_inputs, void *const *first_outputs,
                                 mi355_plan const *second, void const *const *second_inputs, void *const *second_outputs,
                                 int fingerprint, mi355_prepared **prepared) {
  MI355_REQUIRE_INIT();
  mi355_plan const *const plans[] = {first, second};
  void const *const *const inputs[] = {first_inputs, second_inputs};
  void *const *const outputs[] = {first_outputs, second_outputs};
  return prepare_operators(plans, inputs, outputs, 2, fingerprint, prepared);
}

extern "C" int mi355_prepared_run(mi355_prepared *prepared) {
  MI355_REQUIRE_INIT();
  if (prepared == nullptr) {
    return fail(MI355_ERR_INVALID, "null argument");
  }
  mi355_prepared &p = *prepared;
  if (p.queue != tls_queue || p.generation != options_generation()) {
    if (int rc = record_prepared(p)) {
      return rc;
    }
  }
  State &s = state();
  hipStream_t const q = s.stream();
  for (RecordedLaunch &l : p.list.launches) {
    MI355_HIP(hipLaunchKernel(l.fn, l.grid, l.block, l.args.data(), l.lds, q));
  }
  s.last() = p.info;
  return MI355_OK;
}

extern "C" int mi355_prepared_free(mi355_prepared *prepared) {
  delete prepared;
  return MI355_OK;
}

namespace mi355 {
namespace {
// A timed loop's launches: those of one call (see launch.h), and for long loops `kRepeats` calls'
// worth of them as one chain of kernel nodes -- one graph launch enqueues them all, for a
// fraction of the host time of as many kernel launches.
struct LaunchReplay {
  LaunchList list;
  static constexpr int kRepeats = 256;
  hipGraph_t chain = nullptr;
  hipGraphExec_t chain_exec = nullptr;
  bool chain_tried = false;
  ~LaunchReplay() {
    if (chain_exec != nullptr) {
      (void)hipGraphExecDestroy(chain_exec);
    }
    if (chain != nullptr) {
      (void)hipGraphDestroy(chain);
    }
  }
  // false (and no chain) when the runtime refuses any step: the caller launches kernel by kernel
  bool build_chain() {
    if (chain_tried) {
      return chain_exec != nullptr;
    }
    chain_tried = true;
    if (list.launches.empty() || hipGraphCreate(&chain, 0) != hipSuccess) {
      return false;
    }
    hipGraphNode_t prev = nullptr;
    for (int r = 0; r < kRepeats; r++) {
      for (RecordedLaunch &l : list.launches) {
        hipKernelNodeParams k{};
        k.func = const_cast<void *>(l.fn);
        k.gridDim = l.grid;
        k.blockDim = l.block;
        k.sharedMemBytes = l.lds;
        k.kernelParams = l.args.data();
        hipGraphNode_t node = nullptr;
        if (hipGraphAddKernelNode(&node, chain, prev == nullptr ? nullptr : &prev, prev == nullptr ? 0 : 1, &k) !=
            hipSuccess) {
          (void)hipGetLastError();
          return false;
        }
        prev = node;
      }
    }
    if (hipGraphInstantiate(&chain_exec, chain, nullptr, nullptr, 0) != hipSuccess) {
      (void)hipGetLastError();
      chain_exec = nullptr;
      return false;
    }
    return true;
  }
};

// The last call each queue profiled, kept with its launches: a caller that warms up in one call and
// times in the next (same plan, same tensors) pays for the chain once, outside its timed call.
struct KeptReplay {
  bool fp16 = false;
  unsigned generation = 0;
  DevProgram prog;
  std::unique_ptr<LaunchReplay> replay;
};
KeptReplay g_kept[MI355_NUM_QUEUES];
// what is kept from before the last drop is not used again (a queue's slot is touched only by
// the host thread that drives the queue, so a drop from another thread just moves this on)
std::atomic<unsigned> g_kept_generation{1};
}  // namespace

// (options change which kernels a plan runs on: what was recorded under the old ones is dropped)
void drop_profile_replays() { g_kept_generation.fetch_add(1, std::memory_order_relaxed); }
unsigned options_generation() { return g_kept_generation.load(std::memory_order_relaxed); }
}  // namespace mi355

extern "C" int mi355_customized_profile(mi355_plan const *plan, void const *const *inputs,
                                        void *const *outputs, int fingerprint, int warmup,
                                        int iters, float *ms) {
  MI355_REQUIRE_INIT();
  if (iters < 1 || warmup < 0 || ms == nullptr) {
    return fail(MI355_ERR_INVALID, "bad iteration counts");
  }
  DevProgram prog;
  int rc = prepare(plan, inputs, outputs, fingerprint == 0, prog);
  if (rc != MI355_OK) {
    return rc;
  }
  State &s = state();
  // What a call launches is recorded once and repeated from there (kernel by kernel, or, for
  // loops of 512 launches and more, 256 calls at a time as one chain of kernel nodes), so that
  // the loop times the device and not plan matching, parameter set-up and launch calls on the
  // host.  The loop is also paced: a marker after every batch of 1024, and the host waits for
  // the batch before the one it has just enqueued, which leaves between one and two batches
  // in flight and the device never idle (a queue several thousand launches deep runs each of
  // them slower).
  constexpr int kPaceBatch = 1024;
  long long enqueued = 0;
  KeptReplay &kept = g_kept[tls_queue];
  static_assert(std::is_trivially_copyable<DevProgram>::value, "compared and kept as bytes");
  unsigned const generation = g_kept_generation.load(std::memory_order_relaxed);
  if (kept.replay == nullptr || kept.generation != generation || kept.fp16 != (fingerprint == 0) ||
      std::memcmp(&kept.prog, &prog, sizeof(prog)) != 0) {
    kept.replay.reset(new LaunchReplay);
    kept.generation = generation;
    std::memcpy(&kept.prog, &prog, sizeof(prog));
    kept.fp16 = fingerprint == 0;
    launch_recorder() = &kept.replay->list;
    rc = launch(prog, fingerprint == 0);
    if (rc == kDeclined) {
      kept.replay->list.launches.clear();
      if ((rc = prepare(plan, inputs, outputs, fingerprint == 0, prog, nullptr, true)) == MI355_OK) {
        rc = launch(prog, fingerprint == 0);
      }
    }
    launch_recorder() = nullptr;
    if (rc != MI355_OK) {
      kept.replay.reset();
      return rc;
    }
  }
  LaunchReplay &replay = *kept.replay;
  auto launch_once = [&]() -> int {
    for (RecordedLaunch &l : replay.list.launches) {
      MI355_HIP(hipLaunchKernel(l.fn, l.grid, l.block, l.args.data(), l.lds, s.stream()));
    }
    return MI355_OK;
  };
  static_assert(kPaceBatch % LaunchReplay::kRepeats == 0, "a batch is a whole number of chains");
  bool const chained = warmup + iters >= 2 * LaunchReplay::kRepeats && replay.build_chain();
  auto launch_paced = [&](int count) -> int {
    int i = 0;
    while (i < count) {
      int done = 1;
      if (chained && count - i >= LaunchReplay::kRepeats && enqueued % LaunchReplay::kRepeats == 0) {
        MI355_HIP(hipGraphLaunch(replay.chain_exec, s.stream()));
        done = LaunchReplay::kRepeats;
      } else {
        int const r = launch_once();
        if (r != MI355_OK) {
          return r;
        }
      }
      i += done;
      enqueued += done;
      if (enqueued % kPaceBatch == 0) {
        long long const batch = enqueued / kPaceBatch;
        MI355_HIP(hipEventRecord(s.pace[tls_queue][batch & 1], s.stream()));
        if (batch > 1) {
          MI355_HIP(hipEventSynchronize(s.pace[tls_queue][(batch - 1) & 1]));
        }
      }
    }
    return MI355_OK;
  };
  if ((rc = launch_paced(warmup)) != MI355_OK) {
    return rc;
  }
  MI355_HIP(hipEventRecord(s.ev0[tls_queue], s.stream()));
  if ((rc = launch_paced(iters)) != MI355_OK) {
    return rc;
  }
  MI355_HIP(hipEventRecord(s.ev1[tls_queue], s.stream()));
  MI355_HIP(hipEventSynchronize(s.ev1[tls_queue]));
  float total = 0.0f;
  MI355_HIP(hipEventElapsedTime(&total, s.ev0[tls_queue], s.ev1[tls_queue]));
  *ms = total / iters;
  return MI355_OK;
}
