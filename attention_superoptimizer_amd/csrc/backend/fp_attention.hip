// Fingerprints of the un-fused attention graph in one launch: S = Q . K, E = exp(S), R = the sums of E's rows,
// P = E / R and O = P . V, all of them written.
//
// The ring is Z_227 x Z_113, and an exponential has residue 0 modulo 113 and depends on its argument modulo
// 113 alone: after the scores everything is one residue.  The division is a factor common to a row, so O is
// the row of E . V times it, and needs the row's sum only at its end.
//
// A workgroup owns 16 RG rows of one matrix, KW wavefronts to 16 rows, each with every KW-th chunk of 64 keys.  A chunk of K and V goes from memory (the next chunk is in
// flight while this one is multiplied) through registers, where 4 x 4 patches are reduced to bytes and turned,
// into LDS as MFMA operands; K^T is the first operand, so a lane ends up with 16 consecutive scores of one row,
// looks their exponentials up and has the second product's operand.  S and E leave through a strip of the
// wavefront's own: stored as they are, sixteen lanes in a row would write sixteen rows, which a compute unit's
// vector cache takes at a quarter of its rate.  Once the row sums are there, each wavefront reads back the E it
// stored and writes P.
//
// What bounds it: the vector instructions that reduce K and V to residues again in every workgroup, recombine
// and look up.  As a product, the row kernel and a product [32, 256, 64] . [32, 64, 1024] took 12.3, 10.9 and 13.3
// us; 24.5 here.
#include "common.h"

#include <algorithm>

namespace mi355 {

namespace {

constexpr int kChunk = 64;                    // keys
constexpr int kPitch = 80, kPlane = 64 * kPitch;  // bytes of an LDS row of 64 residues, of a plane of 64 of them
constexpr int kStripPitch = 144, kStrip = 16 * kStripPitch;  // 16 rows of 64 values
constexpr int kExpBelow = 56;                 // table entries below 0 (see the lookup)
constexpr int kInverseAt = 704, kSumsAt = 944, kStripsAt = 1456;
constexpr int rows_lds(int waves, int kw) { return kStripsAt + waves * kStrip + kw * 3 * kPlane; }
typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

struct FpRows {
  uint16_t const *q, *k, *v;
  uint16_t *s, *e, *r, *p, *o;
  int m, n, d, dv, slices;
  unsigned total;
};

template <int RG, int KW>
__global__ __launch_bounds__(64 * RG * KW) void fp_attention_rows_kernel(FpRows const A, FpTables const t) {
  constexpr int W = RG * KW, ROWS = 16 * RG, PATCHES = 4 / RG, SETS = W / 4;  // patches a thread stages; of 256 threads
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int const tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), g = lane / 16, c = lane % 16;
  int const kw = wave % KW, rg = wave / KW;
  uint32_t *const exps = reinterpret_cast<uint32_t *>(lds) + kExpBelow;  // [-56, 113): residue as a signed byte | the value << 16
  uint8_t *const inverse = lds + kInverseAt;                             // [227]
  int *const sums = reinterpret_cast<int *>(lds + kSumsAt);              // [KW][ROWS], then the rows' factors [ROWS]
  unsigned char *const strip = lds + kStripsAt + wave * kStrip;
  unsigned char *const tiles = lds + kStripsAt + W * kStrip;             // [KW][K mod 113, V mod 227, K mod 227][64][kPitch]
  if (tid < (int)FP_Q + kExpBelow) {
    int const x = tid - kExpBelow;
    uint32_t const p = t.exp_tbl[x < 0 ? x + (int)FP_Q : x];
    exps[x] = ((uint32_t)residue_p_signed(p) & 0xffu) | (fp_from_residues(p, 0u) << 16);
  }
  if (tid < (int)FP_P) {
    inverse[tid] = static_cast<uint8_t>(t.div_p[tid]);
  }
  // an XCD (one L2) gets consecutive workgroups: they share keys and values
  unsigned const xcd = blockIdx.x % 8, each = A.total / 8, more = A.total % 8;
  unsigned const w = xcd * each + (xcd < more ? xcd : more) + blockIdx.x / 8;
  int const b = (int)(w / (unsigned)A.slices), row0 = (int)(w % (unsigned)A.slices) * ROWS + 16 * rg;
  int const m = A.m, n = A.n, d = A.d, dv = A.dv, row = row0 + c;
  uint16_t const *const K = A.k + (size_t)b * d * n, *const V = A.v + (size_t)b * n * dv;

  // ---- query residues: row c, elements 16 g .. + 15
  v4i qf, qp;
  {
    uint16_t const *const q = A.q + ((size_t)b * m + (row < m ? row : m - 1)) * d;
    uint2 x[1][4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      int const at = 16 * g + 4 * u;
      x[0][u] = uint2{0, 0};
      if (at < d) {
        x[0][u] = *reinterpret_cast<uint2 const *>(q + at);
      }
    }
    if (fp_past_residues(fp_bits(x))) {
      fp_into_ring(x);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      uint32_t rp, rq;
      residues_row(x[0][u], rp, rq);
      qf[u] = (int)rq;
      qp[u] = (int)rp;
    }
  }

  // ---- staging: patch (hi, lo) of a chunk of K is 4 elements from 4 hi of 4 keys from 4 lo; of V, 4 elements
  // from 4 lo of the keys 16 (hi / 4) + 4 i + hi % 4.  Column 4 lo + u becomes row lo of matrix tile u, so a
  // lane's scores are those of keys 16 g + 4 r + j, the order V's keys then have.
  // (past the end the last patch stands in: elements of K past d meet zeros of Q, keys past n are masked,
  // elements of V past dv are not stored)
  int const set = tid / 256, hi = tid % 256 / 16, lo = tid % 16;
  uint2 kr[PATCHES][4], vr[PATCHES][4];
  auto fetch = [&](int group) {
#pragma unroll
    for (int u = 0; u < PATCHES; u++) {
      int const key0 = (group * KW + u * SETS + set) * kChunk;
      int const kk = min(4 * hi, d - 4), kc = min(key0 + 4 * lo, n - 4), vc = min(4 * lo, dv - 4);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        kr[u][i] = *reinterpret_cast<uint2 const *>(K + (size_t)(kk + i) * n + kc);
        vr[u][i] = *reinterpret_cast<uint2 const *>(V + (size_t)min(key0 + 16 * (hi / 4) + 4 * i + hi % 4, n - 1) * dv + vc);
      }
    }
  };
  auto put = [&]() {
#pragma unroll
    for (int u = 0; u < PATCHES; u++) {
      unsigned char *const kq = tiles + (u * SETS + set) * 3 * kPlane, *const vp = kq + kPlane, *const kp = vp + kPlane;
      uint32_t p[4], q[4], v[4], unused[4];
      residues_patch(kr[u], p, q);
      residues_patch(vr[u], v, unused);
#pragma unroll
      for (int x = 0; x < 4; x++) {
        int const at = (16 * x + lo) * kPitch + 4 * hi;
        *reinterpret_cast<uint32_t *>(kq + at) = q[x];
        *reinterpret_cast<uint32_t *>(kp + at) = p[x];
        *reinterpret_cast<uint32_t *>(vp + at) = v[x];
      }
    }
  };
  auto stage = [&]() {
    put();
    if (fp_past_residues(fp_bits(kr) | fp_bits(vr))) {  // (looked at last: the first values are not kept waiting)
      fp_into_ring(kr);
      fp_into_ring(vr);
      put();
    }
  };
  // 16 consecutive values of row c in every lane, two to a word, out as rows: lane l stores chunk l % 8 of rows
  // l / 8 and 8 + l / 8
  int const l8 = lane / 8, ch8 = lane % 8;
  auto send = [&](uint32_t const (&x)[8], uint16_t *to, int key0) {
    *reinterpret_cast<uint4v *>(strip + c * kStripPitch + 32 * g) = uint4v{x[0], x[1], x[2], x[3]};
    *reinterpret_cast<uint4v *>(strip + c * kStripPitch + 32 * g + 16) = uint4v{x[4], x[5], x[6], x[7]};
    asm volatile("" ::: "memory");  // (a wavefront's LDS operations complete in order)
#pragma unroll
    for (int i = 0; i < 2; i++) {
      int const r = row0 + 8 * i + l8;
      uint4v const v = *reinterpret_cast<uint4v const *>(strip + (8 * i + l8) * kStripPitch + 16 * ch8);
      if (r < m && key0 + 8 * ch8 < n) {
        *reinterpret_cast<uint4v *>(to + ((size_t)b * m + r) * n + key0 + 8 * ch8) = v;
      }
    }
    asm volatile("" ::: "memory");
  };

  // a barrier for what is in LDS: the one of the language also waits for every value stored so far to have arrived
  auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  v4i o[4];
  int rs = 0;
#pragma unroll
  for (int x = 0; x < 4; x++) {
    o[x] = v4i{0, 0, 0, 0};
  }
  v4i const base_p = {kSumBaseFewP, kSumBaseFewP, kSumBaseFewP, kSumBaseFewP};
  v4i const base_q = {kSumBaseFewQ, kSumBaseFewQ, kSumBaseFewQ, kSumBaseFewQ};
  int const chunks = (n + kChunk - 1) / kChunk, groups = (chunks + KW - 1) / KW;
  fetch(0);
  for (int group = 0; group < groups; group++) {
    meet();
    stage();
    meet();
    if (group + 1 < groups) {
      fetch(group + 1);
    }
    int const key0 = (group * KW + kw) * kChunk;
    if (key0 < n) {
      unsigned char const *const kq = tiles + kw * 3 * kPlane, *const vp = kq + kPlane, *const kp = vp + kPlane;
      // keys past n (exp(0) is not zero): the first `inside` bytes of every e[j] count
      int const inside = (n - key0 - 16 * g) / 4;
      uint32_t const mask = inside >= 4 ? ~0u : inside <= 0 ? 0u : (1u << (8 * inside)) - 1;
      v4i e;
      uint32_t s16[8], e16[8];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        v4i const x = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<v4i const *>(kq + (16 * j + c) * kPitch + 16 * g), qf,
                                                            base_q, 0, 0, 0);
        v4i const y = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<v4i const *>(kp + (16 * j + c) * kPitch + 16 * g), qp,
                                                            base_p, 0, 0, 0);
        // A score is within 64 * 66^2 of the base: in (0, 2^20).  2320 = ceil(2^18 / 113) gives its quotient or
        // one more: the remainder is in [-51, 95], and the table starts below zero.
        uint32_t b4[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          uint32_t const z = fp_from_based_sums<true>((uint32_t)y[r], (uint32_t)x[r]);
          b4[r] = exps[(int)mad24((uint32_t)__umul24((uint32_t)x[r], 2320u) >> 18, -(int)FP_Q, (uint32_t)x[r])];
          // key 4 r + j of the lane's sixteen
          uint32_t const value = b4[r] >> 16;
          s16[2 * r + j / 2] = j % 2 == 0 ? z : s16[2 * r + j / 2] | (z << 16);
          e16[2 * r + j / 2] = j % 2 == 0 ? value : e16[2 * r + j / 2] | (value << 16);
        }
        e[j] = (int)(pack_bytes(b4[0], b4[1], b4[2], b4[3]) & mask);
        rs = __builtin_amdgcn_sdot4(e[j], 0x01010101, rs, false);
      }
      send(s16, A.s, key0);
      send(e16, A.e, key0);
#pragma unroll
      for (int x = 0; x < 4; x++) {
        o[x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<v4i const *>(vp + (16 * x + c) * kPitch + 16 * g), e, o[x], 0, 0, 0);
      }
    }
  }
  // ---- the rows' sums over all their keys, and their inverses
  rs = (int)reduce_p(rs);
  rs += __shfl_xor(rs, 16, 64);
  rs += __shfl_xor(rs, 32, 64);
  uint32_t y = reduce_p(rs);
  if (KW > 1) {
    if (g == 0) {
      sums[kw * ROWS + 16 * rg + c] = (int)y;
    }
    meet();
    int all = 0;
#pragma unroll
    for (int u = 0; u < KW; u++) {
      all += sums[u * ROWS + 16 * rg + c];
    }
    y = reduce_p(all);
  }
  uint32_t const inv = inverse[y];
  meet();  // (every wavefront has the sums, and is done with the tiles)
  if (kw == 0 && g == 0) {
    sums[16 * rg + c] = (int)inv;
    if (row < m) {
      A.r[(size_t)b * m + row] = static_cast<uint16_t>(fp_from_residues(y, 0u));
    }
  }
  // ---- O, the wavefronts' keys together
  int *const part = reinterpret_cast<int *>(tiles);  // [KW - 1][RG][16][64]
  if (KW > 1 && kw > 0) {
#pragma unroll
    for (int x = 0; x < 16; x++) {
      part[(((kw - 1) * RG + rg) * 16 + x) * 64 + lane] = (int)reduce_p(o[x / 4][x % 4]);
    }
  }
  meet();
  if (kw == 0 && row < m) {
    uint16_t *const og = A.o + ((size_t)b * m + row) * dv;
#pragma unroll
    for (int e = 0; e < 4; e++) {  // a lane's columns are 16 g .. + 15: 4 e + x from tile x
      uint32_t z[4];
#pragma unroll
      for (int x = 0; x < 4; x++) {
        int sum = (int)reduce_p(o[x][e]);
#pragma unroll
        for (int u = 0; u < KW - 1; u++) {
          sum += part[((u * RG + rg) * 16 + 4 * x + e) * 64 + lane];
        }
        z[x] = fp_from_residues(reduce_p((int)__umul24((uint32_t)sum, inv)), 0u);
      }
      if (16 * g + 4 * e < dv) {
        *reinterpret_cast<uint2 *>(og + 16 * g + 4 * e) = uint2{z[0] | (z[1] << 16), z[2] | (z[3] << 16)};
      }
    }
  }
  // ---- P: the values of E are 113 u with u < 227, and those of P 113 (u inverse mod 227)
  uint32_t const inv_of[2] = {(uint32_t)sums[16 * rg + l8], (uint32_t)sums[16 * rg + 8 + l8]};
#pragma unroll 2
  for (int group = 0; group < groups; group++) {
    int const key = (group * KW + kw) * kChunk + 8 * ch8;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      int const r = row0 + 8 * i + l8;
      if (r < m && key < n) {
        size_t const at = ((size_t)b * m + r) * n + key;  // (what this lane stored above)
        uint4v x = *reinterpret_cast<uint4v const *>(A.e + at);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          auto times = [&](uint32_t v) {
            return __umul24(residue_p(__umul24(__umul24(v, 580u) >> 16, inv_of[i])), (uint32_t)FP_Q);
          };
          x[u] = times(x[u] & 0xffffu) | (times(x[u] >> 16) << 16);
        }
        *reinterpret_cast<uint4v *>(A.p + at) = x;
      }
    }
  }
}

}  // namespace

}  // namespace mi355

using namespace mi355;

extern "C" int mi355_fp_attention_rows(uint16_t const *Q, uint16_t const *K, uint16_t const *V, uint16_t *S, uint16_t *E, uint16_t *R,
                                       uint16_t *P, uint16_t *O, int batch, int m, int n, int d, int dv, int *taken) {
  MI355_REQUIRE_INIT();
  if (taken == nullptr) {
    return fail(MI355_ERR_INVALID, "no place for the answer");
  }
  *taken = 0;
  if (batch < 0 || m < 0 || n < 0 || d < 0 || dv < 0) {
    return fail(MI355_ERR_INVALID, "negative extent");
  }
  // One patch of K and V wide, rows of whole 16-byte chunks; a lane's sums of n products of bytes stay in 31 bits.
  // Few rows of many keys are a chain here and spread over the chip there (one head of 16 rows, us as above:
  // 1536 keys 60.8 / 69.6, 2048 69.3 / 64.5; 32 heads of 64 rows 81 / 83; 16 of 256 77.7 / 94).
  bool aligned = true;
  for (void const *p : {(void const *)Q, (void const *)K, (void const *)V, (void const *)S, (void const *)E, (void const *)P, (void const *)O}) {
    aligned = aligned && (reinterpret_cast<uintptr_t>(p) & 15) == 0;
  }
  if (state().fp_vector_dot_only || batch == 0 || m == 0 || n < 8 || n % 8 != 0 || n > 65536 || d < 4 || d > 64 || d % 4 != 0 || dv < 4 || dv > 64 ||
      dv % 4 != 0 || !aligned || (n > 1536 && (long long)batch * m * n < (4LL << 20))) {
    return MI355_OK;
  }
  if ((long long)batch * ((m + 15) / 16) > 2147483647LL) {
    return MI355_OK;
  }
  auto go = [&](auto *fn, int rg, int kw) -> int {
    int const slices = (m + 16 * rg - 1) / (16 * rg), lds = rows_lds(rg * kw, kw);
    FpRows const A{Q, K, V, S, E, R, P, O, m, n, d, dv, slices, (unsigned)batch * (unsigned)slices};
    MI355_GRANT_LDS(fn, lds);
    MI355_HIP(launch_kernel(fn, A.total, 64 * rg * kw, lds, state().stream(), A, tables()));
    return MI355_OK;
  };
  // Eight wavefronts, to 16 rows where those workgroups all run at once, to 32 where they do not (us of a
  // verification, with the other graph's launches: 16 x 256 rows x 2048 keys 77.7 / 86.2, 32 x 256 x 1024 83.5 /
  // 72.1); four where that many chunks of keys are not there (256 keys: 43.0 / 45.0).
  int rc;
  if ((long long)batch * ((m + 15) / 16) > 256) {
    rc = go(fp_attention_rows_kernel<2, 4>, 2, 4);
  } else if (n > 4 * kChunk) {
    rc = go(fp_attention_rows_kernel<1, 8>, 1, 8);
  } else {
    rc = go(fp_attention_rows_kernel<1, 4>, 1, 4);
  }
  if (rc != MI355_OK) {
    return rc;
  }
  *taken = 1;
  return MI355_OK;
}
