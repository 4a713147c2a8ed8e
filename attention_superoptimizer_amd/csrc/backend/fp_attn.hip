// Fingerprints of attention plans (load Q, K, V; S = Q . K; E = exp(S); [P = E / row sum]; O = E . V or
// P . V; sums over the for-loop) without a tile of 16-bit values anywhere.
//
// The ring is Z_227 x Z_113, and an exponential has residue 0 modulo 113 and depends on its argument
// modulo 113 alone.  So S is needed modulo 113 only, everything after it modulo 227 only: two int8
// matrix products with a table lookup between them.  The division by a row's sum is a factor common
// to the row, applied to the row of O.  (Plans that divide by the row sum of the SCORES, before the
// exponential, need that sum modulo 227: SCORES adds the second product.)
//
// A workgroup of four wavefronts owns up to 64 query rows of a logical block.  A wavefront has 16 rows,
// or shares them with the others and takes every KW-th chunk of 64 keys where there are few rows.  A
// chunk of K and V goes from memory (the next chunk is in flight while this one is multiplied) through
// registers, where 4 x 4 patches are reduced to bytes and turned, into LDS as MFMA operands; K^T is the
// first operand, so a lane ends up with 16 scores of one query, looks their exponentials up and has the
// second product's operand without exchanging anything (V's keys are stored in the order that gives).
//
// What bounds it: the vector instructions that reduce and look up (the matrix products are a tenth).
// The interpreter ran these plans operator by operator on 16-bit tiles in LDS: 32 x 16 blocks of
// 64 x 64 tiles, 4 iterations: 64 us there; 14.5 with residues one value at a time and staging writes
// that met in the banks, 12.9 here.
#include "common.h"
#include "tb_program.h"

namespace mi355 {

namespace {

constexpr int kThreads = 256, kChunk = 64;   // keys
constexpr int kPitch = 80;                   // bytes of an LDS row of 64 residues
constexpr int kPlane = 64 * kPitch;
constexpr int kExpBelow = 56;                // table entries below 0 (see the lookup)
typedef int v4i __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int scalar(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Where a tile starts: elements per step of the three block coordinates and of the iteration.
struct FpTile {
  uint16_t *ptr;
  long long lin[4];
  int ld;
};
// What the kernel needs of a program (a record of 3 KB whose operators it would look up by number).
struct FpAttn {
  FpTile q, k, v, o, r;  // r.ptr: null when the row sums are not stored
  int m, d, n, dv, forloop;
  int divide, scores;
  int grid_x, grid_y, slices, kw;
};

__host__ __device__ __forceinline__ FpTile fp_tile(DevProgram const &P, int op) {
  FpTile t{nullptr, {0, 0, 0, 0}, 0};
  if (op < 0) {
    return t;
  }
  DevOp const &d = P.ops[op];
  t.ptr = static_cast<uint16_t *>(d.kind == DOP_LOAD ? const_cast<void *>(P.in[d.io]) : P.out[d.io]);
  t.ld = d.d_cols;
  for (int i = 0; i < 3; i++) {
    t.lin[i] = d.g_bs[i] + (long long)d.row_bs[i] * d.d_cols + d.col_bs[i];
  }
  t.lin[3] = d.g_fs + (long long)d.row_fs * d.d_cols + d.col_fs;
  return t;
}
__host__ __device__ __forceinline__ FpAttn fp_attn_args(DevProgram const &P) {
  return FpAttn{fp_tile(P, P.fg[0]), fp_tile(P, P.fg[1]), fp_tile(P, P.fg[2]), fp_tile(P, P.fg[3]), fp_tile(P, P.fg[4]),
                P.t[P.ops[P.fg[0]].dst].rows, P.t[P.ops[P.fg[0]].dst].cols, P.t[P.ops[P.fg[1]].dst].cols,
                P.t[P.ops[P.fg[2]].dst].cols, P.forloop_range, P.fg[5] & 1, (P.fg[5] >> 1) & 1, P.grid[0], P.grid[1],
                P.pl_geo[0], P.pl_geo[1]};
}
__device__ __forceinline__ uint16_t *tile_at(FpTile const &t, int bx, int by, int bz, int it) {
  return t.ptr + bx * t.lin[0] + by * t.lin[1] + bz * t.lin[2] + it * t.lin[3];
}

template <int KW, bool SCORES>
__device__ __forceinline__ void fp_attn_block(FpAttn const &P, FpTables const t, unsigned char *lds, int bx, int by, int bz,
                                              int slice) {
  constexpr int RG = 4 / KW, PLANES = SCORES ? 3 : 2;
  int const tid = threadIdx.x, lane = tid % 64, wave = scalar(tid / 64), g = lane / 16, c = lane % 16;
  int const kw = wave % KW, rg = wave / KW;
  int8_t *const exps = reinterpret_cast<int8_t *>(lds) + kExpBelow;       // [-56, 113)
  uint8_t *const inverse = reinterpret_cast<uint8_t *>(lds) + 176;       // [227]
  int *const sums = reinterpret_cast<int *>(lds + 416);                  // [KW][16 RG]
  unsigned char *const tiles = lds + 416 + 256;                          // [KW][PLANES][64][kPitch]
  if (tid < (int)FP_Q + kExpBelow) {
    int const x = tid - kExpBelow;
    exps[x] = static_cast<int8_t>(residue_p_signed(t.exp_tbl[x < 0 ? x + (int)FP_Q : x]));
  }
  if (tid < (int)FP_P) {
    inverse[tid] = static_cast<uint8_t>(t.div_p[tid]);
  }

  bool const divide = P.divide != 0;
  int const m = P.m, d = P.d, n = P.n, dv = P.dv;
  int const F = P.forloop, chunks = (n + kChunk - 1) / kChunk, groups = (chunks + KW - 1) / KW;
  int const ld_q = P.q.ld, ld_k = P.k.ld, ld_v = P.v.ld;

  // ---- query residues: row c, elements 16 g .. + 15
  int const row = (slice * RG + rg) * 16 + c;
  v4i qf, qp;
  {
    uint16_t const *q = tile_at(P.q, bx, by, bz, 0) + (long long)(row < m ? row : m - 1) * ld_q;
    uint2 x[1][4];
#pragma unroll
    for (int w = 0; w < 4; w++) {
      int const at = 16 * g + 4 * w;
      x[0][w] = uint2{0, 0};
      if (at < d) {
        x[0][w] = *reinterpret_cast<uint2 const *>(q + at);
      }
    }
    if (fp_past_residues(fp_bits(x))) {
      fp_into_ring(x);
    }
#pragma unroll
    for (int w = 0; w < 4; w++) {
      uint32_t rp, rq;
      residues_row(x[0][w], rp, rq);
      qf[w] = (int)rq;
      qp[w] = (int)rp;
    }
  }

  // ---- staging: patch (hi, lo) of a chunk of K is 4 rows from 4 hi, 4 columns from 4 lo; of V, 4 columns
  // from 4 lo of the keys 16 (hi / 4) + 4 i + hi % 4.  Column 4 lo + u becomes row lo of matrix tile u: the
  // lanes of a write differ in their banks, and a lane's scores are those of keys 16 g + 4 r + j, which is
  // the order V's keys then have.
  int const hi = tid / 16, lo = tid % 16;
  // (past the end of a tile the last patch stands in: elements of K past d meet zeros of Q, keys past n
  // are masked, elements of V past dv are not stored)
  uint2 kr[KW][4], vr[KW][4];
  auto fetch = [&](int it, int group) {
    uint16_t const *const k = tile_at(P.k, bx, by, bz, it);
    uint16_t const *const v = tile_at(P.v, bx, by, bz, it);
#pragma unroll
    for (int w = 0; w < KW; w++) {
      int const key0 = (group * KW + w) * kChunk;
      int const kk = min(4 * hi, d - 4), kc = min(key0 + 4 * lo, n - 4), vc = min(4 * lo, dv - 4);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        kr[w][i] = *reinterpret_cast<uint2 const *>(k + (long long)(kk + i) * ld_k + kc);
        int const vk = min(key0 + 16 * (hi / 4) + 4 * i + hi % 4, n - 1);
        vr[w][i] = *reinterpret_cast<uint2 const *>(v + (long long)vk * ld_v + vc);
      }
    }
  };
  auto put = [&]() {
#pragma unroll
    for (int w = 0; w < KW; w++) {
      unsigned char *const kq = tiles + w * PLANES * kPlane, *const vp = kq + kPlane, *const kp = vp + kPlane;
      uint32_t p[4], q[4], v[4], unused[4];
      residues_patch(kr[w], p, q);
      residues_patch(vr[w], v, unused);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        int const at = (16 * u + lo) * kPitch + 4 * hi;
        *reinterpret_cast<uint32_t *>(kq + at) = q[u];
        if (SCORES) {
          *reinterpret_cast<uint32_t *>(kp + at) = p[u];
        }
        *reinterpret_cast<uint32_t *>(vp + at) = v[u];
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

  v4i o[4], total[4];
  int rs = 0, r_total = 0;
#pragma unroll
  for (int x = 0; x < 4; x++) {
    o[x] = total[x] = v4i{0, 0, 0, 0};
  }
  // scores modulo 113 start from a multiple of 113 that keeps them above zero
  constexpr int kBase = 113 * 2500;
  v4i const zero = {0, 0, 0, 0}, base = {kBase, kBase, kBase, kBase};
  // (sums of bytes: a chunk adds less than 2^20 to an element of O, so they are folded long before
  // they could reach 2^31)
  int folded = 0;
  fetch(0, 0);
  int const steps = F * groups;
  for (int s = 0, it = 0, group = 0; s < steps; s++) {
    __syncthreads();
    stage();
    __syncthreads();
    int const this_group = group, next_it = group + 1 < groups ? it : it + 1;
    bool const last = group + 1 == groups;  // of the iteration
    group = last ? 0 : group + 1;
    if (s + 1 < steps) {
      fetch(next_it, group);
    }
    int const key0 = (this_group * KW + kw) * kChunk;
    if (key0 < n) {
      unsigned char const *const kq = tiles + kw * PLANES * kPlane, *const vp = kq + kPlane, *const kp = vp + kPlane;
      // keys past the tile (exp(0) is not zero): the first `inside` bytes of every e[j] count
      int const inside = (n - key0 - 16 * g) / 4;
      uint32_t const mask = inside >= 4 ? ~0u : inside <= 0 ? 0u : (1u << (8 * inside)) - 1;
      v4i e;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        v4i const k = *reinterpret_cast<v4i const *>(kq + (16 * j + c) * kPitch + 16 * g);
        v4i const x = __builtin_amdgcn_mfma_i32_16x16x64_i8(k, qf, base, 0, 0, 0);
        if (SCORES) {
          v4i const y = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<v4i const *>(kp + (16 * j + c) * kPitch + 16 * g),
                                                              qp, zero, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; r++) {
            rs += r < inside ? y[r] : 0;
          }
        }
        // A score is within 64 * 66^2 of the base: in (0, 2^20).  2320 = ceil(2^18 / 113) gives its quotient or one more:
        // the remainder is in [-49, 112], and the table starts below zero.
        int b[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          b[r] = exps[(int)mad24((uint32_t)__umul24((uint32_t)x[r], 2320u) >> 18, -(int)FP_Q, (uint32_t)x[r])];
        }
        e[j] = (int)(pack_bytes((uint32_t)b[0], (uint32_t)b[1], (uint32_t)b[2], (uint32_t)b[3]) & mask);
        if (!SCORES) {
          rs = __builtin_amdgcn_sdot4(e[j], 0x01010101, rs, false);
        }
      }
#pragma unroll
      for (int x = 0; x < 4; x++) {
        v4i const v = *reinterpret_cast<v4i const *>(vp + (16 * x + c) * kPitch + 16 * g);
        o[x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v, e, o[x], 0, 0, 0);
      }
    }
    if (last) {
      it = next_it;
      if (divide) {
        // the row's sum over all its keys, then its inverse
        rs = (int)reduce_p(rs);
        rs += __shfl_xor(rs, 16, 64);
        rs += __shfl_xor(rs, 32, 64);
        uint32_t y = reduce_p(rs);
        if (KW > 1) {
          if (g == 0) {
            sums[kw * 16 * RG + rg * 16 + c] = (int)y;
          }
          __syncthreads();
          int all = 0;
#pragma unroll
          for (int w = 0; w < KW; w++) {
            all += sums[w * 16 * RG + rg * 16 + c];
          }
          y = reduce_p(all);
        }
        if (P.r.ptr != nullptr) {  // (each wavefront holds the whole sum: one of them counts)
          r_total += kw == 0 && g == 0 ? (int)y : 0;
        }
        uint32_t const inv = inverse[y];
#pragma unroll
        for (int x = 0; x < 4; x++) {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            total[x][r] += (int)__umul24(reduce_p(o[x][r]), inv);
            o[x][r] = 0;
          }
        }
        rs = 0;
      }
      folded += groups;
      if (folded >= 1000) {
        folded = 0;
#pragma unroll
        for (int x = 0; x < 4; x++) {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            o[x][r] = (int)reduce_p(o[x][r]);
            total[x][r] = (int)reduce_p(total[x][r]);
          }
        }
        rs = (int)reduce_p(rs);
      }
    }
  }
  if (!divide) {
#pragma unroll
    for (int x = 0; x < 4; x++) {
      total[x] = o[x];
    }
    rs = (int)reduce_p(rs);
    rs += __shfl_xor(rs, 16, 64);
    rs += __shfl_xor(rs, 32, 64);
    r_total = g == 0 ? (int)reduce_p(rs) : 0;
  }
  if (KW > 1) {  // the wavefronts' keys together
    int *const part = reinterpret_cast<int *>(tiles);  // [KW - 1][RG][17][64]
    __syncthreads();
    if (kw > 0) {
      int *const mine = part + ((kw - 1) * RG + rg) * 17 * 64 + lane;
#pragma unroll
      for (int x = 0; x < 16; x++) {
        mine[x * 64] = (int)reduce_p(total[x / 4][x % 4]);
      }
      mine[16 * 64] = r_total;
    }
    __syncthreads();
    if (kw == 0) {
#pragma unroll
      for (int w = 0; w < KW - 1; w++) {
        int const *const theirs = part + (w * RG + rg) * 17 * 64 + lane;
#pragma unroll
        for (int x = 0; x < 16; x++) {
          total[x / 4][x % 4] = (w == 0 ? (int)reduce_p(total[x / 4][x % 4]) : total[x / 4][x % 4]) + theirs[x * 64];
        }
        r_total += theirs[16 * 64];
      }
    }
  }
  if (kw != 0 || row >= m) {
    return;
  }
  uint16_t *const og = tile_at(P.o, bx, by, bz, 0) + (long long)row * P.o.ld;
#pragma unroll
  for (int e = 0; e < 4; e++) {  // a lane's columns are 16 g .. + 15: 4 e + x from tile x
    if (16 * g + 4 * e < dv) {
      uint32_t z[4];
#pragma unroll
      for (int x = 0; x < 4; x++) {
        z[x] = fp_from_residues(reduce_p(total[x][e]), 0u);
      }
      *reinterpret_cast<uint2 *>(og + 16 * g + 4 * e) = uint2{z[0] | (z[1] << 16), z[2] | (z[3] << 16)};
    }
  }
  if (P.r.ptr != nullptr && g == 0) {
    tile_at(P.r, bx, by, bz, 0)[(long long)row * P.r.ld] = static_cast<uint16_t>(fp_from_residues(reduce_p(r_total), 0u));
  }
}

constexpr int attn_lds(int kw, bool scores) { return 416 + 256 + kw * (scores ? 3 : 2) * kPlane; }

template <int KW, bool SCORES>
__device__ __forceinline__ void fp_attn_workgroup(FpAttn const &P, FpTables const t, unsigned char *lds, int w) {
  int const slice = w % P.slices;
  w /= P.slices;
  fp_attn_block<KW, SCORES>(P, t, lds, w % P.grid_x, w / P.grid_x % P.grid_y, w / P.grid_x / P.grid_y, slice);
}

template <int KW, bool SCORES>
__global__ __launch_bounds__(kThreads) void fp_attn_kernel(FpAttn const P, FpTables const t) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  // an XCD (one L2) gets consecutive blocks: they share keys and values
  unsigned const total = gridDim.x, xcd = blockIdx.x % 8, each = total / 8, more = total % 8;
  fp_attn_workgroup<KW, SCORES>(P, t, lds, (int)(xcd * each + (xcd < more ? xcd : more) + blockIdx.x / 8));
}

// many programs in one launch: workgroup -> program by a prefix table
__global__ __launch_bounds__(kThreads) void fp_attn_multi_kernel(DevProgram const *__restrict__ progs,
                                                                int const *__restrict__ first_block, int n, FpTables const t) {
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
  FpAttn const P = fp_attn_args(progs[scalar(lo)]);
  int const v = w - first_block[lo];
  if (P.scores) {
    P.kw == 1 ? fp_attn_workgroup<1, true>(P, t, lds, v) : P.kw == 2 ? fp_attn_workgroup<2, true>(P, t, lds, v) : fp_attn_workgroup<4, true>(P, t, lds, v);
  } else {
    P.kw == 1 ? fp_attn_workgroup<1, false>(P, t, lds, v) : P.kw == 2 ? fp_attn_workgroup<2, false>(P, t, lds, v) : fp_attn_workgroup<4, false>(P, t, lds, v);
  }
}

}  // namespace

// Recognises the family in a lowered uint16 program; marks it (fused = 5) and notes its operators:
// fg = loaders of Q, K, V, saver of O, saver of the row sums or -1, 1 (divided) | 2 (by the sum of the
// scores); pl_geo = workgroups per logical block, wavefronts per row group.
bool fp_attn_applicable(DevProgram &P) {
  int loads[3], n_loads = 0, mm1 = -1, mm2 = -1, exp = -1, red = -1, div = -1, out_o = -1, out_r = -1;
  for (int o = 0; o < P.num_ops; o++) {
    DevOp const &d = P.ops[o];
    int const s = mm1 < 0 ? -1 : P.ops[mm1].dst;  // the scores, exponentials once exp is there
    switch (d.kind) {
      case DOP_LOAD:
        if (n_loads == 3) {
          return false;
        }
        loads[n_loads++] = o;
        break;
      case DOP_MATMUL:
        if (mm1 < 0) {
          mm1 = o;
        } else if (mm2 < 0 && exp >= 0 && d.src0 == (div >= 0 ? P.ops[div].dst : s)) {
          mm2 = o;
        } else {
          return false;
        }
        break;
      case DOP_UNARY:
        if (exp >= 0 || mm1 < 0 || d.sub != TB_EXP_OP || d.dst != s) {
          return false;
        }
        exp = o;
        break;
      case DOP_REDUCE:
        if (red >= 0 || mm1 < 0 || d.src0 != s || d.red_inner != 1 || d.red_deg != P.t[s].cols) {
          return false;
        }
        red = o;
        break;
      case DOP_BINARY:
        if (div >= 0 || d.sub != TB_DIV_OP || exp < 0 || red < 0 || d.src0 != s || d.src1 != P.ops[red].dst ||
            P.t[d.src1].rows != P.t[s].rows || P.t[d.src1].cols != 1) {
          return false;
        }
        div = o;
        break;
      case DOP_OUTPUT:
        if (mm2 >= 0 && d.src0 == P.ops[mm2].dst && out_o < 0) {
          out_o = o;
        } else if (red >= 0 && d.src0 == P.ops[red].dst && out_r < 0) {
          out_r = o;
        } else {
          return false;
        }
        break;
      default:
        return false;
    }
  }
  if (n_loads != 3 || mm2 < 0 || out_o < 0) {
    return false;
  }
  bool const scores = red >= 0 && red < exp;
  if (scores && (div < 0 || out_r >= 0)) {
    return false;  // (a sum of scores is only a divisor)
  }
  auto loader = [&](int tensor) {
    for (int o : loads) {
      if (P.ops[o].dst == tensor) {
        return o;
      }
    }
    return -1;
  };
  int const q = loader(P.ops[mm1].src0), k = loader(P.ops[mm1].src1), v = loader(P.ops[mm2].src1);
  if (q < 0 || k < 0 || v < 0 || q == k || k == v || q == v) {
    return false;
  }
  DevTensor const &tq = P.t[P.ops[q].dst], &tk = P.t[P.ops[k].dst], &tv = P.t[P.ops[v].dst];
  DevTensor const &to = P.t[P.ops[out_o].src0];
  if (tq.cols > 64 || tv.cols > 64 || tq.cols % 4 != 0 || tv.cols % 4 != 0 || tk.cols % 4 != 0 || tk.cols > 8192 ||
      tk.rows != tq.cols || tv.rows != tk.cols || to.rows != tq.rows || to.cols != tv.cols) {
    return false;
  }
  // the query tile does not move with the for-loop; every 4 x 4 patch of K and V, 4 elements of Q and O
  // are 8-byte accesses
  DevOp const &dq = P.ops[q];
  if (P.forloop_range > 1 && (dq.row_fs != 0 || dq.col_fs != 0 || dq.g_fs != 0)) {
    return false;
  }
  for (int o : {q, k, v, out_o}) {
    DevOp const &d = P.ops[o];
    bool ok = d.d_cols % 4 == 0 && d.col_fs % 4 == 0 && d.g_fs % 4 == 0 &&
              (reinterpret_cast<uintptr_t>(d.kind == DOP_LOAD ? P.in[d.io] : P.out[d.io]) & 7) == 0;
    for (int i = 0; i < 3; i++) {
      ok = ok && d.col_bs[i] % 4 == 0 && d.g_bs[i] % 4 == 0;
    }
    if (!ok) {
      return false;
    }
  }
  int const row_groups = (tq.rows + 15) / 16, rg = row_groups >= 3 ? 4 : row_groups;
  P.fused = 5;
  P.fg[0] = q;
  P.fg[1] = k;
  P.fg[2] = v;
  P.fg[3] = out_o;
  P.fg[4] = out_r;
  P.fg[5] = (div >= 0 ? 1 : 0) | (scores ? 2 : 0);
  P.pl_geo[0] = (row_groups + rg - 1) / rg;
  P.pl_geo[1] = 4 / rg;
  P.lds_bytes = attn_lds(P.pl_geo[1], scores);
  return (long long)P.grid[0] * P.grid[1] * P.grid[2] * P.pl_geo[0] <= 2147483647LL;
}

int launch_fp_attn(DevProgram const &P, hipStream_t stream) {
  FpAttn const A = fp_attn_args(P);
  auto *fn = A.scores ? (A.kw == 1 ? fp_attn_kernel<1, true> : A.kw == 2 ? fp_attn_kernel<2, true> : fp_attn_kernel<4, true>)
                      : (A.kw == 1 ? fp_attn_kernel<1, false> : A.kw == 2 ? fp_attn_kernel<2, false> : fp_attn_kernel<4, false>);
  MI355_GRANT_LDS(fn, P.lds_bytes);
  MI355_HIP(launch_kernel(fn, (unsigned)fp_program_blocks(P), kThreads, P.lds_bytes, stream, A, tables()));
  return MI355_OK;
}

int launch_fp_attn_multi(DevProgram const *progs, int const *first_block, int n, int blocks, int lds_bytes, hipStream_t stream) {
  MI355_GRANT_LDS(fp_attn_multi_kernel, lds_bytes);
  MI355_HIP(launch_kernel(fp_attn_multi_kernel, (unsigned)blocks, kThreads, lds_bytes, stream, progs, first_block, n, tables()));
  return MI355_OK;
}

}  // namespace mi355
