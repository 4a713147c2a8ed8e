// Shared state and helpers of the gfx950 backend (internal; not part of the ABI).
#pragma once

#include "mi355_abi.h"
#include "launch.h"
#include <hip/hip_runtime.h>
#include <cstdarg>
#include <cstdint>
#include <cstdio>

namespace mi355 {

// Fingerprint ring constants (reference include/mirage/type.h:26-34).
constexpr uint32_t FP_P = 227;
constexpr uint32_t FP_Q = 113;
constexpr uint32_t FP_EXP_BASE = 3;
constexpr uint32_t FP_PQ = 25651;
constexpr uint32_t FP_P_MUL_Q_MOD_1 = 227;
constexpr uint32_t FP_Q_MUL_P_MOD_1 = 25425;

// Operator type codes (reference include/mirage/type.h:50-62, 79-103).
enum : int {
  KN_EXP_OP = 1007,
  KN_ADD_OP = 1008,
  KN_MUL_OP = 1009,
  KN_DIV_OP = 1010,
  KN_SILU_OP = 1011,  // extension
  TB_INPUT_OP = 2001,
  TB_OUTPUT_OP = 2002,
  TB_MATMUL_OP = 2003,
  TB_EXP_OP = 2007,
  TB_ADD_OP = 2008,
  TB_MUL_OP = 2009,
  TB_DIV_OP = 2010,
  TB_SILU_OP = 2012,  // extension
  TB_REDUCTION_0_OP = 2101,
  TB_REDUCTION_2_TO_DIMX_OP = 2106,
  TB_CONCAT_0_OP = 2200,
  TB_CONCAT_2_OP = 2202,
};

extern thread_local int tls_queue;  // the calling thread's queue, see mi355_queue_select

struct State {
  bool ready = false;
  int device = 0;
  // Work is enqueued on the calling host thread's selected queue (queue 0 unless the
  // thread chose another); the others exist so independent candidates can overlap their
  // small kernels and host threads can enqueue side by side.
  hipStream_t queues[MI355_NUM_QUEUES] = {};
  hipStream_t stream() const { return queues[tls_queue]; }
  char *arena = nullptr;
  size_t arena_bytes = 0;
  // device copies of the lookup tables, reference layout
  uint16_t *exp_tbl = nullptr, *div_p = nullptr, *div_q = nullptr;
  int *flag_host = nullptr;   // answers of mi355_fp_equal, pinned: one int per queue, 64 bytes apart
  int *flag = nullptr;        // the same memory as the device addresses it
  int *queue_flag() const { return flag + 16 * tls_queue; }
  int *queue_flag_host() const { return flag_host + 16 * tls_queue; }
  int *cmp_host = nullptr;    // MI355_COMPARE_SLOTS mismatch flags of deferred compares, in
                              // pinned host memory
  int *cmp_slots = nullptr;   // the same memory as the device addresses it
  hipEvent_t marks[MI355_NUM_MARKS][MI355_NUM_QUEUES] = {};
  hipEvent_t ev0[MI355_NUM_QUEUES] = {}, ev1[MI355_NUM_QUEUES] = {};  // timer pair per queue
  hipEvent_t pace[MI355_NUM_QUEUES][2] = {};  // markers that bound how far a timed loop runs ahead
  int max_lds = 65536;
  // staging of batched launches (mi355_customized_fp_batch): per queue a small ring of
  // pinned host / device buffer pairs that carry the program records of one call
  static constexpr int kBatchSlots = 16;
  static constexpr size_t kBatchSlotBytes = (size_t)256 << 10;
  struct BatchSlot {
    char *host = nullptr;
    char *dev = nullptr;
    hipEvent_t copied = nullptr;  // the host buffer may be rewritten once this has passed
  };
  BatchSlot batch[MI355_NUM_QUEUES][kBatchSlots];
  int batch_next[MI355_NUM_QUEUES] = {};
  // what the last customized-op call of each queue launched (a queue is driven by one host
  // thread at a time, so per-queue records never mix)
  mi355_launch_info launches[MI355_NUM_QUEUES] = {};
  mi355_launch_info &last() { return launches[tls_queue]; }
  int force_interpreter = 0;
  int attention_mode = 0;  // 0 auto, 1 latency kernel only, 2 throughput kernel when it fits
  int fp_vector_dot_only = 0;  // 1: fingerprint matmuls never take the matrix-core kernels
  int fp_big_tiles = 1;        // 0: large kernel-level matmuls keep 64 x 64 tiles
  int fp_big_tiles_ok = 1;     // 0: the self-check of the 128-row tile kernels failed on this
                               // device / build: they stay off whatever fp_big_tiles says
  int plan_smem_layout = 0;  // 1: loader tiles take the LDS layout their plan declares
  int direct_lanes = 0;      // MI355_OPT_DIRECT_LANES
  int gemm_mode = 0;         // MI355_OPT_GEMM_MODE
  int f16_matmul_route = 0;  // MI355_OPT_F16_MATMUL_ROUTE
  int any_size_kernels = 0;  // MI355_OPT_ANY_SIZE_KERNELS
  // phase timestamps of the direct-staging attention kernel (MI355_OPT_PHASE_TRACE): while
  // set, launches of that kernel record six wall-clock stamps per wavefront here
  unsigned long long *phase_trace = nullptr;        // null while tracing is off
  unsigned long long *phase_trace_store = nullptr;  // the allocation (first use of the option)
  size_t phase_trace_bytes = 0;
  // fused-kernel workspace: fp16 range sums of split for-loops
  // (each queue has its own slice of scratch_base, so concurrent queues never share)
  size_t scratch_bytes = 0;  // per queue
  char *scratch_base = nullptr;
  void *scratch() const {
    return scratch_base == nullptr ? nullptr : scratch_base + (size_t)tls_queue * scratch_bytes;
  }
  // residue planes of the matrix-core fingerprint matmul (per queue, like scratch)
  size_t planes_bytes = 0;
  char *planes_base = nullptr;
  char *planes() const {
    return planes_base == nullptr ? nullptr : planes_base + (size_t)tls_queue * planes_bytes;
  }
  // Tickets of launches whose last workgroup goes on with the work of all (attention_fold.h): per queue
  // kTickets ints, zero whenever no launch that uses them runs.
  static constexpr int kTickets = 1 << 16;
  int *tickets = nullptr;
};

State &state();
// `count` tickets of a queue that nobody else has until they are given back, or null: a launch that is made again
// and again has its own, so that two of them never meet.  Given back they go to a later launch of the same queue,
// behind the earlier one in it; `life` tells this mi355_init's from an earlier one's.
int *take_tickets(int queue, int count, unsigned &life);
void give_tickets(int queue, int *tickets, int count, unsigned life);

// Raises the dynamic LDS limit of a kernel to what the device has, once per kernel: the call costs
// the host several microseconds.  A launch that requests at most 64 KB needs none.
int grant_lds(void const *fn, int lds);
#define MI355_GRANT_LDS(fn, lds)                                                \
  do {                                                                          \
    if (int rc_ = ::mi355::grant_lds(reinterpret_cast<void const *>(fn), lds)) { \
      return rc_;                                                               \
    }                                                                           \
  } while (0)

// Matrix-core fingerprint matmul (fp_mfma.hip): whether a single matmul is large enough to
// repay the extra launch that splits its operands into residue planes, and its launch.
bool mfma_matmul_pays(int batch, int m, int n, int k);
int launch_mfma_matmul(uint16_t const *A, uint16_t const *B, uint16_t *C, int batch, int m, int n,
                       int k);
int sync_all_queues();
// Drops what mi355_customized_profile keeps of its last call per queue and the launches of prepared
// operators (tb_interp.hip); options_generation() counts how often.
void drop_profile_replays();
unsigned options_generation();
// The vendor library's GEMM on the calling thread's queue (vendor_gemm.cc): row-major C =
// A . B for `batch` matrices, each operand in either storage order; MI355_ERR_UNSUPPORTED
// when the library cannot be loaded.  vendor_gemm_release drops its per-queue handles.
int vendor_gemm(void const *A, void const *B, void *C, int batch, int m, int n, int k, int a_column_major,
                int b_column_major);
int vendor_gemm_release();
// Looks up the device address of the file-scope scratch array behind
// mi355_customized_fp_static (tb_interp.hip); called by mi355_init with `device` current.
int static_scratch_setup(int device);
int fail(int code, char const *fmt, ...);

#define MI355_HIP(expr)                                                             \
  do {                                                                              \
    hipError_t e_ = (expr);                                                         \
    if (e_ != hipSuccess) {                                                         \
      return ::mi355::fail(MI355_ERR_HIP, "%s failed: %s (%s:%d)", #expr,           \
                           hipGetErrorString(e_), __FILE__, __LINE__);              \
    }                                                                               \
  } while (0)

#define MI355_REQUIRE_INIT()                                                        \
  do {                                                                              \
    if (!::mi355::state().ready) {                                                  \
      return ::mi355::fail(MI355_ERR_NOT_INITIALISED, "mi355_init has not run");    \
    }                                                                               \
  } while (0)

// a b + c with 24-bit a and b: an instruction of full rate, spelled out because the compiler, which sees
// that only the low bits of a residue are asked for, puts a 64-bit multiply-add at a quarter of it in
// its place.  Bits of `a` beyond 24 cost the result its bits beyond 24.
__device__ __forceinline__ uint32_t mad24(uint32_t a, int b, uint32_t c) {
  uint32_t r;
  asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
  return r;
}
// Residues of a 16-bit value.  The compiler lowers `%` by a constant to 32-bit multiply-highs, which
// run at a quarter of the rate of a 24-bit multiply; for values below 2^16 a 24-bit reciprocal is exact
// (37118 = ceil(2^22 / 113); 36954 = floor(2^23 / 227), so the value is taken one higher).
__device__ __forceinline__ uint32_t residue_q(uint32_t x) {
  return mad24((uint32_t)__umul24(x, 37118u) >> 22, -(int)FP_Q, x);
}
__device__ __forceinline__ uint32_t residue_p(uint32_t x) {
  return mad24(((uint32_t)__umul24(x, 36954u) + 36954u) >> 23, -(int)FP_P, x);
}
// the residue modulo 227 in [-113, 113]: what a signed byte holds
__device__ __forceinline__ int residue_p_signed(uint32_t x) {
  return (int)mad24(((uint32_t)__umul24(x, 36954u) + 36954u * 114u) >> 23, -(int)FP_P, x);
}
// Residues of any 32-bit value: one multiply-high; the quotient times the modulus by a 24-bit multiply,
// of which only the low bits matter (a residue is below 2^8 / 2^15).
__device__ __forceinline__ uint32_t mod_p(uint32_t x) { return mad24(x / FP_P, -(int)FP_P, x) & 0xffu; }
__device__ __forceinline__ uint32_t mod_q(uint32_t x) { return mad24(x / FP_Q, -(int)FP_Q, x) & 0xffu; }
__device__ __forceinline__ uint32_t mod_pq(uint32_t x) { return mad24(x / FP_PQ, -(int)FP_PQ, x); }
// The ring value with residues p modulo 227 (p < 227) and q modulo 113 (any 16-bit q).  227 is 1
// modulo 113, so p + 227 t has residue p + t there: t = q - p.
__device__ __forceinline__ uint32_t fp_from_residues(uint32_t p, uint32_t q) {
  return mad24(residue_q(q + 2 * FP_Q - p), FP_P, p);
}
// four of them as bytes
__device__ __forceinline__ uint32_t pack_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  uint32_t const lo = __builtin_amdgcn_perm(b, a, 0x0c0c0400u), hi = __builtin_amdgcn_perm(d, c, 0x0c0c0400u);
  return lo | (hi << 16);
}
__device__ __forceinline__ uint32_t residues_q4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return pack_bytes(residue_q(a), residue_q(b), residue_q(c), residue_q(d));
}
__device__ __forceinline__ uint32_t residues_p4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return pack_bytes(residue_p(a), residue_p(b), residue_p(c), residue_p(d));
}
__device__ __forceinline__ uint32_t residues_p4_signed(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return pack_bytes((uint32_t)residue_p_signed(a), (uint32_t)residue_p_signed(b), (uint32_t)residue_p_signed(c),
                    (uint32_t)residue_p_signed(d));
}

// Residues of two values below 2^15 (16 bits each) as signed bytes, the low bytes of the halves of p and
// q: what the int8 matrix products want, at three instructions a value for both fields (ten through
// residue_p_signed and residue_q).  The quotient is estimated in packed fp16: added to 1536 it is rounded
// to an integer, whose low byte is the quotient's.  An estimate one off where the value lies close to the
// middle between two multiples leaves a remainder that still fits: over all of [0, 32768) they are in
// [-125, 117] modulo 227 and in [-66, 63] modulo 113.
typedef _Float16 fp_half2 __attribute__((ext_vector_type(2)));
typedef unsigned short fp_ushort2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void residue_pairs(uint32_t v, uint32_t &p, uint32_t &q) {
  fp_ushort2 const x = __builtin_bit_cast(fp_ushort2, v);
  fp_half2 const h = __builtin_convertvector(x, fp_half2), one_and_half_k = {(_Float16)1536.0f, (_Float16)1536.0f};
  fp_half2 const by_p = __builtin_bit_cast(fp_half2, 0x1c831c83u), by_q = __builtin_bit_cast(fp_half2, 0x20882088u);
  fp_ushort2 const tp = __builtin_bit_cast(fp_ushort2, __builtin_elementwise_fma(h, by_p, one_and_half_k));
  fp_ushort2 const tq = __builtin_bit_cast(fp_ushort2, __builtin_elementwise_fma(h, by_q, one_and_half_k));
  p = __builtin_bit_cast(uint32_t, (fp_ushort2)(x - tp * (unsigned short)FP_P));
  q = __builtin_bit_cast(uint32_t, (fp_ushort2)(x - tq * (unsigned short)FP_Q));
}
// A caller may write any 16-bit value: those of 2^15 and up are brought into the ring first, by at most two
// subtractions of 227 * 113 (below it x - 25651 wraps to more than x).  That would be two instructions a
// value (82.9 -> 87.6 us of a verification); so a wavefront looks at the top bits of what it has staged, a
// quarter of one, and only where it finds one set does it stage again (no difference in the kernels' times).
template <int A, int B>
__device__ __forceinline__ uint32_t fp_bits(uint2 const (&x)[A][B]) {
  uint32_t seen = 0;
#pragma unroll
  for (int a = 0; a < A; a++) {
#pragma unroll
    for (int b = 0; b < B; b++) {
      seen |= x[a][b].x | x[a][b].y;
    }
  }
  return seen;
}
__device__ __forceinline__ bool fp_past_residues(uint32_t seen) { return __any((int)(seen & 0x80008000u)) != 0; }
template <int A, int B>
__device__ __forceinline__ void fp_into_ring(uint2 (&x)[A][B]) {
  fp_ushort2 const ring = {(unsigned short)FP_PQ, (unsigned short)FP_PQ};
  auto pair = [&](uint32_t v) {
    fp_ushort2 r = __builtin_bit_cast(fp_ushort2, v);
    r = __builtin_elementwise_min(r, (fp_ushort2)(r - ring));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(r, (fp_ushort2)(r - ring)));
  };
#pragma unroll
  for (int a = 0; a < A; a++) {
#pragma unroll
    for (int b = 0; b < B; b++) {
      x[a][b] = uint2{pair(x[a][b].x), pair(x[a][b].y)};
    }
  }
}
// of four values in a row
__device__ __forceinline__ void residues_row(uint2 v, uint32_t &p, uint32_t &q) {
  uint32_t p0, q0, p1, q1;
  residue_pairs(v.x, p0, q0);
  residue_pairs(v.y, p1, q1);
  p = __builtin_amdgcn_perm(p1, p0, 0x06040200u);
  q = __builtin_amdgcn_perm(q1, q0, 0x06040200u);
}
// of the columns of four rows of four
__device__ __forceinline__ void residues_patch(uint2 const *rows, uint32_t *p, uint32_t *q) {
  auto turn = [](uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t *out) {
    uint32_t const ab = __builtin_amdgcn_perm(b, a, 0x06020400u), cd = __builtin_amdgcn_perm(d, c, 0x06020400u);
    out[0] = __builtin_amdgcn_perm(cd, ab, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(cd, ab, 0x07060302u);
  };
#pragma unroll
  for (int h = 0; h < 2; h++) {
    uint32_t pp[4], qq[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      residue_pairs(h == 0 ? rows[i].x : rows[i].y, pp[i], qq[i]);
    }
    turn(pp[0], pp[1], pp[2], pp[3], p + 2 * h);
    turn(qq[0], qq[1], qq[2], qq[3], q + 2 * h);
  }
}

// Fingerprint value from sums of products of such residues over k <= FEW ? 128 : 32768, the sums started
// from multiples of the moduli that keep them above zero: a negative sum would need a fix-up.  FEW: the
// sums are below 2^22, where 2^30 / 227 and 2^30 / 113 rounded up give exact quotients by 24-bit
// multiply-highs, which run at four times the rate of 32-bit ones.
constexpr int kSumBaseFewP = 227 * 9000, kSumBaseFewQ = 113 * 5000;
constexpr int kSumBaseP = 227 * 2256000, kSumBaseQ = 113 * 1270000;
template <bool FEW>
__device__ __forceinline__ uint32_t fp_from_based_sums(uint32_t sum_p, uint32_t sum_q) {
  auto hi24 = [](uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_mul_hi_u32_u24 %0, %1, %2" : "=v"(r) : "v"(a), "s"(b));
    return r;
  };
  uint32_t const p = mad24(FEW ? hi24(sum_p << 2, 4730141u) : __umulhi(sum_p, 605457945u) >> 5, -(int)FP_P, sum_p);
  uint32_t const y = sum_q - p;
  return mad24(mad24(FEW ? hi24(y << 2, 9502141u) : __umulhi(y, 1216273925u) >> 5, -(int)FP_Q, y), FP_P, p);
}

// A sum of residue products, |x| < 2^31, modulo 227: one signed multiply-high (605457945 =
// ceil(2^37 / 227) is exact below 2^31); of the quotient times 227, by a 24-bit multiply, the low byte is
// right.  A negative multiple of 227 leaves 227.
__device__ __forceinline__ uint32_t reduce_p(int x) {
  uint32_t const r = mad24(static_cast<uint32_t>(__mulhi(x, 605457945) >> 5), -(int)FP_P, static_cast<uint32_t>(x)) & 0xffu;
  return r < r - FP_P ? r : r - FP_P;
}
// 0 <= x < 2^31 modulo 113 (1216273925 = ceil(2^37 / 113)); the general mod_q takes a fix-up more
__device__ __forceinline__ uint32_t reduce_q(uint32_t x) {
  return mad24(__umulhi(x, 1216273925u) >> 5, -(int)FP_Q, x) & 0xffu;
}
// Fingerprint value of a matmul output from its two residue sums (matrix-core kernels): |sum_p| <
// 2^31 (operands recentred to [-113, 113]), 0 <= sum_q < 2^31 - 226.
__device__ __forceinline__ uint32_t fp_from_residue_sums(int sum_p, int sum_q) {
  uint32_t const p = reduce_p(sum_p);
  return mad24(reduce_q(static_cast<uint32_t>(sum_q) + 2 * FP_Q - p), FP_P, p);
}

// The fingerprint lookup tables in device memory and the ring operations built on them
// (kernel-level operators, and the operand prologue of the matrix-core matmul).
struct FpTables {
  uint16_t const *exp_tbl, *div_p, *div_q;
};

__device__ __forceinline__ uint32_t fp_exp_value(FpTables t, uint32_t x) {
  // reference element_unary_kernel.cu:85-89: an exponential's residue modulo 113 is zero
  return fp_from_residues(t.exp_tbl[residue_q(x)], 0u);
}

__device__ __forceinline__ uint32_t fp_div_value(FpTables t, uint32_t x, uint32_t y) {
  // reference element_binary_kernel.cu:155-160
  return fp_from_residues(residue_p(__umul24(residue_p(x), t.div_p[residue_p(y)])),
                          __umul24(residue_q(x), t.div_q[residue_q(y)]));
}

__device__ __forceinline__ uint32_t fp_silu_value(FpTables t, uint32_t x) {
  // extension: x / (1 + exp(-x)) from the ring primitives above
  uint32_t neg = mod_pq(FP_PQ - x);
  uint32_t den = mod_pq(1u + fp_exp_value(t, neg));
  return fp_div_value(t, x, den);
}

inline FpTables tables() {
  State &s = state();
  return FpTables{s.exp_tbl, s.div_p, s.div_q};
}

}  // namespace mi355
