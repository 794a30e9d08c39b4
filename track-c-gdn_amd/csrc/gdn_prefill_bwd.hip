// GDN chunked varlen prefill, backward (gfx950 / CDNA4, wave64, MFMA).
//
// The reference is forward-only (gdn_prefill_qk4_v8_d128_k_last/solution/
// triton/kernel.py:1); a training step needs the gradients of the prefill's
// inputs.  These kernels compute them from the states entering every chunk,
// h, which gdn_prefill_h_fwd writes (the h of the reference's
// chunk_gated_delta_rule_fwd_h, kernel.py:1153-1160).
//
// Per chunk (C = 64 rows, gam = chunk-local cumsum of the log-decay g,
// E = e^gam, Dc = e^{gam_L - gam}, S the state entering the chunk, dSn the
// gradient of the state leaving it) the forward is
//   Ar = tril_strict(e^{gam_i-gam_j} K K^T), A = diag(beta) Ar, Tm = (I + A)^-1,
//   P = scale tril_incl(e^{gam_i-gam_j} Q K^T), X = beta (V - E K S^T),
//   Vn = Tm X, O = scale E Q S^T + P Vn, S' = e^{gam_L} S + Vn^T Dc K,
// and its reverse is arranged in three launches:
//
//  1. gdn_bwd_prep_kernel, persistent workgroups over the (chunk, v-head)
//     units, all chunks at once: the state-gradient transition of the chunk,
//        M = e^{gam_L} I - W2^T (beta E K),   W2 = Tm^T Dc K            [K x K]
//        R = dO^T (scale E Q) - G1^T (beta E K),  G1 = Tm^T P^T dO      [V x K]
//     so that dS = dSn M + R.  M is written as ready MFMA A-operand
//     fragments, R in the accumulator layout of the chain kernel, and Tm for
//     the gradient kernel.
//  2. gdn_bwd_chain_kernel, one workgroup per (sequence, v-head), or
//     gdn_bwd_chain_few_kernel, one per eighth or quarter of its state rows
//     when the chains are few: walks the chunks
//     from last to first with dS^T in MFMA accumulators, storing dSn of
//     every chunk (bf16) and the gradient of the initial state.
//  3. gdn_bwd_grad_kernel, persistent workgroups over the (chunk, qk-head)
//     units, a unit's v-heads in turn: with S and dSn known, every gradient
//     of the chunk:
//        dVn = P^T dO + Dc K dSn^T,  dX = Tm^T dVn,  dV = beta dX,
//        dP = dO Vn^T,  dA = -dX Vn^T (strictly lower),
//        dQ = scale E dO S + dPm K,
//        dK = Dc Vn dSn - beta E dX S + dPm^T Q + (dAb + dAb^T) K,
//        dbeta = rowsum(dA Ar) + rowsum(dX (V - E K S^T)),
//        dgam  = rowsum - colsum of (dP P) and of (dA A) + scale E rowsum(Q (dO S))
//                - beta E rowsum(dX K S^T) - Dc rowsum(Vn K dSn^T)
//                (+ sum_i Dc rowsum(Vn K dSn^T) + e^{gam_L} <dSn, S> at gam_L),
//        dg = reverse cumsum of dgam within the chunk,
//     with dPm = scale e^{gam_i-gam_j} dP (j <= i), dAb = beta_i e^{gam_i-gam_j} dA.
//     (dA is the inverse's gradient -Tm^T (dVn X^T) Tm^T: its outer factors
//     turn dVn into dX and X into Vn, so neither dVn X^T nor the two 64^3
//     products around it are formed.)  dq / dk of the v-heads that share a
//     qk-head are summed in registers, in v-head order, and stored once.
//
// All products run on MFMA 16x16x32 bf16 with fp32 accumulation; the matrix
// operands live in LDS as bf16 rows of the form [m][r] and are read either
// straight (one 16-byte read: row m, reduction slots r) or through
// transposing LDS reads (ds_read_b64_tr_b16) when the product reduces over
// the other index.  Tm comes from an fp32 forward substitution.  Rows past a
// chunk's end are zero with beta = 0 and g = 0, which makes every one of
// their contributions vanish.  The waves of a workgroup exchange data only
// through LDS, so their barriers wait for LDS operations alone
// (lds_barrier): global loads and stores stay in flight across them.

#include "gdn_prefill_common.h"
#include "gdn_prefill_split.h"
#include "gdn_backward_step.h"
#include "../../include/gdn_hip.h"

#include <algorithm>

namespace {

using namespace gdn;

// [*][128] bf16 LDS rows of 272 B: the packed 8-byte writes of 16 tokens then
// hit distinct banks (288 B, which favours the 16-byte reads instead, made
// the gradient kernel 1% slower).
constexpr int LDK = D + 8;
constexpr int LDC = C + 8;           // [*][64] bf16 rows (144 B)
constexpr size_t kMBytes = size_t(D) * D * 2;   // M record (bf16 fragments)
constexpr size_t kRBytes = size_t(D) * D * 2;   // R record (bf16, accumulator layout); then dSn (bf16 [v][k])
constexpr size_t kTmBytes = size_t(C) * C * 2;  // Tm record (bf16 [t][t'], zero above the diagonal)
constexpr int kGradThreads = 512;

typedef short i16x8_t __attribute__((ext_vector_type(8)));

// MFMA 16x16x32 operand (lane l: row / column m0 + l % 16, reduction slots
// r0 + 8 (l / 16) .. +7) of a bf16 matrix stored [m][r] (r contiguous).
__device__ __forceinline__ bf16x8_t op_mr(const uint16_t* base, int ld, int m0, int r0, int lane) {
  return ld16_bf(base + (m0 + (lane & 15)) * ld + r0 + 8 * (lane >> 4));
}

// The same operand of a bf16 matrix stored [r][m] (m contiguous) in LDS: lane
// j of each 16-lane group reads 4 elements of row r0 + 8 q + j / 4 at column
// m0 + 4 (j % 4); the transposing read hands lane i the elements of column
// m0 + i of rows r0 + 8 q .. +3, the second read those of the next 4 rows.
__device__ __forceinline__ bf16x8_t op_rm(const uint16_t* base, int ld, int m0, int r0, int lane) {
  const int j = lane & 15;
  const uint16_t* p = base + (r0 + 8 * (lane >> 4) + (j >> 2)) * ld + m0 + 4 * (j & 3);
  const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)p);
  const i16x4_t hi =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(p + 4 * ld));
  const i16x8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8_t, v);
}

// op_rm with the reduction slots in the order of two stacked accumulator
// tiles: slot e of lane group q is row r0 + 16 (e / 4) + 4 q + e % 4.
__device__ __forceinline__ bf16x8_t op_rmp(const uint16_t* base, int ld, int m0, int r0, int lane) {
  const int j = lane & 15;
  const uint16_t* p = base + (r0 + 4 * (lane >> 4) + (j >> 2)) * ld + m0 + 4 * (j & 3);
  const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)p);
  const i16x4_t hi =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(p + 16 * ld));
  const i16x8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8_t, v);
}

// An operand's 8 values times f0 (slots 0-3) and f1 (slots 4-7), rounded back to bf16.
__device__ __forceinline__ bf16x8_t scale_bf8(bf16x8_t x, const f32x4& f0, const f32x4& f1) {
  f32x4 lo, hi;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    lo[e] = f0[e] * float(x[e]);
    hi[e] = f1[e] * float(x[4 + e]);
  }
  return pack2_bf(lo, hi);
}

// 4 adjacent bf16 values as floats, and back (round to nearest even).
__device__ __forceinline__ f32x4 bf4_f32(const uint2& w) {
  float x0, x1, x2, x3;
  unpack_bf16x2(w.x, x0, x1);
  unpack_bf16x2(w.y, x2, x3);
  return f32x4{x0, x1, x2, x3};
}

__device__ __forceinline__ void st_bf4(uint16_t* p, const f32x4& x) {
  *reinterpret_cast<uint2*>(p) = uint2{cvt_pk_bf16(x[0], x[1]), cvt_pk_bf16(x[2], x[3])};
}

// Sum over the 4 lane groups (same lane % 16) of a wave, in every lane: a
// permlane swap of a value with itself leaves one half's values in all lanes
// of one result and the other half's in the other.
__device__ __forceinline__ float group4_sum(float x) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Three such sums with half the exchanges: x's in lane group 0, y's in group 1
// (and 3), z's in group 2, each added in group4_sum's order.
__device__ __forceinline__ float group4_sum3(float x, float y, float z) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(z), false, false);
  const float xz = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  const auto i = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  const float yy = __uint_as_float(i[0]) + __uint_as_float(i[1]);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(xz), __float_as_uint(yy), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Gate data of one chunk in LDS: gam | beta | e^gam | e^{gam_L - gam} (64 each),
// then gam_L, e^{gam_L}.  One wave's work (wave 3 of the preparation, wave 1
// of the gradients): lane t takes token t of the chunk.
constexpr int GB_GAM = 0, GB_BETA = C, GB_E = 2 * C, GB_DC = 3 * C, GB_L = 4 * C, GB_EL = 4 * C + 1;
constexpr int GB_SZ = 4 * C + 4;
constexpr int GB_DA = GB_SZ, GB_DB = GB_SZ + C, GB_G = GB_SZ + 2 * C;   // GateFactors (training step only)

// The gate inputs of token `lane` of the chunk: loaded early, used
// by chunk_gates_calc once the chunk's rows are on their way.
struct GateIn {
  uint16_t a, b;       // as loaded: converted where they are used, so that nothing waits for them before
  float dt, alog;
};

__device__ __forceinline__ GateIn gate_inputs(const float* A_log, const uint16_t* a, const float* dt_bias,
                                              const uint16_t* b, int HV, int hv, int t0, int len, int lane) {
  const size_t i = size_t(t0 + min(lane, len - 1)) * HV + hv;
  return GateIn{a[i], b[i], dt_bias[hv], A_log[hv]};
}

// g = -exp(A_log) softplus(a + dt_bias), beta = sigmoid(b) per token (zero
// past the chunk end), the chunk-local cumsum gam, e^gam and e^{gam_L - gam},
// with the forward kernels' hardware exp2 / log2 forms.
__device__ __forceinline__ void chunk_gates_calc(const GateIn& in, int len, int lane, float* gb) {
  constexpr float kLog2e = 1.44269504088896341f, kLn2 = 0.69314718055994531f;
  float g = 0.f, be = 0.f;
  if (lane < len) {
    const float x = bf16_bits_to_f32(in.a) + in.dt;
    const float sp = fmaxf(x, 0.f) + kLn2 * __builtin_amdgcn_logf(1.f + __builtin_amdgcn_exp2f(-fabsf(x) * kLog2e));
    g = -__builtin_amdgcn_exp2f(in.alog * kLog2e) * sp;
    be = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-bf16_bits_to_f32(in.b) * kLog2e));
  }
  const float gam = wave_inclusive_scan(g);
  const float gl = __shfl(gam, 63);
  gb[GB_GAM + lane] = gam;
  gb[GB_BETA + lane] = be;
  gb[GB_E + lane] = __builtin_amdgcn_exp2f(gam * kLog2e);
  gb[GB_DC + lane] = __builtin_amdgcn_exp2f((gl - gam) * kLog2e);
  if (lane == 0) {
    gb[GB_L] = gl;
    gb[GB_EL] = __builtin_amdgcn_exp2f(gl * kLog2e);
  }
}

// One chunk's rows of one head of a [T, heads, 128] tensor, as a buffer from
// token t0's row: byte offset (t * heads * 128 + column) * sizeof(T) of token
// t0 + t.  Rows at or past len fall outside it (a load gives zeros, a store
// writes nothing), so the accesses need no branch and every path through a
// loop issues the same memory instructions: with branches around them the
// compiler's waits for the next step's loads also waited for stores issued
// after them.
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t head_rows(T* base, int heads, int head, int t0, int len) {
  return uniform_buffer(base + (size_t(t0) * heads + head) * D,
                        len > 0 ? uint32_t((len * heads - head) * D * int(sizeof(T))) : 0u);
}

__device__ __forceinline__ uint4 buffer_load_b128(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, int(off), 0, 0));
}
__device__ __forceinline__ uint2 buffer_load_b64(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, int(off), 0, 0));
}

// A chunk's 64 rows into a [64][LDK] LDS buffer, rows past the chunk zero, in
// two steps so that the HBM reads of several tensors are in flight together:
// rows_fetch issues this thread's 16-byte reads (of the 1024 of a tensor),
// rows_store writes them.
template <int kThreads>
__device__ __forceinline__ void rows_fetch(uint4 (&w)[1024 / kThreads], __amdgpu_buffer_rsrc_t src, int heads,
                                           int tid) {
#pragma unroll
  for (int it = 0; it < 1024 / kThreads; ++it) {
    const int x = tid + it * kThreads;
    w[it] = buffer_load_b128(src, uint32_t((x >> 4) * heads * D + (x & 15) * 8) * 2u);
  }
}

template <int kThreads>
__device__ __forceinline__ void rows_store(uint16_t* dst, const uint4 (&w)[1024 / kThreads], int tid) {
#pragma unroll
  for (int it = 0; it < 1024 / kThreads; ++it) {
    const int x = tid + it * kThreads, r = x >> 4, cc = (x & 15) * 8;
    *reinterpret_cast<uint4*>(dst + r * LDK + cc) = w[it];
  }
}

// ---------------------------------------------------------------------------
// 1. Transition of the state gradient per (chunk, v-head): M, R and Tm.
//
// M record: 32 fragments of 1 KB, fragment (kt, s) = kt * 4 + s holds for
// lane l the 8 bf16 of M^T[16 kt + l % 16][j] at j = 32 s + 16 (e / 4) +
// 4 (l / 16) + e % 4, e = 0..7: the A operand of the chain kernel's product
// dS^T M-side, whose B operand is two stacked accumulator tiles of dS^T.
// R record: R^T tiles in pairs (kt, kt + 1) of a row block vt, vt-major,
// lane l's 2 x 4 values (bf16, 16 bytes) at 16 l: rows 16 kt + 4 (l / 16) + i,
// column 16 vt + l % 16 -- the chain kernel's accumulator layout.  bf16 like
// M and like the dSn operand the chain multiplies by M: R enters dS = dSn M +
// R with the same rounding.
//
// Bound by HBM at 32 768 tokens qk16/v32: 0.35 ms for the 1.75 GB it must move
// (1.82 GB by the counters, 5.2 TB/s).  It replaces a form that took 0.95 ms:
// one workgroup of 8 waves per CU (160 KB of LDS, scaled copies of K and Q
// among it) whose other waves waited for one wave's inverse of the whole block.
// Workgroups of 4 waves, two per CU (78 KB of LDS each), so that one's serial
// inverse overlaps the other's products and stores:
//   P1  the lower 16x16 tiles of A (fp32) and P; wave w inverts A's diagonal
//       tile w by forward substitution
//   P2  wave j: the blocks below the diagonal of block column j of
//       Tm = (I + A)^-1, T_ij = -T_ii sum_m A_im T_mj, on fp32 MFMA (a block
//       column needs no other); every wave: G0 = P^T dO for its 32 columns
//   P3  W2, G1, M and R for the wave's 32 columns, operands from the wave's
//       own accumulators and transposing reads of K and Q as loaded: the row
//       factors beta E, scale E and Dc are applied to the other operand, in
//       fp32 where that is an accumulator
// All reductions over tokens take them in the order of stacked accumulator
// tiles (op_rmp).
constexpr int kPrepThreads = 256;

// Forward substitution of one unit lower triangular 16 x 16 block I + A
// (A fp32 [16][16] in LDS, strictly lower), lane l taking column l % 16:
// x_r = delta_rc - sum_{m<r} A_rm x_m, column by column.
__device__ __forceinline__ void unit_lower_inverse16(const float* sA, int c, float (&x)[16]) {
#pragma unroll
  for (int r = 0; r < 16; ++r) x[r] = r == c ? 1.f : 0.f;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    f32x4 a[16];
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (r > 4 * mb) a[r] = *reinterpret_cast<const f32x4*>(sA + 16 * r + 4 * mb);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (r > 4 * mb + e) x[r] = fmaf(-a[r][e], x[4 * mb + e], x[r]);
  }
}

template <typename CuT>
__global__ __launch_bounds__(kPrepThreads, 2) void gdn_bwd_prep_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const float* __restrict__ A_log,
    const uint16_t* __restrict__ a, const float* __restrict__ dt_bias, const uint16_t* __restrict__ b,
    const CuT* __restrict__ cu, int N, int T, int HQ, int HV, float scale,
    const uint16_t* __restrict__ d_out, int h_chunks, int slots, int heads, char* __restrict__ mrec,
    char* __restrict__ rrec, uint16_t* __restrict__ tmrec, int2* __restrict__ chunks) {
  __shared__ __align__(16) uint16_t sK[C * LDK];
  __shared__ __align__(16) uint16_t sQ[C * LDK];
  __shared__ __align__(16) uint16_t sdO[C * LDK];     // dO; then Tm ([64][LDC])
  __shared__ __align__(16) uint16_t sP[C * LDC];
  __shared__ __align__(16) float sA[10][16 * 16];     // lower tiles of A, row by row
  __shared__ __align__(16) float sD[4][16 * 16];      // the inverses of the diagonal tiles
  __shared__ __align__(16) float gbuf[2][GB_SZ];
  __shared__ int4 next_unit[2];
  uint16_t* sTm = sdO;

  const int tid0 = threadIdx.x, lane0 = tid0 & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6);
  // Persistent workgroups walk the units -- a chunk slot and `heads` v-heads
  // of one qk-head, v-heads fastest -- and a unit's v-heads in turn.  The next
  // step's rows and gate inputs are loaded into registers while this one is
  // worked on; wave 3 looks up the unit after the next.
  const int groups = HV / heads, units = slots * groups;
  struct At {
    int unit, m, t0, len;
  };
  // the first unit at or after `unit` (in this workgroup's stride) that holds
  // a chunk (unit >= units: none); wave 3 notes the token range of every slot
  // it passes for the gradient kernel (length 0: no chunk)
  auto seek = [&](int unit) {
    At x{unit, 0, 0, 0};
    for (; x.unit < units; x.unit += int(gridDim.x)) {
      const int slot = x.unit / groups;
      x.len = 0;
      if (slot < h_chunks) {
        int n, ci;
        locate_chunk(cu, N, T, slot, lane0, n, ci);
        if (n >= 0) {
          int bos, slen;
          seq_bounds(cu, n, T, bos, slen);
          x.t0 = __builtin_amdgcn_readfirstlane(bos + C * ci);
          x.len = __builtin_amdgcn_readfirstlane(min(C, slen - C * ci));
        }
      }
      if (wave == 3 && lane0 == 0 && x.unit == slot * groups) chunks[slot] = int2{x.t0, x.len};
      if (x.len > 0) break;
    }
    return x;
  };
  auto head_of = [&](const At& x) { return (x.unit % groups) * heads + x.m; };
  struct Regs {
    uint4 k[4], q[4], o[4];
  };
  auto fetch = [&](const At& x, Regs& r, int tid) {
    const int hv = head_of(x), hq = hv / (HV / HQ);
    if (x.m == 0) {
      rows_fetch<kPrepThreads>(r.k, head_rows(k, HQ, hq, x.t0, x.len), HQ, tid);
      rows_fetch<kPrepThreads>(r.q, head_rows(q, HQ, hq, x.t0, x.len), HQ, tid);
    }
    rows_fetch<kPrepThreads>(r.o, head_rows(d_out, HV, hv, x.t0, x.len), HV, tid);
  };
  auto gate_in = [&](const At& x, int lane) {
    return gate_inputs(A_log, a, dt_bias, b, HV, head_of(x), x.t0, x.len, lane);
  };

  // the tiles of sP above the diagonal that an operand read covers stay zero
  for (int x = tid0; x < 2 * 16 * 16; x += kPrepThreads) {
    const int up = x >> 8, r = (x >> 4) & 15, c = x & 15;
    sP[(32 * up + r) * LDC + 32 * up + 16 + c] = 0;
  }

  At at = seek(int(blockIdx.x));
  if (at.unit >= units) return;
  At after = seek(at.unit + int(gridDim.x));      // the unit after at's
  Regs cur;
  fetch(at, cur, tid0);
  if (wave == 3) chunk_gates_calc(gate_in(at, lane0), at.len, lane0, gbuf[0]);
  // This wave's tiles (ti, tj) of A and P: diagonal tile `wave` and one or two
  // below the diagonal; their Q K^T and K K^T, transposed (rows s = 16 tj +
  // 4 g + i, column t = 16 ti + c), serve all v-heads of the unit.
  const int ti1 = wave == 0 ? 1 : wave == 3 ? 3 : 2, tj1 = wave < 2 ? 0 : 1;
  const int ti2 = 3, tj2 = wave == 2 ? 0 : 2;
  const bool three = wave >= 2;
  f32x4 qk[3], kk[3];
  for (int it = 0, un = 0; at.unit < units; ++it) {
    // Lane indices opaque to the compiler at the top of each phase: their
    // address arithmetic is formed where it is used instead of being kept in
    // registers across phases and steps.
    int tid = tid0, lane = lane0, g, c;
    auto fresh_lane = [&] {
      asm volatile("" : "+v"(lane), "+v"(tid));
      g = lane >> 4;
      c = lane & 15;
    };
    fresh_lane();
    const int slot = at.unit / groups, hv = head_of(at), m = at.m;
    const float* gb = gbuf[it & 1];
    const size_t rec = size_t(slot) * HV + hv;
    if (m == 0) {
      rows_store<kPrepThreads>(sK, cur.k, tid);
      rows_store<kPrepThreads>(sQ, cur.q, tid);
    }
    rows_store<kPrepThreads>(sdO, cur.o, tid);
    lds_barrier();

    // P1: the tiles; dO as operands of this wave's columns v = 32 wave + 16 u + c
    bf16x8_t dof[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int u = 0; u < 2; ++u) dof[s][u] = op_rmp(sdO, LDK, 32 * wave + 16 * u, 32 * s, lane);
    auto tiles = [&](auto count) {
#pragma unroll
      for (int j = 0; j < decltype(count)::value; ++j) {
        const int ti = j == 0 ? wave : j == 1 ? ti1 : ti2, tj = j == 0 ? wave : j == 1 ? tj1 : tj2;
        if (m == 0) {
          f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            const bf16x8_t ka = op_mr(sK, LDK, 16 * tj, 32 * s, lane);
            x = mfma16_bf(ka, op_mr(sQ, LDK, 16 * ti, 32 * s, lane), x);
            y = mfma16_bf(ka, op_mr(sK, LDK, 16 * ti, 32 * s, lane), y);
          }
          qk[j] = x;
          kk[j] = y;
        }
        const int t = 16 * ti + c, s0 = 16 * tj + 4 * g;
        const float gt = gb[GB_GAM + t], be = gb[GB_BETA + t];
        const f32x4 gs = *reinterpret_cast<const f32x4*>(&gb[GB_GAM + s0]);
        f32x4 pv, av;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float ex = t >= s0 + i ? exp_fast(gt - gs[i]) : 0.f;
          pv[i] = scale * (ex * qk[j][i]);
          av[i] = t > s0 + i ? be * (ex * kk[j][i]) : 0.f;
        }
        st_bf4(sP + t * LDC + s0, pv);
        *reinterpret_cast<f32x4*>(&sA[(ti * (ti + 1)) / 2 + tj][16 * c + 4 * g]) = av;
      }
    };
    if (three) tiles(IC<3>());
    else tiles(IC<2>());
    {
      // a wave's LDS operations complete in order: its own tile needs no barrier
      float x[16];
      unit_lower_inverse16(sA[(wave * (wave + 1)) / 2 + wave], c, x);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sD[wave][16 * (4 * g + i) + c] = g == 0 ? x[i] : g == 1 ? x[4 + i] : g == 2 ? x[8 + i] : x[12 + i];
    }
    At nx = at;
    ++nx.m;
    if (nx.m == heads) nx = after;
    const bool more = nx.unit < units;
    GateIn gin{};
    if (wave == 3 && more) gin = gate_in(nx, lane);
    lds_barrier();

    // P2: Tm; G0 = P^T dO
    fresh_lane();
    Regs nxt;
    fetch(more ? nx : at, nxt, tid);
    bf16x8_t g0[2][2];
    {
      f32x4 acc[4][2];
#pragma unroll
      for (int tb = 0; tb < 4; ++tb) {
        acc[tb][0] = acc[tb][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = tb / 2; s < 2; ++s) {
          const bf16x8_t po = op_rmp(sP, LDC, 16 * tb, 32 * s, lane);
#pragma unroll
          for (int u = 0; u < 2; ++u) acc[tb][u] = mfma16_bf(po, dof[s][u], acc[tb][u]);
        }
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int u = 0; u < 2; ++u) g0[s][u] = pack2_bf(acc[2 * s][u], acc[2 * s + 1][u]);
    }
    auto st_tm = [&](int ti, int tj, const f32x4& x) {
      uint16_t* p = sTm + (16 * ti + 4 * g) * LDC + 16 * tj + c;
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i * LDC] = f32_to_bf16_bits(x[i]);
    };
    auto column = [&](auto col) {
      constexpr int j = decltype(col)::value;
      f32x4 x[4 - j];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[0][e] = sD[j][16 * (4 * g + e) + c];
      st_tm(j, j, x[0]);
#pragma unroll
      for (int i = j + 1; i < 4; ++i) {
        f32x4 z = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int mm = j; mm < i; ++mm) {
          const f32x4 av = *reinterpret_cast<const f32x4*>(&sA[(i * (i + 1)) / 2 + mm][16 * c + 4 * g]);
#pragma unroll
          for (int e = 0; e < 4; ++e) z = __builtin_amdgcn_mfma_f32_16x16x4f32(av[e], x[mm - j][e], z, 0, 0, 0);
        }
        const f32x4 dv = *reinterpret_cast<const f32x4*>(&sD[i][16 * c + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) y = __builtin_amdgcn_mfma_f32_16x16x4f32(dv[e], z[e], y, 0, 0, 0);
        x[i - j] = -y;
        st_tm(i, j, x[i - j]);
      }
    };
    if (wave == 0) column(IC<0>());
    else if (wave == 1) column(IC<1>());
    else if (wave == 2) column(IC<2>());
    else {
      column(IC<3>());
#pragma unroll
      for (int x = 0; x < 6; ++x) {           // zero above the diagonal
        const int ti = x < 3 ? 0 : x < 5 ? 1 : 2, tj = x < 3 ? x + 1 : x < 5 ? x - 1 : 3;
        *reinterpret_cast<uint2*>(sTm + (16 * ti + c) * LDC + 16 * tj + 4 * g) = uint2{0, 0};
      }
      if (more) chunk_gates_calc(gin, nx.len, lane, gbuf[(it + 1) & 1]);
      if (m == 0 && after.unit < units) {
        const At x = seek(after.unit + int(gridDim.x));
        if (lane == 0) next_unit[un & 1] = int4{x.unit, x.t0, x.len, 0};
      }
    }
    lds_barrier();

    // P3
    fresh_lane();
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int y = tid + x * kPrepThreads;
      reinterpret_cast<uint4*>(tmrec + rec * C * C)[y] =
          *reinterpret_cast<const uint4*>(sTm + (y >> 3) * LDC + 8 * (y & 7));
    }
    bf16x8_t w2[2][2], g1[2][2];
    {
      // W2 = Tm^T Dc K and G1 = Tm^T G0, then times -beta E
      f32x4 wa[4][2], ga[4][2];
      bf16x8_t dk[2][2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const f32x4 d0 = *reinterpret_cast<const f32x4*>(&gb[GB_DC + 32 * s + 4 * g]);
        const f32x4 d1 = *reinterpret_cast<const f32x4*>(&gb[GB_DC + 32 * s + 16 + 4 * g]);
        const f32x4 e0 = *reinterpret_cast<const f32x4*>(&gb[GB_E + 32 * s + 4 * g]);
        const f32x4 e1 = *reinterpret_cast<const f32x4*>(&gb[GB_E + 32 * s + 16 + 4 * g]);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          dk[s][u] = scale_bf8(op_rmp(sK, LDK, 32 * wave + 16 * u, 32 * s, lane), d0, d1);
          dof[s][u] = scale_bf8(dof[s][u], scale * e0, scale * e1);
        }
      }
#pragma unroll
      for (int tb = 0; tb < 4; ++tb) {
#pragma unroll
        for (int u = 0; u < 2; ++u) wa[tb][u] = ga[tb][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = tb / 2; s < 2; ++s) {
          const bf16x8_t tm = op_rmp(sTm, LDC, 16 * tb, 32 * s, lane);
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            wa[tb][u] = mfma16_bf(tm, dk[s][u], wa[tb][u]);
            ga[tb][u] = mfma16_bf(tm, g0[s][u], ga[tb][u]);
          }
        }
        const f32x4 be = *reinterpret_cast<const f32x4*>(&gb[GB_BETA + 16 * tb + 4 * g]);
        const f32x4 e = *reinterpret_cast<const f32x4*>(&gb[GB_E + 16 * tb + 4 * g]);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            wa[tb][u][i] *= -be[i] * e[i];
            ga[tb][u][i] *= -be[i] * e[i];
          }
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          w2[s][u] = pack2_bf(wa[2 * s][u], wa[2 * s + 1][u]);
          g1[s][u] = pack2_bf(ga[2 * s][u], ga[2 * s + 1][u]);
        }
    }
    // M = e^{gam_L} I - W2^T beta E K: rows j = 32 wave + 16 u + 4 g + i, column 16 kt + c.
    // R^T = K^T (-beta E G1) + Q^T (scale E dO): rows 16 kt + 4 g + i, column v.
    const float eL = gb[GB_EL];
    char* mr = mrec + rec * kMBytes + wave * 1024 + lane * 16;
    char* rr = rrec + rec * kRBytes + (8 * wave) * 1024 + lane * 16;
#pragma unroll
    for (int kp = 0; kp < 4; ++kp) {
      uint2 rw[2][2];
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        const int kt = 2 * kp + o;
        bf16x8_t kf[2], qf[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          kf[s] = op_rmp(sK, LDK, 16 * kt, 32 * s, lane);
          qf[s] = op_rmp(sQ, LDK, 16 * kt, 32 * s, lane);
        }
        uint2 mw[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f32x4 ma, ra = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < 4; ++i) ma[i] = kp == wave && o == u && 4 * g + i == c ? eL : 0.f;
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            ma = mfma16_bf(w2[s][u], kf[s], ma);
            ra = mfma16_bf(kf[s], g1[s][u], ra);
            ra = mfma16_bf(qf[s], dof[s][u], ra);
          }
          mw[u] = uint2{cvt_pk_bf16(ma[0], ma[1]), cvt_pk_bf16(ma[2], ma[3])};
          rw[u][o] = uint2{cvt_pk_bf16(ra[0], ra[1]), cvt_pk_bf16(ra[2], ra[3])};
        }
        *reinterpret_cast<uint4*>(mr + kt * 4096) = uint4{mw[0].x, mw[0].y, mw[1].x, mw[1].y};
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
        *reinterpret_cast<uint4*>(rr + (4 * u + kp) * 1024) =
            uint4{rw[u][0].x, rw[u][0].y, rw[u][1].x, rw[u][1].y};
    }
    if (more && nx.m == 0) {
      const int4 x = next_unit[un & 1];
      after = At{__builtin_amdgcn_readfirstlane(x.x), 0, __builtin_amdgcn_readfirstlane(x.y),
                 __builtin_amdgcn_readfirstlane(x.z)};
      ++un;
    }
    // the next step overwrites what this one reads last
    lds_barrier();
    cur = nxt;
    at = nx;
  }
}

// ---------------------------------------------------------------------------
// 2. The state-gradient chain per (sequence, v-head), last chunk first:
//    dS = dSn M + R, dSn (bf16 [v][k]) over the chunk's R record;  finally dh0 = dS.
// A wave keeps dS^T[k][v] for 16 state rows v as 8 accumulator tiles (k
// blocks); the B operand of step s is the pair of tiles kt = 2 s, 2 s + 1.
// The rows of dS evolve independently (dS = dSn M + R row by row).  The 16
// rows of dSn that a wave writes are the bytes of the R block that only it
// reads, and it has them in registers by then.
struct ChainLane {
  int vb;              // 16-row block of the state this wave holds
  int g, c, lane;
  size_t state;        // element offset of this lane's state row in a [N, HV, 128, 128] tensor
  uint32_t line;       // byte offset of this lane's pieces in whole-line stores of a 16-row tile
};

__device__ __forceinline__ ChainLane chain_lane(int vb, int n, int HV, int hv, int lane) {
  const int g = lane >> 4, c = lane & 15;
  return ChainLane{vb, g, c, lane, ((size_t(n) * HV + hv) * D + 16 * vb + c) * D, state_lines_lane(g, c)};
}

__device__ __forceinline__ void chain_load(f32x4 (&acc)[8], const float* d_ht, const ChainLane& w) {
#pragma unroll
  for (int kt = 0; kt < 8; ++kt)
    acc[kt] = d_ht ? *reinterpret_cast<const f32x4*>(d_ht + w.state + 16 * kt + 4 * w.g)
                   : f32x4{0.f, 0.f, 0.f, 0.f};
}

__device__ __forceinline__ void chain_fetch_r(uint4 (&r)[4], const char* rec, const ChainLane& w) {
#pragma unroll
  for (int kp = 0; kp < 4; ++kp)
    r[kp] = *reinterpret_cast<const uint4*>(rec + ((w.vb * 4 + kp) * 64 + w.lane) * 16);
}

// dSn as the B operand of the product.
__device__ __forceinline__ void chain_pack(bf16x8_t (&bop)[4], const f32x4 (&acc)[8]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) bop[s] = pack2_bf(acc[2 * s], acc[2 * s + 1]);
}

// dSn to its record as whole 128-byte lines.
__device__ __forceinline__ void chain_put(const bf16x8_t (&bop)[4], char* rec, const ChainLane& w) {
#pragma unroll
  for (int pp = 0; pp < 2; ++pp) {
    u32x4_t d1, d2;
    state_lines(w.c, bop[2 * pp], bop[2 * pp + 1], d1, d2);
    char* p = rec + w.vb * 4096 + 128 * pp + w.line;
    *reinterpret_cast<u32x4_t*>(p) = d1;
    *reinterpret_cast<u32x4_t*>(p + 8 * D * 2) = d2;
  }
}

__device__ __forceinline__ f32x4 chain_r_tile(const uint4 (&r)[4], int kt) {
  return bf4_f32((kt & 1) ? uint2{r[kt / 2].z, r[kt / 2].w} : uint2{r[kt / 2].x, r[kt / 2].y});
}

__device__ __forceinline__ void chain_store(float* dh0, const f32x4 (&acc)[8], const ChainLane& w) {
  if (dh0) {
#pragma unroll
    for (int kt = 0; kt < 8; ++kt)
      *reinterpret_cast<f32x4*>(dh0 + w.state + 16 * kt + 4 * w.g) = acc[kt];
  }
}

// One workgroup of 8 waves per chain: M through LDS, copied (and R loaded into
// registers) two chunks ahead by the waves themselves.  Bound by HBM while
// the chains fill the chip: 96 KB per chunk and chain (32 768 tokens qk16/v32:
// 328 us; 376 us with dSn stored in 8-byte pieces of half lines).
template <typename CuT>
__global__ __launch_bounds__(512, 1) void gdn_bwd_chain_kernel(
    const CuT* __restrict__ cu, int N, int T, int HV, int h_chunks, const char* __restrict__ mrec,
    char* rrec, const float* __restrict__ d_ht, float* __restrict__ dh0) {
  constexpr int kThreads = 512;
  __shared__ __align__(16) uint16_t sM[3][D * D];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = int(blockIdx.x) / HV, hv = int(blockIdx.x) - n * HV;
  int bos, slen;
  seq_bounds(cu, n, T, bos, slen);
  const int nc = (slen + C - 1) / C;
  const int coff = chunk_offset(cu, n, T, lane);
  const ChainLane w = chain_lane(wave, n, HV, hv, lane);
  f32x4 acc[8];
  chain_load(acc, d_ht, w);
  int last = nc - 1;
  if (coff + last >= h_chunks) last = -1;     // records at or past h_chunks (clamped to the workspace's slots) were not formed
  // three LDS buffers for M and three register sets for R, rotated by
  // unrolling the chunk loop by three
  constexpr int kMCopies = int(kMBytes / 16) / kThreads;
  auto rec_of = [&](int ch) { return size_t(coff + ch) * HV + hv; };
  auto copy_m = [&](int ch, int buf) {
    const char* ms = mrec + rec_of(ch) * kMBytes;
#pragma unroll
    for (int x = 0; x < kMCopies; ++x)
      lds_dma16_saddr(ms, uint32_t((x * kThreads + tid) * 16), &sM[buf][(x * kThreads + wave * 64) * 8]);
  };
  auto fetch_r = [&](int ch, uint4 (&r)[4]) { chain_fetch_r(r, rrec + rec_of(ch) * kRBytes, w); };
  // one chunk: dSn out, dS = dSn M + R (cur = R of chunk ch), and the copies
  // for chunk ch - 2 (R into nxt2, M into LDS buffer (it + 2) % 3)
  auto step = [&](int ch, int it, uint4 (&cur)[4], uint4 (&nxt2)[4]) {
    const int buf = it % 3;
    if (ch > 1) {
      copy_m(ch - 2, (it + 2) % 3);
      fetch_r(ch - 2, nxt2);
    }
    bf16x8_t bop[4];
    chain_pack(bop, acc);
    chain_put(bop, rrec + rec_of(ch) * kRBytes, w);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
      acc[kt] = chain_r_tile(cur, kt);
#pragma unroll
      for (int s = 0; s < 4; ++s)
        acc[kt] = mfma16_bf(ld16_bf(&sM[buf][((kt * 4 + s) * 64 + lane) * 8]), bop[s], acc[kt]);
    }
    // Vector memory operations complete in issue order: with at most this
    // chunk's copies (M and R two chunks ahead) and its 4 dSn stores still
    // outstanding, everything the next chunk reads has landed.
    if (ch > 1) wait_vm<kMCopies + 4 + 4>();
    else wait_vm<4>();
    lds_barrier();
  };
  uint4 r0[4], r1[4], r2[4];
  if (last >= 0) {
    copy_m(last, 0);
    fetch_r(last, r0);
    if (last > 0) {
      copy_m(last - 1, 1);
      fetch_r(last - 1, r1);
    }
  }
  wait_vm<0>();
  lds_barrier();
  for (int ch = last, it = 0; ch >= 0; ch -= 3, it += 3) {
    step(ch, it, r0, r2);
    if (ch >= 1) step(ch - 1, it + 1, r1, r0);
    if (ch >= 2) step(ch - 2, it + 2, r2, r1);
  }
  chain_store(dh0, acc, w);
}

// When the chains leave most CUs idle: 8 / NR workgroups per chain, NR waves
// of 16 state rows in each, and the latency of one chunk's step is what
// counts.  kCopyWaves more waves copy M into a ring of four LDS buffers, up to four
// chunks ahead, and store dSn, which the row waves leave in LDS.  A row wave
// has the chunk's M operands in registers before the chunk begins: behind the
// products of each half of the k blocks it reads the next chunk's operands,
// so its step is 32 products with the reads under them.  4096 tokens qk4/v8
// (64 chunks, 8 chains), us per launch: 86 with the kernel above cut to two
// waves (16 copies, 32 reads, 8 stores and 32 products in a row); 51 with copy
// waves and the row waves' own whole-line stores (56 with 8-byte pieces).
constexpr int kRing = 4, kCopyWaves = 2;

template <typename CuT, int NR>
__global__ __launch_bounds__(64 * (NR + kCopyWaves), 1) void gdn_bwd_chain_few_kernel(
    const CuT* __restrict__ cu, int N, int T, int HV, int h_chunks, const char* __restrict__ mrec,
    char* rrec, const float* __restrict__ d_ht, float* __restrict__ dh0) {
  constexpr int kSlices = 8 / NR;
  __shared__ __align__(16) uint16_t sM[kRing][D * D];
  __shared__ __align__(16) uint16_t sOut[2][16 * NR * LDK];   // dSn of the even and odd steps
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroup -> (chain = (sequence, v-head), slice of 16 NR state rows): a
  // chain's slices get ids 8 apart, which puts them on one XCD, so M is read
  // from HBM once per chain.
  const int xcd = blockIdx.x & 7, id_row = blockIdx.x >> 3;
  const int chain = 8 * (id_row / kSlices) + xcd, slice = id_row % kSlices;
  if (chain >= N * HV) return;
  const int n = chain / HV, hv = chain - n * HV;
  int bos, slen;
  seq_bounds(cu, n, T, bos, slen);
  const int nc = (slen + C - 1) / C;
  const int coff = chunk_offset(cu, n, T, lane);
  int last = nc - 1;
  if (coff + last >= h_chunks) last = -1;     // as above
  auto rec_of = [&](int ch) { return size_t(coff + ch) * HV + hv; };
  if (wave >= NR) {
    constexpr int kCopies = int(kMBytes / 1024) / kCopyWaves, kStores = 4 * NR / kCopyWaves;
    const int part = wave - NR;               // of M and of dSn
    auto copy_m = [&](int ch, int buf) {
      const char* ms = mrec + rec_of(ch) * kMBytes + part * (kCopies * 1024);
#pragma unroll
      for (int x = 0; x < kCopies; ++x)
        lds_dma16_saddr(ms, uint32_t(x * 1024 + lane * 16), &sM[buf][(part * kCopies + x) * 512]);
    };
    auto store_out = [&](int ch, int parity) {
      char* out = rrec + rec_of(ch) * kRBytes + slice * NR * 4096;
#pragma unroll
      for (int x = 0; x < kStores; ++x) {
        const int at = (part * kStores + x) * 64 + lane;        // 16-byte piece of the rows
        *reinterpret_cast<uint4*>(out + at * 16) =
            *reinterpret_cast<const uint4*>(&sOut[parity][(at >> 4) * LDK + (at & 15) * 8]);
      }
    };
#pragma unroll
    for (int x = 0; x < kRing; ++x)
      if (last - x >= 0) copy_m(last - x, x);
    wait_vm<0>();
    lds_barrier();                            // A: the first four chunks have landed
    lds_barrier();                            // B: chunk `last` is in registers
    for (int ch = last, it = 0; ch >= 0; --ch, ++it) {
      // chunk ch - 4 over chunk ch, and the step before's dSn to its record;
      // chunk ch - 2 has landed when the step ends (operations complete in
      // issue order: behind its copies come at most those of two more chunks
      // and the stores of two steps)
      if (ch >= 4) copy_m(ch - 4, it & 3);
      if (it > 0) store_out(ch + 1, (it - 1) & 1);
      if (ch >= 4) wait_vm<2 * (kCopies + kStores)>();
      else wait_vm<0>();
      lds_barrier();
    }
    if (last >= 0) store_out(0, last & 1);
    return;
  }
  const ChainLane w = chain_lane(NR * slice + wave, n, HV, hv, lane);
  f32x4 acc[8];
  chain_load(acc, d_ht, w);
  bf16x8_t m[8][4];
  uint4 r[kRing][4];
#pragma unroll
  for (int x = 0; x < kRing - 1; ++x)
    if (last - x >= 0) chain_fetch_r(r[x], rrec + rec_of(last - x) * kRBytes, w);
  lds_barrier();                              // A
#pragma unroll
  for (int kt = 0; kt < 8; ++kt)
#pragma unroll
    for (int s = 0; s < 4; ++s) m[kt][s] = ld16_bf(&sM[0][((kt * 4 + s) * 64 + lane) * 8]);
  lds_barrier();                              // B
  // chunk ch (step it): R in r[x], x = it % 4, the next chunk's M in buffer
  // (it + 1) % 4; past the first chunk the records read are chunk 0's, whose
  // values are not used
  auto step = [&](int ch, auto slot) {
    constexpr int x = decltype(slot)::value, nb = (x + 1) % kRing;
    chain_fetch_r(r[(x + 3) % kRing], rrec + rec_of(max(ch - 3, 0)) * kRBytes, w);
    bf16x8_t bop[4];
    chain_pack(bop, acc);
    // one address for the buffer's reads (the compiler would form one per read)
    uint32_t at = uint32_t(nb * D * D + lane * 8);
    asm volatile("" : "+v"(at));
    const uint16_t* next = &sM[0][0] + at;
    uint16_t* out = &sOut[x & 1][(16 * wave + w.c) * LDK + 4 * w.g];
#pragma unroll
    for (int kt = 0; kt < 8; kt += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[kt + u] = chain_r_tile(r[x], kt + u);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[kt + u] = mfma16_bf(m[kt + u][s], bop[s], acc[kt + u]);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int u = 0; u < 4; ++u) m[kt + u][s] = ld16_bf(next + ((kt + u) * 4 + s) * 512);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const uint4 p = __builtin_bit_cast(uint4, bop[kt / 2 + u]);
        *reinterpret_cast<uint2*>(out + 16 * (kt + 2 * u)) = uint2{p.x, p.y};
        *reinterpret_cast<uint2*>(out + 16 * (kt + 2 * u + 1)) = uint2{p.z, p.w};
      }
    }
    lds_barrier();
  };
  for (int ch = last; ch >= 0; ch -= 4) {
    step(ch, IC<0>());
    if (ch >= 1) step(ch - 1, IC<1>());
    if (ch >= 2) step(ch - 2, IC<2>());
    if (ch >= 3) step(ch - 3, IC<3>());
  }
  chain_store(dh0, acc, w);
}

// Gradients of one token's gating
//   g = -exp(A_log) softplus(x), x = a + dt_bias;  beta = sigmoid(b):
//   da = dg (-exp(A_log) sigmoid(x)) (ddt_bias sums them),  db = dbeta beta (1 - beta),
//   dA_log sums dg g.  The factors of dg and dbeta:
struct GateFactors {
  float da, db, g;
};
__device__ __forceinline__ GateFactors gate_factors(float x, float b, float exp_a) {
  const float be = sigmoidf_(b);
  return GateFactors{-exp_a * sigmoidf_(x), be * (1.f - be), -exp_a * softplus_stable(x)};
}

// Sums of x and of y over a workgroup of 256 threads, whole in thread 0.
__device__ __forceinline__ void sum_pair_256(float& x, float& y, float (&red)[2][4]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    x += __shfl_xor(x, off);
    y += __shfl_xor(y, off);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = x;
    red[1][threadIdx.x >> 6] = y;
  }
  __syncthreads();
  x = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
  y = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
}

// ---------------------------------------------------------------------------
// 3. Gradients of one (chunk, v-head) given S (h) and dSn (the chain's dh).
//
// Every matrix is held transposed in the accumulators (rows = the contiguous
// index of the row-major operand, column = token), so a lane's 4 values are
// 8 adjacent bf16 bytes of one token's row: LDS writes and global stores are
// packed, and a row sum is an in-lane sum plus two cross-group steps.
//   P1  K S^T, K dSn^T (wave w: state rows v 16 w .. +15, straight from the
//       registers S and dSn were loaded into); the lower 16x16 tiles of
//       Q K^T and K K^T (kept in registers for P3, P to LDS)
//   P2  X, Vn = Tm X, dVn = P^T dO + Dc K dSn^T, dX = Tm^T dVn, dV, all of
//       them split along v, so a wave only exchanges data with itself
//   P3  the lower tiles of dP = dO Vn^T and dA = -dX Vn^T (the inverse's
//       gradient -Tm^T (dVn X^T) Tm^T with its outer factors applied:
//       Tm^T dVn = dX, Tm X = Vn), their row and column sums
//   P4  dQ and dK, wave w: tokens 32 (w % 2) .. +31, columns 32 (w / 2) .. +31
//
// What bounds it, at 32 768 tokens qk16/v32 (one workgroup per CU, 153 KB of
// LDS): latency within a step ((chunk, v-head)): of its about 24 000 cycles
// the LDS is busy 46% (42% of that bank conflicts), the VALU 37% and the
// matrix cores 17%; HBM carries 3.25 GB in 0.74 ms with fp32 gradients, which
// take 0.70 ms in bf16.  It replaces a form that took 1.65 ms with the same products split
// by rows over 13 barriers per v-head: there Tm was inverted again by one wave
// of every workgroup, S and dSn were read from HBM twice, and nothing of the
// next unit was in flight.  The next step's loads go out over P3 and P4,
// where registers are free: issued together at the top of P4 they held up
// half of the waves (0.86 ms), issued at P1 they spilled (1.19 ms).
// Sums over a token's row go through per-contributor partial arrays (fixed
// summation order).
struct GradParts {
  // rows of the [64][128] products (contributor: wave): dgam, dbeta, Dc rowsum(Vn K dSn^T)
  float row[3][8][C];
  float tg[4][C];    // dgam rows, [64][64] products below the diagonal (contributor: column block)
  float tb[4][C];    // dbeta rows, [64][64] products
  float tc[4][C];    // dgam column sums (to subtract), [64][64] products (contributor: row block)
  float aq[4][C];    // scale E rowsum(Q (dO S)) (contributor: column quarter)
  float dot[2][8];   // <dSn, S> per wave, by parity of the step
};

__device__ __forceinline__ bf16x8_t as_bf8(const uint4& w) { return __builtin_bit_cast(bf16x8_t, w); }

// c + x . y for two packed bf16 pairs, in fp32.
__device__ __forceinline__ float dot2_bf16(uint32_t x, uint32_t y, float c) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, x), __builtin_bit_cast(bf16x2_t, y), c,
                                         false);
}

// 4 consecutive values of a gradient row from element `at` of the buffer, as fp32 or bf16.
template <typename GradT>
__device__ __forceinline__ void st_grad(__amdgpu_buffer_rsrc_t rows, int at, const f32x4& x) {
  if constexpr (std::is_same<GradT, float>::value)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, x), rows, at * 4, 0, 0);
  else
    buffer_store_b64(rows, uint32_t(at) * 2u, cvt_pk_bf16(x[0], x[1]), cvt_pk_bf16(x[2], x[3]));
}

constexpr int GLC = C + 16;          // [*][64] bf16 rows of the gradient kernel (160 B)

// What the gate gradients of a training step add (GradT = uint16_t): da, db
// (bf16, [T, HV]) in place of dg, dbeta, and per (chunk slot, v-head) the
// terms dg g and da of dA_log and ddt_bias summed over the chunk.
struct GateOut {
  void* g;            // dg (fp32) or da (bf16)
  void* beta;         // dbeta (fp32) or db (bf16)
  float2* parts;      // [slots][HV], GradT = uint16_t only
};

template <typename GradT>
__global__ __launch_bounds__(kGradThreads, 1) void gdn_bwd_grad_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const float* __restrict__ A_log, const uint16_t* __restrict__ a, const float* __restrict__ dt_bias,
    const uint16_t* __restrict__ b, int HQ, int HV, float scale, const uint16_t* __restrict__ d_out, const uint16_t* __restrict__ h, int h_chunks,
    int slots, const int2* __restrict__ chunks, const uint16_t* __restrict__ tmrec, const uint16_t* __restrict__ dh,
    GradT* __restrict__ dq, GradT* __restrict__ dk, GradT* __restrict__ dv, GateOut go) {
  constexpr bool kStep = std::is_same<GradT, uint16_t>::value;
  __shared__ __align__(16) uint16_t sK[C * LDK];
  __shared__ __align__(16) uint16_t sQ[C * LDK];
  __shared__ __align__(16) uint16_t sdO[C * LDK];
  __shared__ __align__(16) uint16_t sVn[C * LDK];   // X; then Vn
  __shared__ __align__(16) uint16_t sdX[C * LDK];   // dVn; then dX
  __shared__ __align__(16) uint16_t sS[D * LDK];    // S; then dSn
  __shared__ __align__(16) uint16_t sP[C * GLC];    // P; then dPm
  __shared__ __align__(16) uint16_t sB[C * GLC];    // Tm; then dAb + dAb^T
  __shared__ __align__(16) float gbuf[2][GB_SZ + (kStep ? 3 * C : 0)];
  __shared__ GradParts pt;

  const int tid0 = threadIdx.x, lane0 = tid0 & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6);
  const int G = HV / HQ;
  // Workgroups walk the (chunk slot, qk-head) units, qk-head fastest, and a
  // unit's G v-heads in turn, dq and dk summed over them in registers (v-head
  // order).  The next step's rows, states and gate inputs are loaded into
  // registers while this one is worked on.
  const int units = slots * HQ;
  struct At {
    int unit, m, t0, len;
  };
  // the first unit at or after `unit` (in this workgroup's stride) that holds
  // a chunk; unit >= units when there is none
  auto seek = [&](int unit) {
    At x{unit, 0, 0, 0};
    for (; x.unit < units; x.unit += int(gridDim.x)) {
      const int slot = x.unit / HQ;
      if (slot >= h_chunks) continue;
      const int2 ch = chunks[slot];
      x.t0 = ch.x;
      x.len = ch.y;
      if (ch.y > 0) break;
    }
    return x;
  };
  struct Regs {
    uint4 k[2], q[2], o[2], tm, s[4], ds[4];
    uint2 v[4];
  };
  auto fetch = [&](const At& x, Regs& r, int tid, int lane) {
    const int slot = x.unit / HQ, hq = x.unit - slot * HQ, hv = hq * G + x.m;
    const size_t rec = size_t(slot) * HV + hv;
    if (x.m == 0) {
      rows_fetch<kGradThreads>(r.k, head_rows(k, HQ, hq, x.t0, x.len), HQ, tid);
      rows_fetch<kGradThreads>(r.q, head_rows(q, HQ, hq, x.t0, x.len), HQ, tid);
    }
    rows_fetch<kGradThreads>(r.o, head_rows(d_out, HV, hv, x.t0, x.len), HV, tid);
    r.tm = reinterpret_cast<const uint4*>(tmrec + rec * C * C)[tid];
    const auto vb = head_rows(v, HV, hv, x.t0, x.len);
#pragma unroll
    for (int tb = 0; tb < 4; ++tb)
      r.v[tb] = buffer_load_b64(vb, uint32_t((16 * tb + (lane & 15)) * HV * D + 16 * wave + 4 * (lane >> 4)) * 2u);
  };
  // this wave's 16 rows of a state record (S or dSn) as MFMA operands
  auto fetch_state = [&](const At& x, const uint16_t* rec0, uint4 (&r)[4], int lane) {
    const int slot = x.unit / HQ, hv = (x.unit - slot * HQ) * G + x.m;
    const uint16_t* p = rec0 + (size_t(slot) * HV + hv) * D * D + (16 * wave + (lane & 15)) * D + 8 * (lane >> 4);
#pragma unroll
    for (int s = 0; s < 4; ++s) r[s] = *reinterpret_cast<const uint4*>(p + 32 * s);
  };

  // a step's gate data, formed one step ahead by wave 1
  auto gate_in = [&](const At& x, int lane) {
    const int slot = x.unit / HQ;
    return gate_inputs(A_log, a, dt_bias, b, HV, (x.unit - slot * HQ) * G + x.m, x.t0, x.len, lane);
  };
  auto gates = [&](const GateIn& gi, int len, int lane, float* gb) {
    chunk_gates_calc(gi, len, lane, gb);
    if constexpr (kStep) {
      const GateFactors f = gate_factors(bf16_bits_to_f32(gi.a) + gi.dt, bf16_bits_to_f32(gi.b), expf(gi.alog));
      gb[GB_DA + lane] = f.da;
      gb[GB_DB + lane] = f.db;
      gb[GB_G + lane] = f.g;
    }
  };

  // the tiles of sP above the diagonal that an operand read covers stay zero
  for (int x = tid0; x < 2 * 16 * 16; x += kGradThreads) {
    const int up = x >> 8, r = (x >> 4) & 15, c = x & 15;
    sP[(32 * up + r) * GLC + 32 * up + 16 + c] = 0;
  }

  Regs cur;
  At at = seek(int(blockIdx.x));
  if (at.unit >= units) return;
  fetch(at, cur, tid0, lane0);
  fetch_state(at, h, cur.s, lane0);
  fetch_state(at, dh, cur.ds, lane0);
  if (wave == 1) gates(gate_in(at, lane0), at.len, lane0, gbuf[0]);
  f32x4 dq_acc[2][2], dk_acc[2][2];      // [column block][token block], summed over the v-heads
  for (int it = 0; at.unit < units; ++it) {
    // Lane indices opaque to the compiler at the top of each phase: their
    // address arithmetic is formed where it is used instead of being kept in
    // registers across phases and steps.
    int tid = tid0, lane = lane0, g, c;
    auto fresh_lane = [&] {
      asm volatile("" : "+v"(lane));
      g = lane >> 4;
      c = lane & 15;
    };
    asm volatile("" : "+v"(tid));
    fresh_lane();
    const int slot = at.unit / HQ, hq = at.unit - slot * HQ, hv = hq * G + at.m;
    const int t0 = at.t0, len = at.len, m = at.m;
    float* gb = gbuf[it & 1];

    // P0: rows to LDS
    if (m == 0) {
      rows_store<kGradThreads>(sK, cur.k, tid);
      rows_store<kGradThreads>(sQ, cur.q, tid);
    }
    rows_store<kGradThreads>(sdO, cur.o, tid);
    *reinterpret_cast<uint4*>(sB + (tid >> 3) * GLC + 8 * (tid & 7)) = cur.tm;
    lds_barrier();

    // P1: K S^T and K dSn^T, transposed: rows v = 16 wave + 4 g + i, column t = 16 tb + c
    f32x4 ks[4], kd[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      ks[tb] = f32x4{0.f, 0.f, 0.f, 0.f};
      kd[tb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bf16x8_t ko = op_mr(sK, LDK, 16 * tb, 32 * s, lane);
        ks[tb] = mfma16_bf(as_bf8(cur.s[s]), ko, ks[tb]);
        kd[tb] = mfma16_bf(as_bf8(cur.ds[s]), ko, kd[tb]);
      }
    }
    float dot = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      *reinterpret_cast<uint4*>(sS + (16 * wave + c) * LDK + 32 * s + 8 * g) = cur.s[s];
      const uint32_t ss[4] = {cur.s[s].x, cur.s[s].y, cur.s[s].z, cur.s[s].w};
      const uint32_t dd[4] = {cur.ds[s].x, cur.ds[s].y, cur.ds[s].z, cur.ds[s].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) dot = dot2_bf16(ss[j], dd[j], dot);
    }
    // tiles (ti, tj) of Q K^T and K K^T: wave w takes tile w, waves 6 and 7 also 8 and 9
    f32x4 qk[2], kk[2], ex[2];
    auto tile_of = [&](int j, int& ti, int& tj) {
      const int tile = wave + 2 * j;
      ti = tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3;
      tj = tile - (ti * (ti + 1)) / 2;
    };
    auto qk_tiles = [&](auto count) {
      constexpr int n = decltype(count)::value;
#pragma unroll
      for (int j = 0; j < n; ++j) qk[j] = kk[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < n; ++j) {
          int ti, tj;
          tile_of(j, ti, tj);
          const bf16x8_t ka = op_mr(sK, LDK, 16 * tj, 32 * s, lane);
          qk[j] = mfma16_bf(ka, op_mr(sQ, LDK, 16 * ti, 32 * s, lane), qk[j]);
          kk[j] = mfma16_bf(ka, op_mr(sK, LDK, 16 * ti, 32 * s, lane), kk[j]);
        }
#pragma unroll
      for (int j = 0; j < n; ++j) {
        int ti, tj;
        tile_of(j, ti, tj);
        const int t = 16 * ti + c, s0 = 16 * tj + 4 * g;
        const float gt = gb[GB_GAM + t];
        const f32x4 gs = *reinterpret_cast<const f32x4*>(&gb[GB_GAM + s0]);
        f32x4 pv;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          ex[j][i] = t >= s0 + i ? exp_fast(gt - gs[i]) : 0.f;
          pv[i] = scale * (ex[j][i] * qk[j][i]);
        }
        st_bf4(sP + t * GLC + s0, pv);
      }
    };
    if (wave >= 6) qk_tiles(IC<2>());
    else qk_tiles(IC<1>());
    dot = wave_inclusive_scan(dot);
    if (lane == 63) pt.dot[it & 1][wave] = dot;
    At nx = at;
    ++nx.m;
    if (nx.m == G) nx = seek(at.unit + int(gridDim.x));
    const bool more = nx.unit < units;
    const At ld = more ? nx : at;       // what is loaded next (the last step loads its own inputs again)
    GateIn gin{};
    if (wave == 1) gin = gate_in(ld, lane);
    lds_barrier();

    // P2: everything split along v (this wave's 16 rows of the transposed tiles)
    fresh_lane();
    {
      const int v0 = 16 * wave + 4 * g;     // first of this lane's 4 columns v
      const auto dv_rows = head_rows(dv, HV, hv, t0, len);
      f32x4 xr[4], vn[4], dx[4];
      bf16x8_t xo[2], yo[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) yo[s] = op_rm(sdO, LDK, 16 * wave, 32 * s, lane);
#pragma unroll
      for (int tb = 0; tb < 4; ++tb) {
        const int t = 16 * tb + c;
        const float e = gb[GB_E + t], be = gb[GB_BETA + t], dc = gb[GB_DC + t];
        const f32x4 vv = bf4_f32(cur.v[tb]);
        f32x4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          ks[tb][i] *= e;
          xr[tb][i] = vv[i] - ks[tb][i];
          x[i] = be * xr[tb][i];
          kd[tb][i] *= dc;
        }
        st_bf4(sVn + t * LDK + v0, x);
        // dVn = Dc K dSn^T + P^T dO
        dx[tb] = kd[tb];
#pragma unroll
        for (int s = tb / 2; s < 2; ++s)
          dx[tb] = mfma16_bf(yo[s], op_rm(sP, GLC, 16 * tb, 32 * s, lane), dx[tb]);
        st_bf4(sdX + t * LDK + v0, dx[tb]);
      }
      // Vn = Tm X and dX = Tm^T dVn (Tm lower: rows 0-31 of Tm need only their
      // own 32 columns, rows 32-63 of Tm^T likewise)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        xo[s] = op_rm(sVn, LDK, 16 * wave, 32 * s, lane);
        yo[s] = op_rm(sdX, LDK, 16 * wave, 32 * s, lane);
      }
#pragma unroll
      for (int tb = 0; tb < 4; ++tb) {
        vn[tb] = dx[tb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if (s <= tb / 2) vn[tb] = mfma16_bf(xo[s], op_mr(sB, GLC, 16 * tb, 32 * s, lane), vn[tb]);
          if (s >= tb / 2) dx[tb] = mfma16_bf(yo[s], op_rm(sB, GLC, 16 * tb, 32 * s, lane), dx[tb]);
        }
      }
#pragma unroll
      for (int tb = 0; tb < 4; ++tb) {
        const int t = 16 * tb + c;
        const float be = gb[GB_BETA + t];
        st_bf4(sVn + t * LDK + v0, vn[tb]);
        st_bf4(sdX + t * LDK + v0, dx[tb]);
        f32x4 dvv;
        float sg = 0.f, sb = 0.f, sv = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          dvv[i] = be * dx[tb][i];
          sb = fmaf(dx[tb][i], xr[tb][i], sb);
          sg = fmaf(dvv[i], ks[tb][i], sg);
          sv = fmaf(vn[tb][i], kd[tb][i], sv);
        }
        st_grad<GradT>(dv_rows, t * HV * D + v0, dvv);
        const float sum = group4_sum3(-sg, sb, sv);
        if (g < 3) pt.row[g][wave][t] = sum;
      }
    }
    lds_barrier();

    fresh_lane();
    // the next step's inputs are loaded over P3 and P4
    Regs nxt;
    fetch(ld, nxt, tid, lane);
    // P3: dP and dA tiles (rows s = 16 tj + 4 g + i, column t = 16 ti + c)
    auto da_tiles = [&](auto count) {
      constexpr int n = decltype(count)::value;
      f32x4 dp[n], da[n];
#pragma unroll
      for (int j = 0; j < n; ++j) dp[j] = da[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < n; ++j) {
          int ti, tj;
          tile_of(j, ti, tj);
          const bf16x8_t va = op_mr(sVn, LDK, 16 * tj, 32 * s, lane);
          dp[j] = mfma16_bf(va, op_mr(sdO, LDK, 16 * ti, 32 * s, lane), dp[j]);
          da[j] = mfma16_bf(va, op_mr(sdX, LDK, 16 * ti, 32 * s, lane), da[j]);
        }
#pragma unroll
      for (int j = 0; j < n; ++j) {
        int ti, tj;
        tile_of(j, ti, tj);
        const int t = 16 * ti + c, s0 = 16 * tj + 4 * g;
        const float be = gb[GB_BETA + t];
        f32x4 dpm, dab, cs;
        float rg = 0.f, rb = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // ex is zero above the diagonal
          dpm[i] = scale * ex[j][i] * dp[j][i];
          const float xa = t > s0 + i ? -ex[j][i] * da[j][i] : 0.f;
          dab[i] = be * xa;
          // (a diagonal term would be added to its row and taken off its column)
          cs[i] = t > s0 + i ? fmaf(dpm[i], qk[j][i], dab[i] * kk[j][i]) : 0.f;
          rg += cs[i];
          rb = fmaf(xa, kk[j][i], rb);
        }
        st_bf4(sP + t * GLC + s0, dpm);
        const uint32_t b01 = cvt_pk_bf16(dab[0], dab[1]), b23 = cvt_pk_bf16(dab[2], dab[3]);
        const uint16_t bb[4] = {uint16_t(b01), uint16_t(b01 >> 16), uint16_t(b23), uint16_t(b23 >> 16)};
        if (ti != tj) {
          *reinterpret_cast<uint2*>(sB + t * GLC + s0) = uint2{b01, b23};
#pragma unroll
          for (int i = 0; i < 4; ++i) sB[(s0 + i) * GLC + t] = bb[i];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (t >= s0 + i) {                // dab is zero on the diagonal
              sB[t * GLC + s0 + i] = bb[i];
              sB[(s0 + i) * GLC + t] = bb[i];
            }
        }
        rg = group4_sum(rg);
        rb = group4_sum(rb);
        if (g == 0) {
          pt.tg[tj][t] = rg;
          pt.tb[tj][t] = rb;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x = row16_sum(cs[i]);
          if (c == 0) pt.tc[ti][s0 + i] = x;
        }
      }
    };
    if (wave >= 6) da_tiles(IC<2>());
    else da_tiles(IC<1>());
    if (wave == 1) gates(gin, ld.len, lane, gbuf[(it + 1) & 1]);
    lds_barrier();
    fetch_state(ld, h, nxt.s, lane);
    // P4: dQ = scale E dO S + dPm K;  dK = Dc Vn dSn - beta E dX S + dPm^T Q + (dAb + dAb^T) K
    fresh_lane();
    const int tr0 = 32 * (wave & 1), k0 = 32 * (wave >> 1);
    f32x4 y[2][2], z[2][2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) y[kb][tb] = z[kb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      bf16x8_t so[2], oo[2], xo[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        so[u] = op_rm(sS, LDK, k0 + 16 * u, 32 * s, lane);
        oo[u] = op_mr(sdO, LDK, tr0 + 16 * u, 32 * s, lane);
        xo[u] = op_mr(sdX, LDK, tr0 + 16 * u, 32 * s, lane);
      }
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
          y[kb][tb] = mfma16_bf(so[kb], oo[tb], y[kb][tb]);
          z[kb][tb] = mfma16_bf(so[kb], xo[tb], z[kb][tb]);
        }
    }
    const float e0 = gb[GB_E + tr0 + c], e1 = gb[GB_E + tr0 + 16 + c];
    const float be0 = gb[GB_BETA + tr0 + c], be1 = gb[GB_BETA + tr0 + 16 + c];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      const int t = tr0 + 16 * tb + c;
      const float fq = scale * (tb ? e1 : e0), fx = -(tb ? be1 * e1 : be0 * e0);
      float sq = 0.f;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const f32x4 qv = bf4_f32(*reinterpret_cast<const uint2*>(sQ + t * LDK + k0 + 16 * kb + 4 * g));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          y[kb][tb][i] *= fq;
          z[kb][tb][i] *= fx;
          sq = fmaf(y[kb][tb][i], qv[i], sq);
        }
      }
      sq = group4_sum(sq);
      if (g == 0) pt.aq[wave >> 1][t] = sq;
    }
    // the triangular products: dPm's rows 0-31 end at column 31, dPm^T's rows 32-63 begin at 32
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8_t ko[2], qo[2], po[2], pto[2], bo[2];
      const bool lo = s == 0 || tr0 != 0, hi = s == 1 || tr0 == 0;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        ko[u] = op_rm(sK, LDK, k0 + 16 * u, 32 * s, lane);
        bo[u] = op_mr(sB, GLC, tr0 + 16 * u, 32 * s, lane);
      }
      if (lo) {
#pragma unroll
        for (int u = 0; u < 2; ++u) po[u] = op_mr(sP, GLC, tr0 + 16 * u, 32 * s, lane);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int tb = 0; tb < 2; ++tb) y[kb][tb] = mfma16_bf(ko[kb], po[tb], y[kb][tb]);
      }
      if (hi) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          qo[u] = op_rm(sQ, LDK, k0 + 16 * u, 32 * s, lane);
          pto[u] = op_rm(sP, GLC, tr0 + 16 * u, 32 * s, lane);
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int tb = 0; tb < 2; ++tb) z[kb][tb] = mfma16_bf(qo[kb], pto[tb], z[kb][tb]);
      }
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) z[kb][tb] = mfma16_bf(ko[kb], bo[tb], z[kb][tb]);
    }
    lds_barrier();
#pragma unroll
    for (int s = 0; s < 4; ++s)
      *reinterpret_cast<uint4*>(sS + (16 * wave + c) * LDK + 32 * s + 8 * g) = cur.ds[s];
    fetch_state(ld, dh, nxt.ds, lane);
    lds_barrier();
    fresh_lane();
    {
      f32x4 x[2][2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) x[kb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        bf16x8_t so[2], vo[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          so[u] = op_rm(sS, LDK, k0 + 16 * u, 32 * s, lane);
          vo[u] = op_mr(sVn, LDK, tr0 + 16 * u, 32 * s, lane);
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int tb = 0; tb < 2; ++tb) x[kb][tb] = mfma16_bf(so[kb], vo[tb], x[kb][tb]);
      }
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) {
        const float dc = gb[GB_DC + tr0 + 16 * tb + c];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
          for (int i = 0; i < 4; ++i) z[kb][tb][i] = fmaf(dc, x[kb][tb][i], z[kb][tb][i]);
          dq_acc[kb][tb] = m == 0 ? y[kb][tb] : dq_acc[kb][tb] + y[kb][tb];
          dk_acc[kb][tb] = m == 0 ? z[kb][tb] : dk_acc[kb][tb] + z[kb][tb];
        }
      }
    }
    // the last v-head stores the sums (the buffers are empty before it)
    {
      const int n = m == G - 1 ? len : 0;
      const auto dq_rows = head_rows(dq, HQ, hq, t0, n), dk_rows = head_rows(dk, HQ, hq, t0, n);
#pragma unroll
      for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const int at0 = (tr0 + 16 * tb + c) * HQ * D + k0 + 16 * kb + 4 * g;
          st_grad<GradT>(dq_rows, at0, dq_acc[kb][tb]);
          st_grad<GradT>(dk_rows, at0, dk_acc[kb][tb]);
        }
    }
    if (wave == 0) {
      const int t = lane, blk = lane >> 4;
      float dgam = 0.f, dbt = 0.f, dsum = 0.f, vk = 0.f;
#pragma unroll
      for (int w = 0; w < 8; ++w) {
        dgam += pt.row[0][w][t];
        dbt += pt.row[1][w][t];
        dsum += pt.dot[it & 1][w];
        vk += pt.row[2][w][t];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dgam += pt.aq[j][t];
        if (j <= blk) {
          dgam += pt.tg[j][t];
          dbt += pt.tb[j][t];
        }
        if (j >= blk) dgam -= pt.tc[j][t];
      }
      if (t == C - 1) dgam += gb[GB_EL] * dsum;
      // dg_t = sum_{i >= t} dgam_i.  Of the row terms vk = Dc rowsum(Vn K
      // dSn^T), taken off each row and added whole to the last one, that
      // leaves sum_{i < t} vk_i, formed as such: with strong decay dg is far
      // smaller than the vk of the last rows, and their difference would be
      // its rounding (A_log 3 to 5: dA_log 2.1e-2 off, 5.9e-3 with both sums
      // in one order, 2.8e-3 like this).
      const float suffix = __shfl(wave_inclusive_scan(__shfl(dgam, 63 - t)), 63 - t);
      const float before = __shfl_up(vk, 1);
      const float dgt = suffix + wave_inclusive_scan(t == 0 ? 0.f : before);
      const size_t i = size_t(t0 + t) * HV + hv;
      if constexpr (kStep) {
        float sa = 0.f, sd = 0.f;
        if (t < len) {
          const float dai = dgt * gb[GB_DA + t], dbi = dbt * gb[GB_DB + t];
          sa = dgt * gb[GB_G + t];
          sd = dai;
          reinterpret_cast<uint16_t*>(go.g)[i] = f32_to_bf16_bits(dai);
          reinterpret_cast<uint16_t*>(go.beta)[i] = f32_to_bf16_bits(dbi);
        }
        sa = wave_inclusive_scan(sa);
        sd = wave_inclusive_scan(sd);
        if (lane == 63) go.parts[size_t(slot) * HV + hv] = float2{sa, sd};
      } else if (t < len) {
        reinterpret_cast<float*>(go.g)[i] = dgt;
        reinterpret_cast<float*>(go.beta)[i] = dbt;
      }
    }
    cur = nxt;
    at = nx;
  }
}

// Gradients of the gating, per v-head (one workgroup each), over all tokens.
__global__ __launch_bounds__(256) void gdn_gate_bwd_kernel(
    const float* __restrict__ A_log, const uint16_t* __restrict__ a, const float* __restrict__ dt_bias,
    const uint16_t* __restrict__ b, const float* __restrict__ dg, const float* __restrict__ dbeta, int T,
    int HV, float* __restrict__ da, float* __restrict__ db, float* __restrict__ dA_log,
    float* __restrict__ ddt_bias) {
  __shared__ float red[2][4];
  const int hv = blockIdx.x, tid = threadIdx.x;
  const float ea = expf(A_log[hv]), bias = dt_bias[hv];
  float sa = 0.f, sd = 0.f;
  for (int t = tid; t < T; t += 256) {
    const size_t i = size_t(t) * HV + hv;
    const GateFactors f = gate_factors(bf16_bits_to_f32(a[i]) + bias, bf16_bits_to_f32(b[i]), ea);
    const float dai = dg[i] * f.da;
    da[i] = dai;
    db[i] = dbeta[i] * f.db;
    sa = fmaf(dg[i], f.g, sa);
    sd += dai;
  }
  sum_pair_256(sa, sd, red);
  if (tid == 0) {
    dA_log[hv] = sa;
    ddt_bias[hv] = sd;
  }
}

// dA_log and ddt_bias of a training step: the chunks' partial sums per v-head
// (one workgroup each), chunks in a fixed order.
template <typename CuT>
__global__ __launch_bounds__(256) void gdn_gate_sums_kernel(const CuT* __restrict__ cu, int N, int T,
                                                            int HV, int h_chunks,
                                                            const float2* __restrict__ parts,
                                                            float* __restrict__ dA_log,
                                                            float* __restrict__ ddt_bias) {
  __shared__ float red[2][4];
  const int hv = blockIdx.x, tid = threadIdx.x;
  const int chunks = min(h_chunks, chunk_offset(cu, N, T, tid & 63));
  float sa = 0.f, sd = 0.f;
  for (int s = tid; s < chunks; s += 256) {
    const float2 x = parts[size_t(s) * HV + hv];
    sa += x.x;
    sd += x.y;
  }
  sum_pair_256(sa, sd, red);
  if (tid == 0) {
    dA_log[hv] = sa;
    ddt_bias[hv] = sd;
  }
}

// Workspace of a backward over `slots` chunk slots.
struct BwdWorkspace {
  char* m;
  char* r;           // R; the chain kernel leaves dSn there
  uint16_t* tm;
  int2* chunks;      // first token and length of every chunk slot (length 0: none)
  float2* parts;     // over m, which the chain kernel has consumed by then
  BwdWorkspace(char* ws, size_t slots, size_t HV) {
    const size_t units = slots * HV;
    m = ws;
    r = m + units * kMBytes;
    tm = reinterpret_cast<uint16_t*>(r + units * kRBytes);
    chunks = reinterpret_cast<int2*>(tm + units * (kTmBytes / 2));
    parts = reinterpret_cast<float2*>(m);
  }
  static size_t bytes(size_t slots, size_t HV) {
    return slots * HV * (kMBytes + kRBytes + kTmBytes) + slots * sizeof(int2);
  }
};

// GradT = float: fp32 gradients, dg and dbeta in g_out and beta_out.
// GradT = uint16_t: a training step's, in bf16, with da and db there and the
// per-head sums in dA_log and ddt_bias.
template <typename CuT, typename GradT>
int launch_bwd(const uint16_t* q, const uint16_t* k, const uint16_t* v, const float* A_log,
               const uint16_t* a, const float* dt_bias, const uint16_t* b, const CuT* cu, int N, int T,
               int HQ, int HV, float scale, const uint16_t* h, int h_chunks, const uint16_t* d_out,
               const float* d_ht, GradT* dq, GradT* dk, GradT* dv, GradT* g_out, GradT* beta_out,
               float* dA_log, float* ddt_bias, float* dh0, char* ws, hipStream_t st) {
  const size_t slots = size_t(T) / C + size_t(N);
  // The workspace holds `slots` chunk records per v-head.  Well-formed
  // cu_seqlens give at most that many chunks; with overlapping ranges the
  // chunk count (and h_chunks) can exceed it, and every kernel then stops at
  // the last slot the workspace holds (results unspecified, accesses in bounds).
  h_chunks = int(std::min<size_t>(size_t(h_chunks), slots));
  const size_t units = slots * size_t(HV);
  const BwdWorkspace w(ws, slots, size_t(HV));
  const int cus = device_cus();
  const size_t wgs = size_t(cus > 0 ? cus : 256);
  if (N > 0) {
    // Two persistent workgroups per CU.  A unit takes the v-heads of a qk-head
    // together (K, Q and their products once) where that leaves every
    // workgroup a unit; with fewer, a v-head each.
    const int heads = slots * size_t(HQ) >= 2 * wgs ? HV / HQ : 1;
    const unsigned pgrid = unsigned(std::min(slots * size_t(HV / heads), 2 * wgs));
    hipLaunchKernelGGL((gdn_bwd_prep_kernel<CuT>), dim3(pgrid), dim3(kPrepThreads), 0, st, q, k, A_log, a,
                       dt_bias, b, cu, N, T, HQ, HV, scale, d_out, h_chunks, int(slots), heads, w.m, w.r,
                       w.tm, w.chunks);
    // The reverse chain: one workgroup per chain, or eight or four where they
    // all run at once (a chain's time is then its chunks' latency, which more
    // workgroups of fewer rows cut; with more chains than that HBM bounds the
    // launch).
    const unsigned chains = unsigned(N) * unsigned(HV), chain_ids = 8u * ((chains + 7u) / 8u);
    if (cus > 0 && 8LL * N * HV <= cus)
      hipLaunchKernelGGL((gdn_bwd_chain_few_kernel<CuT, 1>), dim3(8u * chain_ids), dim3(64 * (1 + kCopyWaves)), 0, st, cu, N, T, HV,
                         h_chunks, w.m, w.r, d_ht, dh0);
    else if (cus > 0 && 4LL * N * HV <= cus)
      hipLaunchKernelGGL((gdn_bwd_chain_few_kernel<CuT, 2>), dim3(4u * chain_ids), dim3(64 * (2 + kCopyWaves)), 0, st, cu, N, T, HV,
                         h_chunks, w.m, w.r, d_ht, dh0);
    else
      hipLaunchKernelGGL((gdn_bwd_chain_kernel<CuT>), dim3(chains), dim3(512), 0, st, cu, N, T, HV, h_chunks,
                         w.m, w.r, d_ht, dh0);
    if (T > 0) {
      // one workgroup per CU walks the (chunk, qk-head) units
      const unsigned ggrid = unsigned(std::min(slots * size_t(HQ), wgs));
      hipLaunchKernelGGL((gdn_bwd_grad_kernel<GradT>), dim3(ggrid), dim3(kGradThreads), 0, st, q, k, v,
                         A_log, a, dt_bias, b, HQ, HV, scale, d_out, h, h_chunks, int(slots), w.chunks,
                         w.tm, reinterpret_cast<const uint16_t*>(w.r), dq, dk, dv,
                         GateOut{g_out, beta_out, w.parts});
    }
  }
  if (dA_log)
    hipLaunchKernelGGL((gdn_gate_sums_kernel<CuT>), dim3(unsigned(HV)), dim3(256), 0, st, cu, N, T, HV,
                       h_chunks, w.parts, dA_log, ddt_bias);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GDN_OK : -int(e);
}

// The argument checks of both entry points (outputs apart).
int check_bwd(const uint16_t* q, const uint16_t* k, const uint16_t* v, const float* A_log, const uint16_t* a,
              const float* dt_bias, const uint16_t* b, const void* cu, int N, int T, int HQ, int HV,
              const uint16_t* h, int h_chunks, const uint16_t* d_out, bool outputs) {
  if (N < 0 || T < 0 || HQ <= 0 || HV <= 0 || HV % HQ != 0 || h_chunks < 0) return GDN_ERR_SHAPE;
  if (!cu) return GDN_ERR_NULL;
  if (N > 0 && (!A_log || !dt_bias)) return GDN_ERR_NULL;
  if (T > 0 && (!q || !k || !v || !a || !b || !d_out || !outputs)) return GDN_ERR_NULL;
  if (h_chunks > 0 && !h) return GDN_ERR_NULL;
  return GDN_OK;
}

}  // namespace

extern "C" size_t gdn_prefill_bwd_workspace_bytes(int N, int T, int HQ, int HV) {
  if (N < 0 || T < 0 || HQ <= 0 || HV <= 0 || HV % HQ != 0) return 0;
  return BwdWorkspace::bytes(size_t(T) / C + size_t(N), size_t(HV));
}

extern "C" int gdn_prefill_bwd(const uint16_t* q, const uint16_t* k, const uint16_t* v,
                               const float* A_log, const uint16_t* a, const float* dt_bias,
                               const uint16_t* b, const void* cu_seqlens, int cu_is_int32, int N,
                               int T, int HQ, int HV, float scale, const uint16_t* h, int h_chunks,
                               const uint16_t* d_out, const float* d_final_state, float* dq, float* dk,
                               float* dv, float* dg, float* dbeta, float* d_initial_state,
                               void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = check_bwd(q, k, v, A_log, a, dt_bias, b, cu_seqlens, N, T, HQ, HV, h, h_chunks, d_out,
                           dq && dk && dv && dg && dbeta);
  if (rc != GDN_OK || N == 0) return rc;
  if (!workspace || workspace_bytes < gdn_prefill_bwd_workspace_bytes(N, T, HQ, HV))
    return GDN_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  auto launch = [&](auto* cu) {
    return launch_bwd(q, k, v, A_log, a, dt_bias, b, cu, N, T, HQ, HV, scale, h, h_chunks, d_out,
                      d_final_state, dq, dk, dv, dg, dbeta, static_cast<float*>(nullptr),
                      static_cast<float*>(nullptr), d_initial_state, ws, st);
  };
  return cu_is_int32 ? launch(static_cast<const int32_t*>(cu_seqlens))
                     : launch(static_cast<const int64_t*>(cu_seqlens));
}

extern "C" int gdn_prefill_bwd_step(const uint16_t* q, const uint16_t* k, const uint16_t* v,
                                    const float* A_log, const uint16_t* a, const float* dt_bias,
                                    const uint16_t* b, const void* cu_seqlens, int cu_is_int32, int N,
                                    int T, int HQ, int HV, float scale, const uint16_t* h, int h_chunks,
                                    const uint16_t* d_out, const float* d_final_state, uint16_t* dq,
                                    uint16_t* dk, uint16_t* dv, uint16_t* da, uint16_t* db, float* dA_log,
                                    float* ddt_bias, float* d_initial_state, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  const int rc = check_bwd(q, k, v, A_log, a, dt_bias, b, cu_seqlens, N, T, HQ, HV, h, h_chunks, d_out,
                           dq && dk && dv && da && db);
  if (rc != GDN_OK) return rc;
  if (!dA_log || !ddt_bias) return GDN_ERR_NULL;
  if (workspace_bytes < gdn_prefill_bwd_workspace_bytes(N, T, HQ, HV) || (N > 0 && !workspace))
    return GDN_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  auto launch = [&](auto* cu) {
    return launch_bwd(q, k, v, A_log, a, dt_bias, b, cu, N, T, HQ, HV, scale, h, h_chunks, d_out,
                      d_final_state, dq, dk, dv, da, db, dA_log, ddt_bias, d_initial_state, ws, st);
  };
  return cu_is_int32 ? launch(static_cast<const int32_t*>(cu_seqlens))
                     : launch(static_cast<const int64_t*>(cu_seqlens));
}

extern "C" int gdn_gate_bwd(const float* A_log, const uint16_t* a, const float* dt_bias, const uint16_t* b,
                            const float* dg, const float* dbeta, int T, int HV, float* da, float* db,
                            float* dA_log, float* ddt_bias, void* stream) {
  if (T < 0 || HV <= 0) return GDN_ERR_SHAPE;
  if (!A_log || !dt_bias || !dA_log || !ddt_bias) return GDN_ERR_NULL;
  if (T > 0 && (!a || !b || !dg || !dbeta || !da || !db)) return GDN_ERR_NULL;
  hipLaunchKernelGGL(gdn_gate_bwd_kernel, dim3(unsigned(HV)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     A_log, a, dt_bias, b, dg, dbeta, T, HV, da, db, dA_log, ddt_bias);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GDN_OK : -int(e);
}
