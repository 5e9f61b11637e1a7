// ldpca.hip -- LDPCA sum-product decoding on gfx950.
//
// Replaces beliefPropagation_CUDA / beliefPropagation_CUDA_earlyJump
// (DvcDec/src/LDPCA_cuda.cu:872-1031) and the rate search of LdpcaDecoder
// (DvcDec/src/LdpcaDecoder.cpp:646-771).  Arithmetic follows the reference's
// ParallelMode 0 decoder (beliefPropagation, LdpcaDecoder.cpp:462-580) step
// for step, so every message, decision and iteration count equals the CPU
// path's:
//   * phi(x) = -logf(tanhf((x + 1e-9f)/2)) with the glibc-identical routines
//     of dvc_math.h, in their branch-free form for x >= 0 (every argument
//     here is a magnitude: a row's sum of |phi| is at least each of its
//     terms, so |sum| - |phi_e| >= 0), dvc_bp_phi_fast;
//   * check-node sums accumulate in ascending edge order (= ascending column),
//     the order of `rowTotal[ir[k]] += ...` (:514-515);
//   * variable-node sums accumulate LLR + c2v0 + c2v1 + c2v2 (:527-539);
//   * decisions are the sign bit of the overall LLR (:548); the syndrome test
//     is the row parity (:551-568).
//
// Layout.  One workgroup owns one (bitplane, code) pair.  Messages live in LDS:
// phi[E] holds |phi| of every variable-to-check message with the message's
// sign in the sign bit, stored by check row (row r's edges at rowPtr[r] ..
// rowPtr[r+1]-1, ascending edge order), so a check sums a contiguous run;
// rowTot[m] holds each check's sum of |phi| with the check's sign product
// (including the syndrome bit) in the sign bit.  Thread t owns columns t,
// t+T, ...; a column's three edges come as (row, message slot) words, the
// slot precomputed per code, so the variable-node update, the next check-node input and
// the decision are computed in registers without further exchange.  Two
// barriers per iteration: after the check (row) pass and after the variable
// (column) pass.  The syndrome test's decision parities are XORed into
// per-check bits by the variable pass (LDS atomics, double-buffered across
// iterations), so the check pass reads no column data besides phi.
//
// Batched form.  A persistent grid walks a queue of (bitplane, code offset)
// items in offset-major order.  An item whose code lies above the lowest code
// that already converged with a matching CRC for its bitplane is skipped, and
// a running item notices that at its next iteration and stops.  Every code
// below the final choice always runs to completion, so the kept code is the
// one the sequential search returns.
#include <stdio.h>
#include <string.h>
#include <algorithm>
#include <vector>
#include "dvc_internal.h"
#include "dvc_math.h"
#include "ldpca_kernels.h"

#pragma clang fp contract(off)

namespace dvc {

__device__ __forceinline__ uint32_t f2u(float f) { return __float_as_uint(f); }

// Pointers the kernels read from descriptors in memory are generic, and a
// generic (flat) load is counted by the LDS wait counter as well: a wait for
// an LDS read would also wait for it.  These views make such loads global.
typedef const float __attribute__((address_space(1))) gfloat_t;
typedef const uint8_t __attribute__((address_space(1))) gbyte_t;
typedef const uint32_t __attribute__((address_space(1))) gword_t;
__device__ __forceinline__ gfloat_t *as_global(const float *p) { return (gfloat_t *)p; }
__device__ __forceinline__ gbyte_t *as_global(const uint8_t *p) { return (gbyte_t *)p; }
__device__ __forceinline__ gword_t *as_global(const uint32_t *p) { return (gword_t *)p; }

// A column's three edges as the ladder upload packs them: row | slot << 15,
// slot = the edge's message position in row order; off = slot * 4, the
// message's byte offset in the phi array, is the word shifted right by 13.
__device__ __forceinline__ void col_edges(const ColEdges &c, int row[3], uint32_t off[3]) {
#pragma unroll
  for (int q = 0; q < 3; q++) {
    row[q] = (int)(c.e[q] & 0x1fffu);
    off[q] = c.e[q] >> 13;
  }
}
__device__ __forceinline__ float &at_byte(float *base, uint32_t off) {
  return *(float *)((uint8_t *)base + off);
}
__device__ __forceinline__ float u2f(uint32_t u) { return __uint_as_float(u); }

// Accumulated-syndrome bit i (MSB-first bytes, ByteToBit LdpcaDecoder.cpp:81-107).
__device__ __forceinline__ uint32_t acc_bit(gbyte_t *acc, int i) {
  return (acc[i >> 3] >> (7 - (i & 7))) & 1u;
}

// ------------------------------------------------------------------ CE + LLR
// ComputeCE (LdpcaDecoder.cpp:127-143) and the LR -> LLR conversion (:663-667)
// for one bitplane per workgroup.  The entropy is the reference's sequential
// float sum over the columns, N dependent additions, 16 us of a CIF bitplane when
// one lane makes them (the whole kernel then takes 24 us, the terms computed
// meanwhile).  sum_terms gets the same bits from a scan: while the sum s stays
// within one binade, adding a term t >= 0 moves s by a whole number of its ulps u,
// floor(t/u) or one more, which hangs on s only by its lowest bit, for a t that
// ends in exactly half an ulp (ties go to even).  So a run of terms is a pair of
// whole numbers, the ulps it adds to an even and to an odd s, and two runs compose.
//   * Every thread takes CH consecutive terms.  Approximate sums before and after
//     them, with a bound on how far the sequential sum can be from those, say
//     whether s stays within one binade meanwhile.
//   * Threads of one wave and binade compose their runs by a segmented scan; those
//     near a power of two keep their terms.
//   * The pieces, 35 or so, are applied in order: a run by an addition to s's bits,
//     the rest term by term.
// More than 64 pieces (sums that dwell at a power of two) and terms that are
// negative, not numbers or above 2 (no likelihood ratio of a decoder gives such)
// go lane by lane as before.
// A CIF bitplane takes 15.7 us so, 26 with the additions by one lane (the terms are
// 9 of them: 99 waves' worth of three logf on one CU).  A QCIF one's 1584 additions
// take no longer than the scan (10.3 and 10.4 us): it keeps them.
#define DVC_LOG2 (0.693147181f)
constexpr int CE_T = 1024, CE_W = CE_T / 64, CE_SCAN = 4096;

struct CeShared {
  __align__(16) float tot[CE_W];  // sums of the waves' terms
  int pieces[CE_W];
  int4 piece[64];  // thread of the terms or -1, ulps for an even and an odd sum
};

// The six steps of a scan over a wave: the value of the lane 1, 2, 4, 8 back in
// the row of 16, then of the last lane of the row or of the two rows before.  Where
// a step brings nothing it gives 0.
template <int STEP>
__device__ __forceinline__ int scan_from(int v) {
  if constexpr (STEP < 4) return __builtin_amdgcn_update_dpp(0, v, 0x110 | 1 << STEP, 0xf, 0xf, false);
  if constexpr (STEP == 4) return __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  return __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
}
template <int STEP>
__device__ __forceinline__ void scan_sum(float &v) {
  v += u2f((uint32_t)scan_from<STEP>((int)f2u(v)));
}
// Two runs composed, unless a segment begins in between.
template <int STEP>
__device__ __forceinline__ void scan_runs(int &inc0, int &inc1, int &head) {
  const int a0 = scan_from<STEP>(inc0), a1 = scan_from<STEP>(inc1), h = scan_from<STEP>(head);
  const int n0 = a0 + (a0 & 1 ? inc1 : inc0), n1 = a1 + (a1 & 1 ? inc0 : inc1);
  inc0 = head ? inc0 : n0;
  inc1 = head ? inc1 : n1;
  head |= h;
}

// True: wave 0 has the sum.  Every thread of the workgroup calls it.
template <int CH>
__device__ bool sum_terms(const float *terms, int N, CeShared &sh, float *sum) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, first = tid * CH;
  float t[CH], local = 0.0f;
#pragma unroll
  for (int i = 0; i < CH; i++) {
    t[i] = first + i < N ? terms[first + i] : 0.0f;
    local += t[i];
  }
  float upto = local;
  scan_sum<0>(upto), scan_sum<1>(upto), scan_sum<2>(upto);
  scan_sum<3>(upto), scan_sum<4>(upto), scan_sum<5>(upto);
  float before = __shfl_up(upto, 1);
  if (lane == 0) before = 0.0f;
  if (lane == 63) sh.tot[wave] = upto;
  __syncthreads();
  float waves = 0.0f;
#pragma unroll
  for (int w = 0; w < CE_W; w++) waves += w < wave ? sh.tot[w] : 0.0f;
  before += waves;
  upto += waves;
  // k float additions of terms >= 0 end within k ulps' halves (2^-24 each) of the
  // exact sum, relative to it; the sums here within 30 of them
  const float tol = (float)(first + CH + 64) * 6.3e-8f;
  const uint32_t e = f2u(before * (1.0f - tol)) >> 23;
  const bool valid = first < N, clear = e > 64u && e == f2u(upto * (1.0f + tol)) >> 23;
  int inc0 = 0, inc1 = 1;  // inc1 starts at an odd sum
  if (clear) {
    const float scale = u2f((277u - e) << 23);  // 1/u = 2^(150 - e)
#pragma unroll
    for (int i = 0; i < CH; i++) {
      const float q = t[i] * scale, fl = floorf(q), fr = q - fl;  // all exact, q < 2^24
      const int k = (int)fl, half = fr == 0.5f, up = fr > 0.5f;
      inc0 += k;
      inc1 += k;
      inc0 += up | (half & inc0);
      inc1 += up | (half & inc1);
    }
  }
  inc1 -= 1;
  const int key = clear ? (int)e : -1, key1 = __shfl_up(key, 1);
  int head = lane == 0 || !valid || key < 0 || key != key1;
  const uint64_t heads = __ballot(head);
  scan_runs<0>(inc0, inc1, head), scan_runs<1>(inc0, inc1, head), scan_runs<2>(inc0, inc1, head);
  scan_runs<3>(inc0, inc1, head), scan_runs<4>(inc0, inc1, head), scan_runs<5>(inc0, inc1, head);
  const bool tail = valid && (lane == 63 || (heads >> (lane + 1) & 1u));
  const uint64_t tails = __ballot(tail);
  if (lane == 0) sh.pieces[wave] = __popcll(tails);
  __syncthreads();
  int at = __popcll(tails & ((1ull << lane) - 1)), all = 0;
#pragma unroll
  for (int w = 0; w < CE_W; w++) {
    const int n = sh.pieces[w];
    at += w < wave ? n : 0;
    all += n;
  }
  if (all > 64) return false;
  if (tail) sh.piece[at] = make_int4(clear ? -1 : tid, inc0, inc1, 0);
  __syncthreads();
  if (wave != 0) return true;
  const int4 p = lane < all ? sh.piece[lane] : make_int4(-1, 0, 0, 0);
  float own[CH];
#pragma unroll
  for (int i = 0; i < CH; i++) own[i] = p.x >= 0 && p.x * CH + i < N ? terms[p.x * CH + i] : 0.0f;
  float s = 0.0f;
  for (int j = 0; j < all; j++) {
    if (__builtin_amdgcn_readlane(p.x, j) < 0) {
      const int i0 = __builtin_amdgcn_readlane(p.y, j), i1 = __builtin_amdgcn_readlane(p.z, j);
      s = u2f(f2u(s) + (uint32_t)(f2u(s) & 1u ? i1 : i0));
    } else {
#pragma unroll
      for (int i = 0; i < CH; i++) s += u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(own[i]), j));
    }
  }
  *sum = s;
  return true;
}

// It also clears the step's launch counters and, with the workgroups beyond the
// bitplanes', the control blocks of a split BP launch (a kernel's stores, so that a
// captured step holds no memset; a launch of their own took 5 us).
__global__ __launch_bounds__(CE_T) void ce_llr_kernel(const PlaneDesc *planes, int nplanes, int fixed_start,
                                                      const float *codeRate1584, const float *codeRate6336,
                                                      int numCodes1584, int numCodes6336, int *counters,
                                                      uint4 *clear, int clearQuads) {
  __shared__ __align__(16) float terms[6336 + 64];  // spare: the last group of 64
  __shared__ CeShared sh;
  const int p = blockIdx.x, tid = threadIdx.x;
  if (p >= nplanes) {
    const int i = (p - nplanes) * CE_T + tid;
    if (i < clearQuads) clear[i] = make_uint4(0u, 0u, 0u, 0u);
    return;
  }
  const PlaneDesc d = planes[p];
  const int N = d.N;
  if (p == 0 && tid < 3) counters[tid] = 0;
  int flags = 0;  // 1: a NaN LLR, 2: a term that sum_terms does not take
  if (tid < 64) terms[N + tid] = 0.0f;
  constexpr int PER = (6336 + CE_T - 1) / CE_T;
  float lrs[PER];
#pragma unroll
  for (int j = 0; j < PER; j++)
    if (tid + j * CE_T < N) lrs[j] = as_global(d.LR)[tid + j * CE_T];
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const int k = tid + j * CE_T;
    if (k >= N) break;
    const float lr = lrs[j];
    const float Pco = lr / (1.0f + lr);
    const float tmp = dvc_logf(1 - Pco);
    const float term = (Pco * (-dvc_logf(Pco) + tmp) - tmp) / DVC_LOG2;
    terms[k] = term;
    const float llr = dvc_logf(lr);
    d.LLR[k] = llr;
    flags |= (llr != llr ? 1 : 0) | (term >= 0.0f && term <= 2.0f ? 0 : 2);
  }
  const int nan = __syncthreads_or(flags & 1), slow = __syncthreads_or((flags & 2) != 0);
  float rlb = 0.0f;
  if (N < CE_SCAN || slow || !sum_terms<PER>(terms, N, sh, &rlb)) {
    // past the last column the terms are +0, which leaves the sum as it is
    const float4 *q = (const float4 *)terms;
    if (tid < 64)
#pragma unroll 1
      for (int g = 0; g < (N + 63) >> 6; g++, q += 16) {
        float4 a[16];
#pragma unroll
        for (int i = 0; i < 16; i++) a[i] = q[i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; i++) {
          rlb += a[i].x;
          rlb += a[i].y;
          rlb += a[i].z;
          rlb += a[i].w;
        }
      }
  }
  if (tid >= 64) return;
  rlb /= (float)N;
  // A NaN likelihood ratio makes the entropy NaN; the x86 path's is its
  // default NaN (sign set), which the GPU's NaN bits need not be.  No rate
  // compares below it, so the start code is 0, as at :657-659.
  if (rlb != rlb) rlb = __uint_as_float(0xffc00000u);
  const float *rate = N == 1584 ? codeRate1584 : codeRate6336;
  const int last = (N == 1584 ? numCodes1584 : numCodes6336) - 1;
  // the first code whose rate is not below the entropy, or the last one
  int s = last;
  for (int base = 0; base < last && s == last; base += 64) {
    const int i = base + tid;
    const uint64_t stop = __ballot(i < last && !(rate[i] < rlb));
    if (stop) s = base + __builtin_ctzll(stop);
  }
  if (tid == 0) {
    PlaneState *st = d.state;
    st->entropy = rlb;
    if (st->start < 0 || !fixed_start) st->start = s;
    st->run = st->start;
    st->taint = nan;
  }
}
// ------------------------------------------------------------------ BP
template <int N, int T>
struct BpShape {
  static constexpr int E = 3 * N;
  static constexpr int CPT = (N + T - 1) / T;      // columns per thread
  static constexpr int DEC_WORDS = (CPT * T) / 32;  // ballot words of every column slot
  static constexpr int SYN_WORDS = (N + 31) / 32;
};

// One check's row of messages, slots e0 .. e1-1 of phi: |phi| summed in
// ascending edge order (:514-515) and the messages' sign product; returns the
// row's total with syn times that product in the sign bit.
__device__ __forceinline__ float check_row(const float *phi, int e0, int e1, uint32_t syn) {
  uint32_t sx = 0u;  // XOR of the row's message words: the sign product in bit 31
  float sum = 0.0f;
  // groups of four loads without conditions, then the last 1..3 slots
  // read unconditionally too (the rows are contiguous and phi has spare
  // slots at its end) with those past the row's end taken as +0: sum +
  // 0.0f is sum bit for bit (sum is never -0)
  int j = e0;
  for (; j + 4 <= e1; j += 4) {
    uint32_t f[4];
#pragma unroll
    for (int i = 0; i < 4; i++) f[i] = f2u(phi[j + i]);
#pragma unroll
    for (int i = 0; i < 4; i++) sum += u2f(f[i] & 0x7fffffffu);
    sx ^= f[0] ^ f[1] ^ f[2] ^ f[3];
  }
  if (j < e1) {
    uint32_t f[3];
#pragma unroll
    for (int i = 0; i < 3; i++) f[i] = f2u(phi[j + i]);
    f[1] = j + 1 < e1 ? f[1] : 0u;
    f[2] = j + 2 < e1 ? f[2] : 0u;
#pragma unroll
    for (int i = 0; i < 3; i++) sum += u2f(f[i] & 0x7fffffffu);
    sx ^= f[0] ^ f[1] ^ f[2];
  }
  return u2f(f2u(sum) | ((syn ^ (sx >> 31)) << 31));
}

// c2v of a column's three edges and its overall LLR (:512-539).
template <bool MODE1, class Phi>
__device__ __forceinline__ float column_total(const int row[3], const uint32_t pos[3], float llr, const float *rowTot,
                                              float *phi, const Phi &phi_of, float c2v[3]) {
  uint32_t R[3], ph[3];
  float x[3], v[3];
#pragma unroll
  for (int q = 0; q < 3; q++) {
    R[q] = f2u(rowTot[row[q]]);
    ph[q] = f2u(at_byte(phi, pos[q]));
  }
#pragma unroll
  for (int q = 0; q < 3; q++) x[q] = u2f(R[q] & 0x7fffffffu) - u2f(ph[q] & 0x7fffffffu);
#pragma unroll
  for (int q = 0; q < 3; q++) v[q] = phi_of(x[q]);
#pragma unroll
  for (int q = 0; q < 3; q++)
    // times -1 or 1 by the sign product; with no NaN (ParallelMode 0
    // never runs a NaN bitplane) that is the sign bit flipped
    c2v[q] = MODE1 ? (((R[q] ^ ph[q]) >> 31) ? v[q] * -1.0f : v[q] * 1.0f)
                   : u2f((f2u(v[q]) & 0x7fffffffu) | ((f2u(v[q]) ^ R[q] ^ ph[q]) & 0x80000000u));
  float tmp = llr;
  tmp += c2v[0];
  tmp += c2v[1];
  tmp += c2v[2];
  return tmp;
}
// The next v2c of the edges as messages: phi of the magnitude with the sign.
template <class Phi>
__device__ __forceinline__ void column_messages(float tmp, const float c2v[3], const Phi &phi_of, float f[3]) {
  uint32_t sg[3];
  float x[3], v[3];
#pragma unroll
  for (int q = 0; q < 3; q++) {
    const float v2c = tmp - c2v[q];
    sg[q] = f2u(v2c) >> 31;
    x[q] = (sg[q] ? -1.0f : 1.0f) * v2c;
  }
#pragma unroll
  for (int q = 0; q < 3; q++) v[q] = phi_of(x[q]);
#pragma unroll
  for (int q = 0; q < 3; q++) f[q] = copysignf(v[q], u2f(sg[q] << 31));
}
// A column's decision 1 XORed into its three checks' parity bits.
__device__ __forceinline__ void column_parity(const ColEdges &rows, const int row[3], uint32_t *par) {
#pragma unroll
  for (int q = 0; q < 3; q++) {
    // word row >> 5 = bits 5..12 of the column word, extracted by one
    // v_bfe_u32 (kept as written, so that the word's address is one
    // shift-and-add); the bit's shift takes the row's low 5 bits
    uint32_t w;
    __asm__("v_bfe_u32 %0, %1, 5, 8" : "=v"(w) : "v"(rows.e[q]));
    atomicXor(&par[w], 1u << (row[q] & 31));
  }
}

// MODE1: beliefPropagation_OpenMP's semantics (ParallelMode 1), else
// beliefPropagation's (ParallelMode 0).
//
// NaN likelihood ratios (PlaneState.taint).  On the x86 path a NaN LLR makes
// every message that depends on it NaN.  With ParallelMode 0's sign-bit
// decisions the outcome then hangs on NaN sign bits, and every code of such a
// bitplane fails after MAX_ITERATIONS (the reference run over the golden GOP
// frames and over seeded bitplanes with injected NaNs never converges), so a
// tainted code is recorded as failed after max_iter iterations without being
// run.  ParallelMode 1 decides LLR < 0, false for NaN, so only which values
// are NaN matters: the kernel then keeps NaN through phi (whose branch-free
// form would turn it into a finite value) and IEEE arithmetic carries it like
// the CPU path.
template <int N, int T, bool MODE1>
__global__ __launch_bounds__(T) void bp_persistent_kernel(BpArgs a) {
  using S = BpShape<N, T>;
  constexpr int E = S::E;
  // phi's logf table: (invc * 2^-k, k*ln2 + logc) for each (k, i) that phi's
  // arguments reach, read with per-lane indices
  __shared__ __align__(16) double s_phitab[2 * DVC_PHI_LOGTAB];
  // by check row; 3 spare slots at the end, so that the check pass may read
  // a row's last group of four unconditionally
  __shared__ float phi[E + 3];
  __shared__ float rowTot[N];
  __shared__ uint16_t rowPtr[N + 2];
  __shared__ uint32_t decBits[S::DEC_WORDS];
  __shared__ uint32_t synBits[S::SYN_WORDS];
  __shared__ int s_item;
  // some check failed, a lower code has been accepted (alternate iterations).  One
  // barrier and these, not __syncthreads_or, which takes three and a reduction; with
  // the bitplane's best code asked for a pass ahead and the first column's words kept
  // in registers, no global load is waited for between the passes (one QCIF bitplane
  // 1255 -> 1207 us, 256 CIF frames 374 -> 369 ms)
  __shared__ int s_fail[2], s_cancel[2];
  __shared__ uint32_t s_crc[T / 64];
  __shared__ uint32_t parBits[2][S::SYN_WORDS];  // decision parity per check, written by alternate iterations
  __shared__ int s_changed[2];  // ParallelMode 1: some decision changed in the variable pass (alternate iterations)

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const LadderDev L = a.lad;
  for (int e = tid; e < DVC_PHI_LOGTAB; e += T) dvc_phi_logtab_entry(e, s_phitab);

  for (;;) {
    // ---- grab the next item (lane 0 of the workgroup), broadcast through LDS
    if (tid == 0) {
      int item = -1;
      for (;;) {
        int w = atomicAdd(a.next, 1);
        if (w >= a.total) break;
        int b = w % a.nplanes, off = w / a.nplanes;
        PlaneState *st = a.planes[b].state;
        int level = st->run + off;
        if (off >= a.max_offset || level >= L.numCodes - 1) continue;
        if (a.rate_step && !dynstep_tries(off)) continue;
        if (__hip_atomic_load(&st->best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < level) continue;
        item = w;
        break;
      }
      s_item = item;
    }
    __syncthreads();
    const int w = s_item;
    if (w < 0) return;
    const int b = w % a.nplanes;
    const PlaneDesc pd = a.planes[b];
    PlaneState *st = pd.state;
    const int run = st->run;
    const int level = run + w / a.nplanes;
    const bool taint = st->taint != 0;
    if (!MODE1 && taint) {
      if (tid == 0) pd.rec[level] = make_int4(a.max_iter, REC_FAILED, -1, 0);
      __syncthreads();  // every thread has read s_item before the next grab rewrites it
      continue;
    }
    // phi of the kernel, NaN-preserving on a tainted ParallelMode 1 bitplane
    auto phi_of = [&](float x) {
      const float v = dvc_bp_phi_fast(x, s_phitab);
      return (MODE1 && taint && x != x) ? x : v;
    };
    // ParallelMode 1: the decisions carried into this code are known only for
    // the queue's first code; a later code runs as if its first decisions
    // differ from them and records the one case where that matters
    const bool mode1 = MODE1, exact = level == run;
    const int m = L.syndLength[level];
    const ColEdges *gcol = L.colRows + (size_t)level * N;

    // ---- stage the code's row starts and the syndrome (LdpcaDecoder.cpp:684-693)
    const uint16_t *growPtr = L.rowPtr + (size_t)level * (N + 1);
    for (int i = tid; i <= m; i += T) rowPtr[i] = growPtr[i];
    for (int wd = tid; wd < S::SYN_WORDS; wd += T) {
      uint32_t bits = 0;
      for (int q = 0; q < 32; q++) {
        int k = wd * 32 + q;
        if (k < m) {
          int cur = L.tx[(size_t)level * N + k];
          uint32_t s = acc_bit(as_global(pd.acc), cur);
          if (k > 0) s ^= acc_bit(as_global(pd.acc), L.tx[(size_t)level * N + k - 1]);
          bits |= s << q;
        }
      }
      synBits[wd] = bits;
    }
    // ---- variable-to-check messages start at the channel LLR (:478-481)
    for (int j = 0; j < S::CPT; j++) {
      int k = tid + j * T;
      if (k < N) {
        float v = as_global(pd.LLR)[k];
        uint32_t s = f2u(v) >> 31;
        float mag = (s ? -1.0f : 1.0f) * v;
        uint32_t f = f2u(copysignf(phi_of(mag), v));  // |phi| with the LLR's sign bit
        int row[3];
        uint32_t off[3];
        col_edges(gcol[k], row, off);
#pragma unroll
        for (int q = 0; q < 3; q++) at_byte(phi, off[q]) = u2f(f);
      }
    }
    // this thread's first column, the same in every iteration
    gfloat_t *gLLR = as_global(pd.LLR);
    const ColEdges rows0 = tid < N ? gcol[tid] : ColEdges{{0u, 0u, 0u}};
    const float llr0 = tid < N ? gLLR[tid] : 0.0f;
    if (tid == 0) s_cancel[0] = s_fail[0] = 0;
    __syncthreads();

    int status = 0, iters = 0, poll = 0;
    int sameCount = 0, bcaseSlot = 0;
    for (int t = 0;; t++) {
      // ---- check-node pass: |phi| sums and sign products; parity of the
      // previous decisions (:495-515, :551-568)
      // The previous variable pass XORed each column's decision into its
      // three checks' bits of parBits[(t - 1) & 1]; this pass reads them and
      // clears parBits[t & 1] for the coming variable pass.
      int fail = 0;
      const uint32_t *parPrev = parBits[(t + 1) & 1];
      for (int r = tid; r < m; r += T) {
        const int e0 = rowPtr[r], e1 = rowPtr[r + 1];
        const uint32_t syn = (synBits[r >> 5] >> (r & 31)) & 1u;
        rowTot[r] = check_row(phi, e0, e1, syn);
        if (t > 0 && (syn ^ ((parPrev[r >> 5] >> (r & 31)) & 1u))) fail = 1;
      }
      for (int wd = tid; wd < S::SYN_WORDS; wd += T) parBits[t & 1][wd] = 0u;
      // ParallelMode 1 (beliefPropagation_OpenMP, LdpcaDecoder.cpp:254-264):
      // count consecutive iterations whose decisions all repeat the previous
      // ones; the fourth such iteration ends the code as a failure, before
      // the parity test of the same iteration
      if (mode1 && t > 0) sameCount = s_changed[(t - 1) & 1] ? 0 : sameCount + 1;
      if (tid == 0) s_changed[t & 1] = 0;
      if (fail) s_fail[t & 1] = 1;
      __syncthreads();
      const int anyFail = s_fail[t & 1];
      const bool cancel = s_cancel[t & 1] != 0;
      if (mode1 && !exact && t == 4 && sameCount == 3) {
        // Decisions of iterations 0-3 all equal: had the carried decisions
        // equalled them too, the code would have failed here after 4
        // iterations.  Keep these decisions for the resolution.
        if (tid == 0) s_item = atomicAdd(a.slot_count, 1);
        __syncthreads();
        const int bs = s_item;
        if (bs < a.slot_capacity) {
          uint8_t *dst = a.slots + (size_t)bs * N;
          for (int j = 0; j < S::CPT; j++) {
            const int k = tid + j * T;
            if (k < N) dst[k] = (uint8_t)((decBits[k >> 5] >> (k & 31)) & 1u);
          }
        }
        bcaseSlot = bs + 1;
        __syncthreads();
      }
      if (mode1 && sameCount == 4) { status = 0; iters = t; break; }
      if (t > 0 && !anyFail) { status = 1; iters = t; break; }
      if (cancel) { status = 3; iters = t; break; }
      if (t == a.max_iter) { status = 0; iters = t; break; }

      // ---- variable-node pass: c2v, overall LLR, decision, next v2c (:512-548)
      // The next column's rows and channel LLR are fetched while this
      // column's six phi evaluations run.
      bool changed = false;
      // lane 0 looks whether a lower code has been accepted, for the next check
      // pass: the answer arrives meanwhile
      int best = level;
      const bool ask = poll == 0;
      poll = ask ? a.poll - 1 : poll - 1;
      if (tid == 0) {
        s_fail[(t + 1) & 1] = 0;
        if (ask) best = __hip_atomic_load(&st->best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      ColEdges rowsNext = rows0;
      float llrNext = llr0;
      for (int j = 0; j < S::CPT; j++) {
        const int k = tid + j * T;
        const ColEdges rows = rowsNext;
        const float llr = llrNext;
        if (j + 1 < S::CPT && k + T < N) {
          rowsNext = gcol[k + T];
          llrNext = gLLR[k + T];
        }
        uint32_t dec = 0;
        if (k < N) {
          float c2v[3];
          int row[3];
          uint32_t pos[3];
          col_edges(rows, row, pos);
          const float tmp = column_total<MODE1>(row, pos, llr, rowTot, phi, phi_of, c2v);
          if (!mode1) {
            dec = f2u(tmp) >> 31;
          } else {
            dec = tmp < 0.0f;  // LLR_overall < 0 (LdpcaDecoder.cpp:257-260): -0 decides 0
            if (t == 0) changed |= !exact || as_global(pd.carry)[k] != (uint8_t)dec;
            else changed |= ((decBits[k >> 5] >> (k & 31)) & 1u) != dec;
          }
          if (dec) column_parity(rows, row, parBits[t & 1]);
          float f[3];
          column_messages(tmp, c2v, phi_of, f);
#pragma unroll
          for (int q = 0; q < 3; q++) at_byte(phi, pos[q]) = f[q];
        }
        const uint64_t bal = __ballot(dec);
        if (lane == 0) {
          const int word = (j * T + wave * 64) >> 5;
          decBits[word] = (uint32_t)bal;
          decBits[word + 1] = (uint32_t)(bal >> 32);
        }
      }
      if (changed) s_changed[t & 1] = 1;
      if (tid == 0) s_cancel[(t + 1) & 1] = best < level;
      __syncthreads();
    }

    // ---- converged: CRC-8 of the decisions (linear in the bits, crc8.h:5-6)
    int ok = 0;
    if (status == 1) {
      uint32_t crc = 0;
      for (int j = 0; j < S::CPT; j++) {
        int k = tid + j * T;
        if (k < N && ((decBits[k >> 5] >> (k & 31)) & 1u)) crc ^= L.crcBasis[k];
      }
      for (int o = 32; o > 0; o >>= 1) crc ^= __shfl_xor(crc, o);
      if (lane == 0) s_crc[wave] = crc;
      __syncthreads();
      uint32_t tot = 0;
      for (int i = 0; i < T / 64; i++) tot ^= s_crc[i];
      ok = (tot == pd.crc);
      if (ok) {
        int slot = -1;
        if (tid == 0) {
          slot = atomicAdd(a.slot_count, 1);
          s_item = slot;  // reuse as broadcast
        }
        __syncthreads();
        slot = s_item;
        if (slot < a.slot_capacity) {
          uint8_t *dst = a.slots + (size_t)slot * N;
          for (int j = 0; j < S::CPT; j++) {
            int k = tid + j * T;
            if (k < N) dst[k] = (uint8_t)((decBits[k >> 5] >> (k & 31)) & 1u);
          }
        }
        if (tid == 0) {
          pd.rec[level] = make_int4(iters, 2, slot, 0);
          atomicMin(&st->best, level);
        }
      }
    }
    if (!ok && mode1 && status != 3) {
      // ParallelMode 1 keeps every run code's final decisions: they are the
      // decisions carried into the next code
      if (tid == 0) s_item = atomicAdd(a.slot_count, 1);
      __syncthreads();
      const int slot = s_item;
      if (slot < a.slot_capacity) {
        uint8_t *dst = a.slots + (size_t)slot * N;
        for (int j = 0; j < S::CPT; j++) {
          const int k = tid + j * T;
          if (k < N) dst[k] = (uint8_t)((decBits[k >> 5] >> (k & 31)) & 1u);
        }
      }
      if (tid == 0) pd.rec[level] = make_int4(iters, status == 1 ? 1 : 0, slot, 0);
    } else if (tid == 0 && !ok) {
      pd.rec[level] = make_int4(iters, status == 1 ? 1 : (status == 3 ? 3 : 0), -1, 0);
    }
    if (tid == 0 && mode1) pd.bcase[level] = bcaseSlot;
    __syncthreads();
  }
}

// ------------------------------------------------------------------ split BP
// A codeword on one CU is bound by that CU's VALU: 16 us per CIF iteration, with
// most of the chip idle when a launch has few bitplanes.  Here a cluster of up to
// 8 workgroups works on one codeword.  Every member holds the whole codeword's
// messages in LDS and sums all rows, but updates only its share of the columns
// (64-column groups, dealt round); after the variable pass the members exchange
// their new messages and decisions through memory and go on with the same state,
// so they take every decision alike and only the leader (member 0) reports.
//
// Exchange: agent-scope relaxed stores in column order (whole lines; each reader
// puts the messages into row order itself, its column words loaded while it
// waits), a wait for their completion, then the member's counter; the others poll
// the counters and read with agent-scope loads.  Two buffers and two sets of
// counters alternate, and either is rewritten only after a later exchange that
// every reader of it has arrived at.  Every item handed to the members has at
// least one exchange, so the leader does not hand out the next one before all of
// them have seen it.
//
// No wait can be for a workgroup that is not running: a cluster is closed by its
// leader with the members that have arrived within 30 us of it, a later one
// leaves at once, and every wait is for members or the leader of a closed
// cluster.  The polls are bounded all the same; a member that runs into the bound
// leaves, and its codes' records stay unfinished.  In ParallelMode 0 the search
// then ends at a higher code or at the full rate, which the host refuses
// (unfinished_code); a ParallelMode 1 resolution runs such codes again.
//
// With 8 members an iteration takes 7.2 us against 16: row sums 1.7, columns 1.4,
// stores until complete 1.7, counters 1.0, reading and reordering 1.6.  A CIF
// bitplane's batch decode 0.84 -> 0.42 ms, its plain search over 3 codes 2.16 ->
// 1.08.  (Messages stored in row order, so that they are read without reordering:
// 4-byte stores to as many lines, 0.62 and 1.66; parities taken from everybody's
// decisions while reordering, the LDS atomics then on no arithmetic's back, 0.48
// and 1.23.)
template <int N, int T, bool MODE1>
__global__ __launch_bounds__(T) void bp_split_kernel(BpArgs a) {
  constexpr int NWS = (N + 63) / 64, SYN = (N + 31) / 32, W = T / 64;
  constexpr size_t BUF = split_buf_words(N);
  constexpr int PACK = 2, FLAG = 16, FLAG_STEP = 8;  // words of a control block
  static_assert(FLAG + 2 * kSplitMax * FLAG_STEP <= kCtlWords, "control block too small");
  constexpr int kSpin = 1 << 22;
  __shared__ __align__(16) double s_phitab[2 * DVC_PHI_LOGTAB];
  __shared__ __align__(16) float phi[3 * N + 4];
  __shared__ float rowTot[N];
  __shared__ uint16_t rowPtr[N + 2];
  __shared__ uint32_t decBits[2 * NWS];
  __shared__ uint32_t synBits[SYN], parBits[2 * NWS], parMine[2 * NWS];
  __shared__ int s_item, s_size, s_rank, s_cluster, s_cancel, s_changed, s_abort, s_fail[2];
  __shared__ uint32_t s_crc[W];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const LadderDev L = a.lad;
  for (int e = tid; e < DVC_PHI_LOGTAB; e += T) dvc_phi_logtab_entry(e, s_phitab);
  auto ld32 = [](const uint32_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  auto ld64 = [](const uint64_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  auto st32 = [](uint32_t *p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  auto st64 = [](uint64_t *p, uint64_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };

  // ---- join a cluster
  if (tid == 0) {
    const uint32_t ticket = __hip_atomic_fetch_add(a.area, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int cluster = (int)(ticket / (uint32_t)a.split);
    uint32_t *state = a.area + (size_t)kCtlWords * (1 + cluster);  // members joined, bit 8: closed
    s_cluster = cluster;
    s_abort = 0;
    if (ticket % (uint32_t)a.split == 0) {
      const uint64_t t0 = wall_clock64();  // 100 MHz
      while ((int)(ld32(state) & 0xffu) < a.split - 1 && wall_clock64() - t0 < 3000) __builtin_amdgcn_s_sleep(1);
      const uint32_t old = __hip_atomic_fetch_or(state, 0x100u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_rank = 0;
      s_size = 1 + (int)(old & 0xffu);
    } else {
      const uint32_t old = __hip_atomic_fetch_add(state, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_rank = (old & 0x100u) ? -1 : 1 + (int)(old & 0xffu);
    }
  }
  __syncthreads();
  // out of LDS into scalar registers, and the addresses formed from them too (15
  // vector registers spilled without it, 8 with: 7.69 -> 7.54 us per iteration of a
  // plain search, launches included)
  const int rank = __builtin_amdgcn_readfirstlane(s_rank), cluster = __builtin_amdgcn_readfirstlane(s_cluster);
  if (rank < 0) return;
  uint32_t *ctl = a.area + (size_t)kCtlWords * (1 + cluster);
  uint32_t *xbuf = a.area + kSplitCtlWords + (size_t)cluster * 2 * BUF;
  uint32_t xc = 0;  // exchanges so far, over all items

  for (uint32_t seq = 1;; seq++) {
    // ---- the leader grabs the next item and hands it to the members with the
    // cluster's size: (seq, size << 28 | item + 1) in one word
    if (tid == 0) {
      uint32_t low = 0;
      if (rank == 0) {
        int item = -1;
        for (;;) {
          const int w = atomicAdd(a.next, 1);
          if (w >= a.total) break;
          const int b = w % a.nplanes, off = w / a.nplanes;
          PlaneState *st = a.planes[b].state;
          const int level = st->run + off;
          if (off >= a.max_offset || level >= L.numCodes - 1) continue;
          if (a.rate_step && !dynstep_tries(off)) continue;
          if (__hip_atomic_load(&st->best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < level) continue;
          if (!MODE1 && st->taint) {
            a.planes[b].rec[level] = make_int4(a.max_iter, REC_FAILED, -1, 0);
            continue;
          }
          item = w;
          break;
        }
        low = (uint32_t)s_size << 28 | (uint32_t)(item + 1);
        st64((uint64_t *)(ctl + PACK), (uint64_t)seq << 32 | low);
      } else {
        for (int n = 0; n < kSpin; n++) {
          const uint64_t v = ld64((const uint64_t *)(ctl + PACK));
          if ((uint32_t)(v >> 32) == seq) {
            low = (uint32_t)v;
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
      }
      s_item = (int)(low & 0x0fffffffu) - 1;
      s_size = (int)(low >> 28);
    }
    __syncthreads();
    const int w = __builtin_amdgcn_readfirstlane(s_item), size = __builtin_amdgcn_readfirstlane(s_size);
    if (w < 0) return;
    const int b = w % a.nplanes;
    const PlaneDesc pd = a.planes[b];
    PlaneState *st = pd.state;
    const int run = st->run;
    const int level = run + w / a.nplanes;
    const bool taint = st->taint != 0;
    auto phi_of = [&](float x) {
      const float v = dvc_bp_phi_fast(x, s_phitab);
      return (MODE1 && taint && x != x) ? x : v;
    };
    const bool mode1 = MODE1, exact = level == run;
    const int m = L.syndLength[level];
    const ColEdges *gcol = L.colRows + (size_t)level * N;
    gfloat_t *gLLR = as_global(pd.LLR);

    // ---- the code's row starts, the syndrome and the first messages, as in
    // bp_persistent_kernel, on every member
    const uint16_t *growPtr = L.rowPtr + (size_t)level * (N + 1);
    for (int i = tid; i <= m; i += T) rowPtr[i] = growPtr[i];
    for (int wd = tid; wd < SYN; wd += T) {
      uint32_t bits = 0;
      for (int q = 0; q < 32; q++) {
        const int k = wd * 32 + q;
        if (k < m) {
          const int cur = L.tx[(size_t)level * N + k];
          uint32_t s = acc_bit(as_global(pd.acc), cur);
          if (k > 0) s ^= acc_bit(as_global(pd.acc), L.tx[(size_t)level * N + k - 1]);
          bits |= s << q;
        }
      }
      synBits[wd] = bits;
    }
    for (int k = tid; k < N; k += T) {
      const float v = gLLR[k];
      const float mag = (f2u(v) >> 31 ? -1.0f : 1.0f) * v;
      const float f = copysignf(phi_of(mag), v);
      int row[3];
      uint32_t off[3];
      col_edges(gcol[k], row, off);
#pragma unroll
      for (int q = 0; q < 3; q++) at_byte(phi, off[q]) = f;
    }
    if (tid == 0) s_cancel = s_changed = s_fail[0] = 0;
    for (int wd = tid; wd < 2 * NWS; wd += T) parMine[wd] = 0u;
    // this wave's first column group, the same in every iteration
    const int k0 = (rank + size * wave) * 64 + lane;
    const ColEdges rows0 = k0 < N ? gcol[k0] : ColEdges{{0u, 0u, 0u}};
    const float llr0 = k0 < N ? gLLR[k0] : 0.0f;
    __syncthreads();

    int status = 0, iters = 0;
    int sameCount = 0, bcaseSlot = 0;
    for (int t = 0;; t++) {
      // ---- check pass over all rows
      int fail = 0;
      for (int r = tid; r < m; r += T) {
        const uint32_t syn = (synBits[r >> 5] >> (r & 31)) & 1u;
        rowTot[r] = check_row(phi, rowPtr[r], rowPtr[r + 1], syn);
        if (t > 0 && (syn ^ ((parBits[r >> 5] >> (r & 31)) & 1u))) fail = 1;
      }
      if (mode1 && t > 0) sameCount = s_changed ? 0 : sameCount + 1;
      const bool cancel = s_cancel != 0;
      if (fail) s_fail[t & 1] = 1;
      __syncthreads();
      const int anyFail = s_fail[t & 1];
      if (mode1 && !exact && t == 4 && sameCount == 3 && rank == 0) {
        if (tid == 0) s_item = atomicAdd(a.slot_count, 1);
        __syncthreads();
        const int bs = s_item;
        if (bs < a.slot_capacity) {
          uint8_t *dst = a.slots + (size_t)bs * N;
          for (int k = tid; k < N; k += T) dst[k] = (uint8_t)((decBits[k >> 5] >> (k & 31)) & 1u);
        }
        bcaseSlot = bs + 1;
        __syncthreads();
      }
      if (mode1 && sameCount == 4) { status = 0; iters = t; break; }
      if (t > 0 && !anyFail) { status = 1; iters = t; break; }
      if (cancel) { status = 3; iters = t; break; }
      if (t == a.max_iter) { status = 0; iters = t; break; }
      if (tid == 0) s_changed = s_fail[(t + 1) & 1] = 0;
      for (int wd = tid; wd < 2 * NWS; wd += T) parBits[wd] = 0u;

      // ---- variable pass over this member's columns
      uint32_t *xb = xbuf + (xc & 1u) * BUF;
      uint64_t *xdec = (uint64_t *)(xb + 3 * N), *xpar = xdec + NWS;
      uint32_t stop = 0;
      if (tid == 0 && rank == 0 && t % a.poll == 0)
        stop = __hip_atomic_load(&st->best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < level;
      for (int i = wave; rank + size * i < NWS; i += W) {
        const int ws = rank + size * i, k = ws * 64 + lane;
        uint32_t dec = 0;
        if (k < N) {
          const ColEdges rows = i == wave ? rows0 : gcol[k];
          const float llr = i == wave ? llr0 : gLLR[k];
          float c2v[3], f[3];
          int row[3];
          uint32_t pos[3];
          col_edges(rows, row, pos);
          const float tmp = column_total<MODE1>(row, pos, llr, rowTot, phi, phi_of, c2v);
          dec = mode1 ? tmp < 0.0f : f2u(tmp) >> 31;
          if (dec) column_parity(rows, row, parMine);
          column_messages(tmp, c2v, phi_of, f);
#pragma unroll
          for (int q = 0; q < 3; q++) st32(xb + q * N + k, f2u(f[q]));
        }
        const uint64_t bal = __ballot(dec);
        if (lane == 0) st64(xdec + ws, bal);
      }
      // the columns whose messages this thread brings into row order, two at a
      // time, and the counter once this workgroup's stores have completed
      constexpr int PAIRS = (N / 2 + T - 1) / T;
      const auto has = [&](int i) { return (i + 1) * T <= N / 2 || tid + i * T < N / 2; };
      __syncthreads();  // parMine is complete
      if (tid < NWS) st64(xpar + rank * NWS + tid, (uint64_t)parMine[2 * tid + 1] << 32 | parMine[2 * tid]);
      __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) st32(ctl + FLAG + FLAG_STEP * (kSplitMax * (xc & 1u) + rank), (xc + 1) << 1 | stop);
      uint2 edge[PAIRS][3];
#pragma unroll
      for (int i = 0; i < PAIRS; i++)
#pragma unroll
        for (int q = 0; q < 3; q++)
          if (has(i)) edge[i][q] = ((const uint2 *)gcol)[3 * (tid + i * T) + q];
      if (wave == 0) {
        uint32_t v = 0;
        for (int n = 0;; n++) {
          if (lane < size) v = ld32(ctl + FLAG + FLAG_STEP * (kSplitMax * (xc & 1u) + lane));
          if (!__ballot(lane < size && v >> 1 != ((xc + 1) & 0x7fffffffu))) break;
          if (n == kSpin) {
            s_abort = 1;
            break;
          }
        }
        const uint64_t cancelled = __ballot(v & 1u);
        if (lane == 0) s_cancel = cancelled != 0;
      }
      __syncthreads();
      if (s_abort) return;
      // ---- everybody's messages and decisions
      {
        const uint64_t *xm = (const uint64_t *)xb;
        uint64_t f[PAIRS][3], dv = 0, pv = 0;
#pragma unroll
        for (int i = 0; i < PAIRS; i++)
#pragma unroll
          for (int q = 0; q < 3; q++)
            if (has(i)) f[i][q] = ld64(xm + q * (N / 2) + tid + i * T);
        if (tid < NWS) dv = ld64(xdec + tid);
        static_assert(kSplitMax * NWS <= T, "a thread per word of the members' parities");
        if (tid < size * NWS) pv = ld64(xpar + tid);
        bool changed = mode1 && t == 0 && !exact;
#pragma unroll
        for (int i = 0; i < PAIRS; i++) {
          if (!has(i)) break;
          const ColEdges two[2] = {{{edge[i][0].x, edge[i][0].y, edge[i][1].x}},
                                   {{edge[i][1].y, edge[i][2].x, edge[i][2].y}}};
#pragma unroll
          for (int h = 0; h < 2; h++) {
            int row[3];
            uint32_t pos[3];
            col_edges(two[h], row, pos);
#pragma unroll
            for (int q = 0; q < 3; q++) at_byte(phi, pos[q]) = u2f((uint32_t)(f[i][q] >> (32 * h)));
          }
        }
        if (tid < NWS) {
          const uint32_t lo = (uint32_t)dv, hi = (uint32_t)(dv >> 32);
          if (mode1 && t > 0) changed |= decBits[2 * tid] != lo || decBits[2 * tid + 1] != hi;
          if (mode1 && t == 0 && exact)
            for (int k = 64 * tid; k < min(N, 64 * tid + 64); k++)
              changed |= as_global(pd.carry)[k] != (uint8_t)(dv >> (k & 63) & 1u);
          decBits[2 * tid] = lo;
          decBits[2 * tid + 1] = hi;
        }
        if (tid < size * NWS) {
          const int wd = 2 * (tid % NWS);
          if ((uint32_t)pv) atomicXor(&parBits[wd], (uint32_t)pv);
          if ((uint32_t)(pv >> 32)) atomicXor(&parBits[wd + 1], (uint32_t)(pv >> 32));
        }
        if (tid < NWS) parMine[2 * tid] = parMine[2 * tid + 1] = 0u;
        if (changed) s_changed = 1;
      }
      xc++;
      __syncthreads();
    }
    if (rank != 0) {
      __syncthreads();  // s_item is no longer read
      continue;
    }

    // ---- the leader's report, as in bp_persistent_kernel
    int ok = 0;
    if (status == 1) {
      uint32_t crc = 0;
      for (int k = tid; k < N; k += T)
        if ((decBits[k >> 5] >> (k & 31)) & 1u) crc ^= L.crcBasis[k];
      for (int o = 32; o > 0; o >>= 1) crc ^= __shfl_xor(crc, o);
      if (lane == 0) s_crc[wave] = crc;
      __syncthreads();
      uint32_t tot = 0;
      for (int i = 0; i < W; i++) tot ^= s_crc[i];
      ok = tot == pd.crc;
    }
    // decisions are kept for an accepted code, in ParallelMode 1 for every
    // code that ran to its end
    int slot = -1;
    if (ok || (mode1 && status != 3)) {
      if (tid == 0) s_item = atomicAdd(a.slot_count, 1);
      __syncthreads();
      slot = s_item;
      if (slot < a.slot_capacity) {
        uint8_t *dst = a.slots + (size_t)slot * N;
        for (int k = tid; k < N; k += T) dst[k] = (uint8_t)((decBits[k >> 5] >> (k & 31)) & 1u);
      }
    }
    if (tid == 0) {
      pd.rec[level] = make_int4(iters, ok ? REC_ACCEPTED : status == 1 ? REC_CRC_MISMATCH
                                          : status == 3 ? REC_CANCELLED : REC_FAILED, slot, 0);
      if (ok) atomicMin(&st->best, level);
      if (mode1) pd.bcase[level] = bcaseSlot;
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ ParallelMode 1 resolution
// After a speculative ParallelMode 1 launch, walks each bitplane's codes from
// the queue's first code with the decisions actually carried from code to
// code (LdpcaDecoder.cpp:646-771 with beliefPropagation_OpenMP).  A code that
// recorded the repeat case fails after 4 iterations when the carried
// decisions equal its recorded ones; otherwise its speculative outcome
// stands.  The first accepted code becomes `best`.  When the walk reaches a
// code the launch cancelled or never ran, the bitplane is queued again from
// that code with the carried decisions now known (rerun_count counts them).
// One wave per bitplane; the carried decisions are followed by their slot and
// copied once, at the end of the walk (copied byte by byte after every code, 60
// bitplanes took 102 us, now 8).
// A slot index at or beyond slot_capacity (its decisions were not stored),
// for a failed, mismatching or accepted code or a repeat case, adds 1 << 20
// to rerun_count, which the host reports as exhausted slots.
__global__ __launch_bounds__(64) void mode1_resolve_kernel(const PlaneDesc *planes, int nplanes, int numCodes, int N,
                                                           const uint8_t *slots, int slot_capacity, int *rerun_count) {
  const int p = blockIdx.x;
  if (p >= nplanes) return;
  const PlaneDesc d = planes[p];
  PlaneState *st = d.state;
  const int run0 = st->run, lane = threadIdx.x;
  // the decisions carried into code L: the caller's, then a slot's (16-byte words)
  const uint4 *carry = (const uint4 *)d.carry;
  int L = run0, best = numCodes - 1, run = numCodes;
  for (; L < numCodes - 1; L++) {
    const int4 r = d.rec[L];
    if (r.y == REC_NOT_RUN || r.y == REC_CANCELLED) {
      run = L;
      break;
    }
    const int bs = L != run0 ? d.bcase[L] : 0;
    if (bs - 1 >= slot_capacity || r.z < 0 || r.z >= slot_capacity) {  // every record reached here names a slot
      if (lane == 0) atomicAdd(rerun_count, 1 << 20);
      return;
    }
    bool repeat = false;
    if (bs > 0) {
      const uint4 *b = (const uint4 *)(slots + (size_t)(bs - 1) * N);
      uint32_t diff = 0;
      for (int k = lane; k < N / 16; k += 64) {
        const uint4 u = b[k], v = carry[k];
        diff |= (u.x ^ v.x) | (u.y ^ v.y) | (u.z ^ v.z) | (u.w ^ v.w);
      }
      repeat = __ballot(diff != 0) == 0;
    }
    if (!repeat && r.y == REC_ACCEPTED) {
      best = L;
      break;
    }
    const int fin = repeat ? bs - 1 : r.z;
    if (repeat && lane == 0) d.rec[L] = make_int4(4, REC_FAILED, bs - 1, 0);
    carry = (const uint4 *)(slots + (size_t)fin * N);
  }
  // only the decisions carried out of the walk are needed again, by a resumed one
  if (carry != (const uint4 *)d.carry)
    for (int k = lane; k < N / 16; k += 64) ((uint4 *)d.carry)[k] = carry[k];
  if (lane == 0) {
    st->best = best;  // numCodes - 1 with every BP code failed: full-rate inverse
    st->run = run;
    if (run < numCodes) atomicAdd(rerun_count, 1);
  }
}

// ------------------------------------------------------------------ full rate
// invH_mul (LdpcaDecoder.cpp:624-643) for every bitplane whose BP codes all
// failed.  Bitplane p's product goes to decision slot slot0 + p, a range the BP
// launches do not hand out, so the bitplanes that need one are not counted first
// (that took a launch of its own, 4.6 us in every bitplane step).
// Grid (ceil(N / INVH_ROWS), INVH_COLS).  Every wave finds the bitplanes that
// need the inverse with a ballot over the plane list; column y takes the
// k-th of them for k = y, y + INVH_COLS, ...  Workgroup x computes rows
// [x * INVH_ROWS, + INVH_ROWS) of the product, INVH_ROWS / 4 per wave: a row
// of invH (N bits, MSB-first bytes, rows padded to 32-bit words) is read as
// little-endian words by consecutive lanes, ANDed with the byte-swapped
// syndrome words (a common byte permutation leaves the parity of the AND
// unchanged), and the parity is the popcount of the wave's ballot.
constexpr int INVH_ROWS = 64, INVH_COLS = 8, INVH_THREADS = 256;
constexpr int INVH_MAX_WORDS = (6336 + 31) / 32;  // <= 4 words per lane

__global__ __launch_bounds__(INVH_THREADS) void invh_kernel(const PlaneDesc *planes, int nplanes, LadderDev L,
                                                            uint8_t *slots, int slot0) {
  __shared__ uint32_t sw[INVH_MAX_WORDS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int N = L.N, nw = (N + 31) / 32, C = L.numCodes;
  const int row0 = blockIdx.x * INVH_ROWS + wave * (INVH_ROWS / 4);
  int k = 0;  // bitplanes needing the inverse seen so far (wave-uniform)
  for (int base = 0; base < nplanes; base += 64) {
    const int p = base + lane;
    const bool need = p < nplanes && !(planes[p].state->best < C - 1);
    uint64_t mask = __ballot(need);
    while (mask) {
      const int b = base + __builtin_ctzll(mask);
      mask &= mask - 1;
      if (k++ % INVH_COLS != (int)blockIdx.y) continue;
      const PlaneDesc d = planes[b];
      gbyte_t *acc = as_global(d.acc);
      // full-rate syndrome s_k = a_k ^ a_{k-1} (identity transmission pattern),
      // as MSB-first 32-bit words, bits at k >= N cleared
      __syncthreads();  // the previous bitplane's words are no longer read
      for (int t = tid; t < nw; t += INVH_THREADS) {
        uint32_t a = 0;
        for (int q = 0; q < 4; q++) {
          const int byte = 4 * t + q;
          a = (a << 8) | (byte < N / 8 ? (uint32_t)acc[byte] : 0u);
        }
        const uint32_t prev = t > 0 ? (uint32_t)acc[4 * t - 1] & 1u : 0u;
        uint32_t s = a ^ (a >> 1) ^ (prev << 31);
        const int valid = N - 32 * t;
        if (valid < 32) s &= ~0u << (32 - valid);
        sw[t] = __builtin_bswap32(s);
      }
      __syncthreads();
      uint32_t w[4];
#pragma unroll
      for (int q = 0; q < 4; q++) w[q] = lane + 64 * q < nw ? sw[lane + 64 * q] : 0u;
      if (blockIdx.x == 0 && tid == 0) d.rec[C - 1] = make_int4(0, REC_ACCEPTED, slot0 + b, 1);
      uint8_t *dst = slots + (size_t)(slot0 + b) * N;
      uint32_t mine = 0;  // parity of row row0 + lane (lane < INVH_ROWS / 4)
#pragma unroll 4
      for (int i = 0; i < INVH_ROWS / 4; i++) {
        const int j = row0 + i;
        if (j >= N) break;  // wave-uniform
        const uint32_t *row = (const uint32_t *)(L.invH + (size_t)j * nw * 4);
        uint32_t x = 0;
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (lane + 64 * q < nw) x ^= as_global(row)[lane + 64 * q] & w[q];
        const uint32_t par = __popcll(__ballot(__popc(x) & 1u)) & 1u;
        if (lane == i) mine = par;
      }
      if (lane < INVH_ROWS / 4 && row0 + lane < N) dst[row0 + lane] = (uint8_t)mine;
    }
  }
}

// One workgroup per bitplane: its accepted code's decisions from their slot
// to out + p * N (16-byte words; slots and out are 16-byte aligned).
__global__ void gather_accepted_kernel(const PlaneDesc *planes, int nplanes, int N, const uint8_t *slots,
                                       int slot_capacity, uint8_t *out) {
  const int p = blockIdx.x;
  if (p >= nplanes) return;
  const PlaneDesc d = planes[p];
  const int best = d.state->best;
  if (best < 0) return;
  const int4 r = d.rec[best];
  if (r.y != REC_ACCEPTED || r.z < 0 || r.z >= slot_capacity) return;
  const uint4 *src = (const uint4 *)(slots + (size_t)r.z * N);
  uint4 *dst = (uint4 *)(out + (size_t)p * N);
  for (int i = threadIdx.x; i < N / 16; i += blockDim.x) dst[i] = src[i];
}

// Clears n ints (instead of hipMemsetAsync, so that a captured step holds kernel
// nodes only).
__global__ void zero_ints_kernel(int *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Waits for flag[0] for at most 200 us and says in flag[1 + which] whether it came.
__global__ void await_flag_kernel(int *flag, int which) {
  const uint64_t t0 = wall_clock64();  // 100 MHz
  int seen = 0;
  while (!seen && wall_clock64() - t0 < 20000) seen = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  flag[1 + which] = seen;
}
__global__ void raise_flag_kernel(int *flag) {
  __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ------------------------------------------------------------------ host side
// The runtime spreads streams over a few hardware queues (four by default), and
// kernels of two streams on the same queue run one after the other: 60 mixed
// bitplanes, whose two launches share the CUs, took 2.5 ms on such a pair and 1.55
// on others.  So a stream that is to run beside others is tried: a kernel on each
// of them waits for one on the new stream (and gives up after 200 us).  The streams
// tried meanwhile are kept, so that the next one lands on another queue, eight at
// most; the one that ran beside with[0], then beside the most of the others, stays.
hipError_t create_stream_beside(const hipStream_t *with, int n, hipStream_t *out, uint32_t *beside) {
  constexpr int kTries = 8;
  if (n < 1 || n > kBesideMax) return hipErrorInvalidValue;
  const uint32_t all = (1u << n) - 1;
  hipStream_t tried[kTries] = {};
  int *flag = nullptr, got[1 + kBesideMax] = {}, made = 0, best = 0;
  uint32_t bestMask = 0;
  *out = nullptr;
  hipError_t e = hipMalloc((void **)&flag, sizeof(got));
  while (e == hipSuccess && made < kTries && bestMask != all) {
    hipStream_t t;
    if ((e = hipStreamCreateWithFlags(&t, hipStreamNonBlocking)) != hipSuccess) break;
    tried[made++] = t;
    if ((e = launch_zero_ints(flag, 1 + n, t)) == hipSuccess) e = hipStreamSynchronize(t);
    if (e != hipSuccess) break;
    for (int k = 0; k < n; k++) hipLaunchKernelGGL(await_flag_kernel, dim3(1), dim3(1), 0, with[k], flag, k);
    hipLaunchKernelGGL(raise_flag_kernel, dim3(1), dim3(1), 0, t, flag);
    e = hipGetLastError();
    const hipError_t et = hipStreamSynchronize(t);
    if (e == hipSuccess) e = et;
    for (int k = 0; k < n; k++) {
      const hipError_t ek = hipStreamSynchronize(with[k]);
      if (e == hipSuccess) e = ek;
    }
    if (e == hipSuccess) e = hipMemcpy(got, flag, sizeof(got), hipMemcpyDeviceToHost);
    if (e != hipSuccess) break;
    uint32_t mask = 0;
    for (int k = 0; k < n; k++) mask |= got[1 + k] ? 1u << k : 0u;
    auto score = [](uint32_t m) { return (m & 1u) * 64 + (uint32_t)__builtin_popcount(m); };
    if (score(mask) > score(bestMask)) {
      best = made - 1;
      bestMask = mask;
    }
  }
  // with no more streams or memory to be had, the best one so far will do
  if (made > 0) {
    *out = tried[best];
    if (e != hipSuccess) (void)hipGetLastError();
    e = hipSuccess;
  }
  for (int k = 0; k < made; k++)
    if (k != best) (void)hipStreamDestroy(tried[k]);
  if (flag) (void)hipFree(flag);
  if (beside) *beside = bestMask;
  return e;
}

hipError_t launch_mode1_resolve(const PlaneDesc *planes, int n, int numCodes, int N, const uint8_t *slots,
                                int slot_capacity, int *rerun_count, hipStream_t s) {
  hipLaunchKernelGGL(mode1_resolve_kernel, dim3(n), dim3(64), 0, s, planes, n, numCodes, N, slots, slot_capacity,
                     rerun_count);
  return hipGetLastError();
}

hipError_t launch_zero_ints(int *p, int n, hipStream_t s) {
  hipLaunchKernelGGL(zero_ints_kernel, dim3((n + 63) / 64), dim3(64), 0, s, p, n);
  return hipGetLastError();
}

template <int N, int T>
static hipError_t launch_bp(const BpArgs &a, int grid, hipStream_t s) {
  if (a.mode == 1) hipLaunchKernelGGL((bp_persistent_kernel<N, T, true>), dim3(grid), dim3(T), 0, s, a);
  else hipLaunchKernelGGL((bp_persistent_kernel<N, T, false>), dim3(grid), dim3(T), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_bp_any(int N, int threads, const BpArgs &a, int grid, hipStream_t s) {
  if (!a.lad.regular) return launch_bp_irregular(a, grid, s);
  if (N == 6336) {
    if (threads == 704) return launch_bp<6336, 704>(a, grid, s);
    if (threads == 512) return launch_bp<6336, 512>(a, grid, s);
    return launch_bp<6336, 1024>(a, grid, s);
  }
  if (threads == 1024) return launch_bp<1584, 1024>(a, grid, s);
  if (threads == 512) return launch_bp<1584, 512>(a, grid, s);
  return launch_bp<1584, 256>(a, grid, s);
}

hipError_t launch_bp_split(int N, const BpArgs &a, int clusters, hipStream_t s) {
  if (N != 6336 || !a.lad.regular || a.max_iter < 1 || a.split < 2 || a.split > kSplitMax || clusters < 1 || clusters > kSplitClusters || !a.area)
    return hipErrorInvalidValue;
  if (!a.area_clear) {
    const hipError_t e = launch_zero_ints((int *)a.area, kSplitCtlWords, s);
    if (e != hipSuccess) return e;
  }
  const dim3 grid(clusters * a.split);
  if (a.mode == 1) hipLaunchKernelGGL((bp_split_kernel<6336, 1024, true>), grid, dim3(1024), 0, s, a);
  else hipLaunchKernelGGL((bp_split_kernel<6336, 1024, false>), grid, dim3(1024), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_ce_llr(const PlaneDesc *d_planes, int n, int fixed_start, const Ladder &l1584,
                         const Ladder &l6336, int *counters, uint32_t *area, hipStream_t s) {
  static_assert(kSplitCtlWords % 4 == 0, "cleared in quads");
  const int quads = area ? kSplitCtlWords / 4 : 0;
  hipLaunchKernelGGL(ce_llr_kernel, dim3(n + (quads + CE_T - 1) / CE_T), dim3(CE_T), 0, s, d_planes, n, fixed_start,
                     l1584.d_codeRate, l6336.d_codeRate, l1584.numCodes, l6336.numCodes, counters, (uint4 *)area,
                     quads);
  return hipGetLastError();
}

hipError_t launch_invh(const PlaneDesc *d_planes, int n, const LadderDev &L, uint8_t *slots, int slot0,
                       hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(invh_kernel, dim3((L.N + INVH_ROWS - 1) / INVH_ROWS, INVH_COLS), dim3(INVH_THREADS), 0, s,
                     d_planes, n, L, slots, slot0);
  return hipGetLastError();
}

hipError_t launch_gather_accepted(const PlaneDesc *d_planes, int n, int N, const uint8_t *slots, int slot_capacity,
                                  uint8_t *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(gather_accepted_kernel, dim3(n), dim3(128), 0, s, d_planes, n, N, slots, slot_capacity, out);
  return hipGetLastError();
}

LadderDev ladder_dev(const Ladder &L) {
  LadderDev d;
  d.N = L.N; d.E = L.E; d.numCodes = L.numCodes;
  d.regular = L.regular ? 1 : 0;
  d.colRows = L.d_colRows; d.rowPtr = L.d_rowPtr; d.tx = L.d_tx;
  d.slotEdges = L.d_slotEdges; d.jc = L.d_jc; d.colSlots = L.d_colSlots;
  d.syndLength = L.d_syndLength; d.invH = L.d_invH; d.crcBasis = L.d_crcBasis;
  return d;
}

}  // namespace dvc
