// ldpca_kernels.h -- argument blocks shared by the LDPCA kernels and their
// host-side launchers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "rate_search.h"

namespace dvc {

struct Ladder;

// Per-bitplane mutable state on the device.
struct PlaneState {
  int start;      // nCodeStart (-1: computed by the CE kernel)
  int best;       // lowest code that converged with a matching CRC (numCodes-1 = none)
  float entropy;  // H(X|Y) from ComputeCE
  int run;        // first code of the current launch's queue (start, or the code a
                  // ParallelMode 1 resolution resumes at; numCodes = nothing left)
  int taint;      // 1: some LLR of the bitplane is NaN (set by the CE kernel): a likelihood
                  // ratio condBitProb formed as 0/0 when both of a block's interval sums
                  // underflow to zero (noiseModel.cpp:295-303)
};

struct PlaneDesc {
  int N;
  const float *LR;     // N likelihood ratios
  float *LLR;          // N log-likelihood ratios (written by the CE kernel)
  const uint8_t *acc;  // N/8 accumulated-syndrome bytes
  uint32_t crc;        // encoder CRC-8
  PlaneState *state;
  int4 *rec;           // [numCodes] per code: iterations, status, decision slot, used_inverse
  // ParallelMode 1 only (NULL otherwise):
  uint8_t *carry;      // N decision bytes carried into code `run` (any byte other than 0/1 never matches)
  int *bcase;          // [numCodes] decision slot + 1 of a code's iteration-3 decisions when they
                       // repeat its first three (see bp_persistent_kernel), else 0
};

// What k_put_bitplane needs to find the accepted decisions of a bitplane.
struct BpFrameLink {
  const PlaneState *state;
  const int4 *records;
  const uint8_t *slots;
  int slot_capacity;
  uint8_t *carry;  // ParallelMode 1: receives the accepted decisions (the next bitplane's carry)
};

// Run records per bitplane in the frame decoder's buffers: the most codes a
// ladder has (the irregular QCIF ladder's 66; the regular ladders have 65).
constexpr int kMaxCodes = 66;

// A degree-3 column's edges for the BP kernel: row | message slot << 15 each.
struct ColEdges {
  uint32_t e[3];
};

struct LadderDev {
  int N, E, numCodes;
  int regular;           // every column has degree 3 (colRows), else slotEdges/jc/colSlots
  const ColEdges *colRows;  // per code and column: its three edges as row | message slot << 15
  const uint32_t *slotEdges;  // irregular: per code and message slot (row order) row | column << 13
  const int *jc;              // irregular: column pointers
  const uint16_t *colSlots;   // irregular: per code and edge (column order) its message slot
  const uint16_t *rowPtr, *tx;
  const int *syndLength;
  const uint8_t *invH, *crcBasis;
};

struct BpArgs {
  LadderDev lad;
  const PlaneDesc *planes;
  int nplanes;
  int *next;          // queue head (reset to 0 before a launch)
  int total;          // nplanes * max_offset
  int max_offset;     // codes above start tried per bitplane
  int max_iter;
  uint8_t *slots;     // accepted decisions, N bytes per slot
  int *slot_count;
  int slot_capacity;
  int poll;           // iterations between polls of the bitplane's best code (>= 1)
  int mode;           // 0: beliefPropagation, 1: beliefPropagation_OpenMP (ParallelMode 1)
  int rate_step;      // 1: only the codes the DYNAMICSTEP search tries (dynstep_tries)
  // a launch that splits its codewords over up to `split` workgroups (0, 1: none):
  // the area of split_area_words(N) words that they meet in, its first
  // kSplitCtlWords cleared before the launch, by the launch itself unless
  // area_clear says that launch_ce_llr did it and none has used it since
  int split = 0;
  uint32_t *area = nullptr;
  int area_clear = 0;
};

// Split BP (bp_split_kernel): at most kSplitMax workgroups per codeword and
// kSplitClusters codewords at a time; per cluster a control block of kCtlWords
// words, cleared before a launch (block 0 hands out the tickets), then two
// exchange buffers.
constexpr int kSplitMax = 8, kSplitClusters = 64, kCtlWords = 256;
constexpr int kSplitCtlWords = kCtlWords * (kSplitClusters + 1);
constexpr size_t split_buf_words(int N) {  // messages, decisions, every member's parities
  return (size_t)3 * N + (kSplitMax + 1) * 2 * ((N + 63) / 64);
}
constexpr size_t split_area_words(int N) { return kSplitCtlWords + (size_t)kSplitClusters * 2 * split_buf_words(N); }

// Decision slots of a launch of n bitplanes over C codes.  The BP kernel hands
// out the first `bp` of them: ParallelMode 0 accepts each (bitplane, code) at
// most once, and a bitplane that accepts code C - 1 does so through the inverse;
// ParallelMode 1 keeps every run code's decisions and its repeat-case decisions.
// The n after them are the bitplanes' inverse slots.
struct SlotPlan { int bp, total; };
inline SlotPlan slot_plan(int n, int C, int mode) {
  return mode == 1 ? SlotPlan{2 * C * n + 1, 2 * C * n + 1 + n} : SlotPlan{(C - 1) * n + 1, C * n + 1};
}

LadderDev ladder_dev(const Ladder &L);
hipError_t launch_bp_any(int N, int threads, const BpArgs &a, int grid, hipStream_t s);
// The split form of a launch on a regular ladder: clears the area's control
// blocks if they are not, then `clusters` groups of a.split workgroups.
hipError_t launch_bp_split(int N, const BpArgs &a, int clusters, hipStream_t s);
hipError_t launch_zero_ints(int *p, int n, hipStream_t s);
// A non-blocking stream whose kernels run beside those of the n streams `with`, or,
// where the hardware queues do not suffice, beside with[0] and as many of the
// others as can be.  Bit k of *beside (may be NULL): it runs beside with[k].
constexpr int kBesideMax = 31;
hipError_t create_stream_beside(const hipStream_t *with, int n, hipStream_t *out, uint32_t *beside);
hipError_t launch_mode1_resolve(const PlaneDesc *planes, int n, int numCodes, int N, const uint8_t *slots,
                                int slot_capacity, int *rerun_count, hipStream_t s);
// Entropy, LLRs and start codes of n bitplanes; also clears the three launch
// counters (queue head, decision slots handed out, bitplanes to resume) and, if
// there is one, the control blocks of the area of a split BP launch (16-byte
// aligned).
hipError_t launch_ce_llr(const PlaneDesc *d_planes, int n, int fixed_start, const Ladder &l1584,
                         const Ladder &l6336, int *counters, uint32_t *area, hipStream_t s);
// BP on an irregular ladder (bp_irregular_kernel).
hipError_t launch_bp_irregular(const BpArgs &a, int grid, hipStream_t s);
// Full-rate inverse of the bitplanes whose BP codes all failed, bitplane p's
// into decision slot slot0 + p.
hipError_t launch_invh(const PlaneDesc *d_planes, int n, const LadderDev &L, uint8_t *slots, int slot0,
                       hipStream_t s);
// Copies bitplane p's accepted decisions (N bytes, N a multiple of 16) to
// out + p * N for every p < n; one with no accepted record in range is skipped.
hipError_t launch_gather_accepted(const PlaneDesc *d_planes, int n, int N, const uint8_t *slots, int slot_capacity,
                                  uint8_t *out, hipStream_t s);

}  // namespace dvc
