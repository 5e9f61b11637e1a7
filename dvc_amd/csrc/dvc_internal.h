// dvc_internal.h -- shared host-side state of the gfx950 decoding library.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <functional>
#include <mutex>
#include <string>
#include <vector>
#include "../../include/dvc_accel.h"

namespace dvc {
struct ColEdges;  // ldpca_kernels.h
}

namespace dvc {

void set_error(const std::string &msg);

#define DVC_HIP(call)                                                                  \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess) {                                                            \
      dvc::set_error(std::string(#call) + ": " + hipGetErrorString(e_));               \
      return DVC_EDEVICE;                                                              \
    }                                                                                  \
  } while (0)

#define DVC_CHECK(cond, code, msg)                                                     \
  do {                                                                                 \
    if (!(cond)) { dvc::set_error(msg); return (code); }                               \
  } while (0)

// Host copy of one ladder (all codes of one code length) and its device image.
struct Ladder {
  int N = 0, E = 0, period = 0, numCodes = 0;
  bool regular = true;             // every column has degree 3 (the Reg*.lad ladders)
  std::vector<int> jc;             // N+1 column pointers
  std::vector<int> encIr;          // E encoder rows
  std::vector<int> bitsPerPeriod;  // numCodes
  std::vector<int> idx;            // numCodes*period
  std::vector<int> syndLength;     // numCodes
  std::vector<float> codeRate;     // numCodes
  std::vector<int> decIr;          // numCodes*E decoder rows per edge
  std::vector<uint8_t> invH;       // N * invRowBytes, MSB-first
  int invRowBytes = 0;             // 4*ceil(N/32)
  std::vector<uint8_t> crcBasis;   // N: CRC-8 of the message with only bit k set

  // Device image, per BP code c (0..numCodes-2):
  //   d_colRows[c*N + k]       column k's edges 3k..3k+2, one word each:
  //                            row | slot << 15, slot = the edge's message
  //                            position in row order (rowPtr[row] + its rank
  //                            among the row's edges in ascending edge order)
  //   d_rowPtr[c*(N+1) + r]    number of edges in rows below r (r <= m): row
  //                            r's messages sit at rowPtr[r] + rank
  //   d_tx[c*N + k]            accumulated-syndrome position of syndrome bit k
  ColEdges *d_colRows = nullptr;
  // Irregular ladders (column degrees differ) instead of d_colRows:
  //   d_slotEdges[c*E + s]  message slot s (row order) as row | column << 13
  //   d_jc[k]               column pointers (N+1)
  //   d_colSlots[c*E + l]   edge l's message slot (l in column order)
  uint32_t *d_slotEdges = nullptr;
  int *d_jc = nullptr;
  uint16_t *d_colSlots = nullptr;
  uint16_t *d_rowPtr = nullptr, *d_tx = nullptr;
  int *d_syndLength = nullptr;
  float *d_codeRate = nullptr;
  uint8_t *d_invH = nullptr, *d_crcBasis = nullptr;
};

// Loads dir/<kind><N>.ladder (kind "reg" or "irreg") and its cached inverse.
int load_ladder(const std::string &dir, const char *kind, int N, Ladder &L);
// BP launch shape: threads per workgroup for a launch of `planes` bitplanes, and
// the persistent grid for its `items` queued (bitplane, code) items beside a
// concurrent launch of `other` bitplanes of the other code length (the context's
// tuning, but for small QCIF launches).
int bp_threads(const dvc_ctx *c, int N, int planes);
int bp_grid(const dvc_ctx *c, int N, int items, int planes, int other);
// Whether a batch of `planes` bitplanes of one length runs in the launch shape that
// the tuning names; fewer bitplanes run split or with 1024 threads, and an irregular
// ladder has one shape.
bool bp_tuned(const dvc_ctx *c, int N, int planes);
// The BP launch of `planes` bitplanes' queued items (a.total of them): persistent,
// or split over several workgroups per codeword when a.area is given and the
// launch would leave most CUs idle.  lanes: launches like it that other streams
// issue at the same time.  sequential: codes one after another.
struct BpArgs;
hipError_t launch_bp(const dvc_ctx *c, int N, int planes, int other, int lanes, bool sequential, const BpArgs &a,
                     hipStream_t s);
int upload_ladder(Ladder &L);
// Quantisation table entry Qtable[q][index] (reconstruction.cpp:9-78), 0 outside 1..8 x 0..15.
int qtable_entry(int q, int index);
// QuantizationTableBits[q][index] (reconstruction.cpp:44-53) and zigzag[band] (global.cpp:36-41).
int qbits_entry(int q, int index);
int zigzag_entry(int band);
// Motion-cost factor tables of the context (made on first use).
int ensure_cost_tables(dvc_ctx *c);
// Per-band entry points' device state (band.hip), freed with the context.
struct BandState;
void band_free(dvc_ctx *c);
// Looks up the allocation-free entry point's scratch array on the context's
// (current) device, once per device (noalloc.hip).
int noalloc_attach(dvc_ctx *c);
void free_ladder(Ladder &L);
// Host copies of the entry points that take host buffers, on up to eight threads
// (host_pool.cpp), and pinned staging kept between calls.
struct HostPool;
struct HostCopy { void *dst; const void *src; size_t bytes; };
void host_parallel(dvc_ctx *c, size_t n, size_t bytes, const std::function<void(size_t)> &fn);
void host_copy(dvc_ctx *c, const std::vector<HostCopy> &list);
void host_pool_free(dvc_ctx *c);
// Device memory to a caller's buffer through pinned memory of the same size,
// the copies out overlapping the transfers; returns when all is there.
int copy_back(dvc_ctx *c, hipStream_t s, void *user, const void *dev, uint8_t *pinned, size_t bytes);
// Pinned host block of at least `bytes` in *p (grown, contents dropped).
int pinned_grow(uint8_t **p, size_t *have, size_t bytes);

}  // namespace dvc

struct dvc_ctx;
// Per-kernel timing with HIP events recorded on the launching stream.
struct KernelTimer {
  std::string name;
  double total_ms = 0.0;
  long launches = 0;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> pending;
};

struct dvc_ctx {
  bool profiling = false;
  std::vector<KernelTimer> timers;
  std::mutex timer_mu;  // engine lanes launch from several host threads
  // Records start/stop events around a launch when profiling is on.
  hipEvent_t timer_begin(const char *name, hipStream_t s, int *slot);
  void timer_end(int slot, hipEvent_t start, hipStream_t s);
  void timer_collect();

  int device = 0;
  int sm_count = 256;
  double *d_costFme = nullptr, *d_costUsi = nullptr;  // motion-cost factor tables
  int max_iter = 50;
  // BP launch configuration (dvc_autotune / dvc_set_tuning): threads per
  // workgroup for each code length, QCIF workgroups per CU, and the interval
  // in iterations at which a running speculative item polls for cancellation
  // (defaults: dvc_autotune's choices on MI355X)
  int bp_threads_cif = 1024;
  int bp_threads_qcif = 512;
  int bp_wg_per_cu_qcif = 4;
  int bp_poll = 1;
  int bp_mode = 0;  // 0: ParallelMode 0 BP semantics, 1: ParallelMode 1 (early jump on repeated decisions)
  int rate_step = 0;  // 1: DYNAMICSTEP rate search (dvc_params.rate_step)
  dvc::Ladder lad1584, lad6336;
  hipStream_t stream = nullptr;
  void *si_scratch = nullptr;  // dvc_side_info_batch's device buffers, kept between calls
  size_t si_scratch_bytes = 0;
  uint8_t *si_host = nullptr;  // its pinned host staging, and the per-band entry points'
  size_t si_host_bytes = 0;
  dvc::HostPool *pool = nullptr;  // host copy threads (made on first use)
  // the LDPCA entry points' workspaces, one per code length (1584, 6336), kept
  // between calls: device memory and pinned staging (inputs up, results back)
  struct LdWork {
    void *dev = nullptr, *host = nullptr;
    size_t devBytes = 0, hostBytes = 0;
  } ld[2];
  hipStream_t stream2 = nullptr;  // the second code length of a mixed batch (made with the first one)
  void *noalloc_scratch = nullptr;  // device address of noalloc.hip's scratch array on this device
  dvc::BandState *band = nullptr;   // per-band entry points' frame state (dvc_band_frame_init)
  dvc::Ladder *ladder(int N) { return N == 1584 ? &lad1584 : (N == 6336 ? &lad6336 : nullptr); }
};
