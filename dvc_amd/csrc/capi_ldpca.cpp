// capi_ldpca.cpp -- context management and the LDPCA entry points of
// include/dvc_accel.h.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <dlfcn.h>
#include <string>
#include <vector>
#include <algorithm>
#include "dvc_internal.h"
#include "host_pair.h"
#include "ldpca_kernels.h"

namespace dvc {

static thread_local std::string g_err;
void set_error(const std::string &msg) { g_err = msg; }

// Directory of this shared library's data files: <lib dir>/data.
static std::string default_data_dir() {
  Dl_info info;
  if (dladdr((void *)&default_data_dir, &info) && info.dli_fname) {
    std::string p(info.dli_fname);
    size_t s = p.find_last_of('/');
    if (s != std::string::npos) return p.substr(0, s) + "/data";
  }
  return "data";
}

int bp_threads(const dvc_ctx *c, int N, int planes) {
  if (N != 1584) return c->bp_threads_cif;
  // A QCIF launch whose bitplanes need fewer codewords than there are CUs (about
  // eight codes each; the searches try 5 on average, rarely more than 12) is bound
  // by one codeword's latency, which 16 waves cut by a tenth; more bitplanes run
  // faster with several smaller workgroups per CU.  ms with 512 and 1024 threads:
  // 1 bitplane 0.307 and 0.276, 8 0.399 and 0.373, 32 0.56 and 0.48, 64 0.776 and
  // 0.804, 128 1.30 and 1.37, 256 2.33 and 2.50.
  if (8 * planes <= c->sm_count) return 1024;
  return c->bp_threads_qcif;
}

// CUs of a launch beside a concurrent one of `other` bitplanes of the other code
// length.  Two launches at once that fill the chip for a round or two of codes
// (eight per bitplane) share its CUs by their work: a CIF codeword's iteration
// takes four times a QCIF one's, 2.5 times an irregular one's.  Either would take
// all CUs for its speculative codes and the other wait for the last of them (60
// mixed bitplanes 2.20 ms, shared 1.65).  Larger pairs keep full grids: the second
// fills the CUs that the first one's tail leaves, where a share would idle (512
// bitplanes 19.0 ms shared, 15.4 so, 16.1 one after the other).
static int launch_cus(const dvc_ctx *c, int N, int planes, int other) {
  if (other <= 0) return c->sm_count;
  const double cif = N == 6336 ? planes : other, qcif = N == 6336 ? other : planes;
  const double wq = qcif * (c->lad1584.regular ? 0.25 : 0.4), part = (N == 6336 ? cif : wq) / (cif + wq);
  if (8 * (cif + wq) > 2 * c->sm_count) return c->sm_count;
  return std::max(1, std::min(c->sm_count - 1, (int)(c->sm_count * part + 0.5)));
}

int bp_grid(const dvc_ctx *c, int N, int items, int planes, int other) {
  // a CIF codeword takes 126 KB of a CU's 160 KB LDS, an irregular QCIF codeword's
  // 16 waves its registers; regular QCIF codewords (38 KB, 8 waves) share one
  const int perCU = N == 6336 || !c->lad1584.regular ? 1 : c->bp_wg_per_cu_qcif;
  return std::max(1, std::min(launch_cus(c, N, planes, other) * perCU, items));
}

// Workgroups per CIF codeword (1: the persistent kernel).  A launch's CUs are
// shared among the codewords its bitplanes need (about eight each), up to the
// eight that a codeword can use.  Four per codeword still pay when a quarter of
// the codes has to wait for a cluster (10 bitplanes, unsplit 0.93 ms a batch: 4
// workgroups 0.66, 3 0.74, 2 0.86); with more than that waiting the gain is gone or
// hangs on how many codes the bitplanes need (16: 0.91 against 0.99, 20: 1.12
// against 1.02).  One bitplane: 0.84 unsplit, 0.48 with 4, 0.42 with 8.  A QCIF
// codeword's iteration is shorter than an exchange between workgroups: never.
static int split_width(int cus, int codewords) {
  if (3 * codewords > cus) return 1;
  return std::max(4, std::min(kSplitMax, cus / codewords));
}
static int bp_split(const dvc_ctx *c, int N, int planes, int other, int lanes, bool sequential, const BpArgs &a) {
  if (!a.area || N != 6336 || !a.lad.regular || a.max_iter < 1) return 1;
  return split_width(launch_cus(c, N, planes, other) / lanes, sequential ? 1 : 8 * planes);
}

bool bp_tuned(const dvc_ctx *c, int N, int planes) {
  if (N == 6336) return split_width(c->sm_count, 8 * planes) == 1;
  return c->lad1584.regular && bp_threads(c, N, planes) == c->bp_threads_qcif;
}

hipError_t launch_bp(const dvc_ctx *c, int N, int planes, int other, int lanes, bool sequential, const BpArgs &a,
                     hipStream_t s) {
  const int split = bp_split(c, N, planes, other, lanes, sequential, a);
  if (split > 1) {
    BpArgs b = a;
    b.split = split;
    const int fit = launch_cus(c, N, planes, other) / lanes / split;
    return launch_bp_split(N, b, sequential ? 1 : std::max(1, std::min({kSplitClusters, fit, a.total})), s);
  }
  return launch_bp_any(N, bp_threads(c, N, sequential ? 1 : planes), a,
                       sequential ? 1 : bp_grid(c, N, a.total, planes, other), s);
}

}  // namespace dvc

using namespace dvc;

hipEvent_t dvc_ctx::timer_begin(const char *name, hipStream_t s, int *slot) {
  *slot = -1;
  if (!profiling) return nullptr;
  std::lock_guard<std::mutex> lock(timer_mu);
  int k = -1;
  for (size_t i = 0; i < timers.size(); i++)
    if (timers[i].name == name) { k = (int)i; break; }
  if (k < 0) { timers.push_back(KernelTimer{name}); k = (int)timers.size() - 1; }
  hipEvent_t e;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  (void)hipEventRecord(e, s);
  *slot = k;
  return e;
}

void dvc_ctx::timer_end(int slot, hipEvent_t start, hipStream_t s) {
  if (slot < 0 || !start) return;
  hipEvent_t e;
  if (hipEventCreate(&e) != hipSuccess) return;
  (void)hipEventRecord(e, s);
  std::lock_guard<std::mutex> lock(timer_mu);
  timers[slot].pending.push_back({start, e});
}

void dvc_ctx::timer_collect() {
  std::lock_guard<std::mutex> lock(timer_mu);
  for (auto &t : timers) {
    for (auto &pe : t.pending) {
      float ms = 0.0f;
      if (hipEventSynchronize(pe.second) == hipSuccess && hipEventElapsedTime(&ms, pe.first, pe.second) == hipSuccess) {
        t.total_ms += ms;
        t.launches++;
      }
      (void)hipEventDestroy(pe.first);
      (void)hipEventDestroy(pe.second);
    }
    t.pending.clear();
  }
}

// Timed launch helper: TIMED(ctx, "name", stream, expr-returning-hipError_t)
#define TIMED(c, name, s, expr)                                  \
  do {                                                           \
    int slot_;                                                   \
    hipEvent_t ev_ = (c)->timer_begin(name, s, &slot_);          \
    DVC_HIP(expr);                                               \
    (c)->timer_end(slot_, ev_, s);                               \
  } while (0)

extern "C" {

const char *dvc_last_error(void) { return g_err.c_str(); }

int dvc_ctx_create(const dvc_params *params, dvc_ctx **out) {
  DVC_CHECK(out != nullptr, DVC_EINVAL, "dvc_ctx_create: out is NULL");
  *out = nullptr;
  dvc_params p{};
  if (params) p = *params;
  DVC_CHECK(p.parallel_mode == 0 || p.parallel_mode == 1, DVC_EINVAL, "dvc_ctx_create: parallel_mode must be 0 or 1");
  DVC_CHECK(p.rate_step == 0 || (p.rate_step == 1 && p.parallel_mode == 0), DVC_EINVAL,
            "dvc_ctx_create: rate_step must be 0, or 1 with parallel_mode 0");
  DVC_CHECK(p.qcif_ladder == 0 || p.qcif_ladder == 1, DVC_EINVAL, "dvc_ctx_create: qcif_ladder must be 0 or 1");
  int ndev = 0;
  DVC_HIP(hipGetDeviceCount(&ndev));
  DVC_CHECK(ndev > 0 && p.device >= 0 && p.device < ndev, DVC_EDEVICE, "dvc_ctx_create: no such HIP device");
  DVC_HIP(hipSetDevice(p.device));
  hipDeviceProp_t prop;
  DVC_HIP(hipGetDeviceProperties(&prop, p.device));
  DVC_CHECK(strncmp(prop.gcnArchName, "gfx950", 6) == 0, DVC_EDEVICE,
            std::string("dvc_ctx_create: this library is built for gfx950, device is ") + prop.gcnArchName);
  dvc_ctx *c = new dvc_ctx();
  c->device = p.device;
  c->max_iter = p.max_iter > 0 ? p.max_iter : 50;
  if (p.bp_threads > 0) c->bp_threads_cif = p.bp_threads;
  c->bp_mode = p.parallel_mode;
  c->rate_step = p.rate_step;
  c->sm_count = prop.multiProcessorCount;
  std::string dir = p.data_dir ? std::string(p.data_dir) : default_data_dir();
  int rc;
  if ((rc = load_ladder(dir, p.qcif_ladder ? "irreg" : "reg", 1584, c->lad1584)) ||
      (rc = load_ladder(dir, "reg", 6336, c->lad6336)) ||
      (rc = upload_ladder(c->lad1584)) || (rc = upload_ladder(c->lad6336))) {
    dvc_ctx_destroy(c);
    return rc;
  }
  hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e != hipSuccess) { dvc_ctx_destroy(c); set_error("hipStreamCreate failed"); return DVC_EDEVICE; }
  if ((rc = noalloc_attach(c))) {
    dvc_ctx_destroy(c);
    return rc;
  }
  *out = c;
  return DVC_OK;
}

int dvc_ctx_destroy(dvc_ctx *c) {
  if (!c) return DVC_OK;
  (void)hipSetDevice(c->device);
  free_ladder(c->lad1584);
  free_ladder(c->lad6336);
  if (c->d_costFme) (void)hipFree(c->d_costFme);
  if (c->d_costUsi) (void)hipFree(c->d_costUsi);
  if (c->si_scratch) (void)hipFree(c->si_scratch);
  if (c->si_host) (void)hipHostFree(c->si_host);
  host_pool_free(c);
  for (auto &w : c->ld) {
    if (w.dev) (void)hipFree(w.dev);
    if (w.host) (void)hipHostFree(w.host);
  }
  band_free(c);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  if (c->stream2) (void)hipStreamDestroy(c->stream2);
  delete c;
  return DVC_OK;
}

int dvc_prepare_data(const char *data_dir) {
  std::string dir = data_dir ? std::string(data_dir) : default_data_dir();
  const std::pair<const char *, int> packs[] = {{"reg", 1584}, {"reg", 6336}, {"irreg", 1584}};
  for (const auto &pk : packs) {
    Ladder L;
    int rc = load_ladder(dir, pk.first, pk.second, L);
    if (rc) return rc;
  }
  return DVC_OK;
}

int dvc_profile(dvc_ctx *c, int enable) {
  DVC_CHECK(c, DVC_EINVAL, "dvc_profile: NULL context");
  c->timer_collect();
  c->timers.clear();
  c->profiling = enable != 0;
  return DVC_OK;
}

int dvc_profile_get(dvc_ctx *c, const char *name, double *total_ms, long *launches) {
  DVC_CHECK(c && name, DVC_EINVAL, "dvc_profile_get: NULL argument");
  c->timer_collect();
  *total_ms = 0.0;
  *launches = 0;
  for (auto &t : c->timers)
    if (t.name == name) { *total_ms = t.total_ms; *launches = t.launches; }
  return DVC_OK;
}

int dvc_ladder_info(dvc_ctx *c, int N, int *num_codes, int *num_edges, int *synd_length) {
  DVC_CHECK(c, DVC_EINVAL, "dvc_ladder_info: NULL context");
  Ladder *L = c->ladder(N);
  DVC_CHECK(L, DVC_EINVAL, "dvc_ladder_info: N must be 1584 or 6336");
  if (num_codes) *num_codes = L->numCodes;
  if (num_edges) *num_edges = L->E;
  if (synd_length) memcpy(synd_length, L->syndLength.data(), sizeof(int) * L->numCodes);
  return DVC_OK;
}

int dvc_ladder_export(dvc_ctx *c, int N, int code, int *ir_out, uint8_t *inv_out) {
  DVC_CHECK(c, DVC_EINVAL, "dvc_ladder_export: NULL context");
  Ladder *L = c->ladder(N);
  DVC_CHECK(L && code >= 0 && code < L->numCodes, DVC_EINVAL, "dvc_ladder_export: bad N or code");
  if (ir_out) memcpy(ir_out, &L->decIr[(size_t)code * L->E], sizeof(int) * L->E);
  if (inv_out) memcpy(inv_out, L->invH.data(), L->invH.size());
  return DVC_OK;
}

// Byte offsets of decode_group's buffers in the context's LDPCA workspace.
// The input region [lr, inEnd) is filled in pinned host memory at the same
// offsets and uploaded in one copy; [state, outEnd) comes back in one copy.
struct LdpcaLayout {
  size_t lr, acc, carry, planes, state, rec, counters, inEnd, out, outEnd, llr, slots, bcase, area, total;
};

static LdpcaLayout ldpca_layout(size_t n, size_t N, size_t C, size_t slotCap, bool mode1) {
  LdpcaLayout o;
  size_t at = 0;
  auto take = [&at](size_t bytes) {
    const size_t r = at;
    at += (bytes + 255) & ~(size_t)255;
    return r;
  };
  o.lr = take(sizeof(float) * n * N);
  o.acc = take(n * (N / 8));
  o.carry = take(mode1 ? n * N : 0);
  o.planes = take(sizeof(PlaneDesc) * n);
  o.state = take(sizeof(PlaneState) * n);
  o.rec = take(sizeof(int4) * n * C);
  o.counters = take(sizeof(int) * 3);
  o.inEnd = at;
  o.out = take(n * N);
  o.outEnd = o.out + n * N;
  o.llr = take(sizeof(float) * n * N);
  o.slots = take(slotCap * N);
  o.bcase = take(mode1 ? sizeof(int) * n * C : 0);
  o.area = take(N == 6336 ? sizeof(uint32_t) * split_area_words((int)N) : 0);
  o.total = at;
  return o;
}

// Grows a code length's LDPCA workspace (device) and its pinned staging (host);
// both are kept between calls and freed by dvc_ctx_destroy.
static int ldpca_workspace(dvc_ctx::LdWork &w, size_t devBytes, size_t hostBytes) {
  if (w.devBytes < devBytes) {
    if (w.dev) DVC_HIP(hipFree(w.dev));
    w.dev = nullptr;
    w.devBytes = 0;
    DVC_HIP(hipMalloc(&w.dev, devBytes));
    w.devBytes = devBytes;
  }
  if (w.hostBytes < hostBytes) {
    if (w.host) DVC_HIP(hipHostFree(w.host));
    w.host = nullptr;
    w.hostBytes = 0;
    DVC_HIP(hipHostMalloc(&w.host, hostBytes, hipHostMallocDefault));
    w.hostBytes = hostBytes;
  }
  return DVC_OK;
}

// Shared driver for one group of bitplanes with the same code length.
// sequential != 0 (n = 1): the codes one after another in increasing order, the
// plain search.  In ParallelMode 0 that is one launch of a single workgroup,
// which takes the codes in order and stops at the first accepted one; with a
// launch and a read-back per code, a QCIF bitplane of 4 codes took 10% longer (1.8
// against 1.63 ms), a CIF one of 9 codes 5%.  ParallelMode 1
// launches each code by itself with the decisions the one before it left.
// ParallelMode 1: items[i].decoded holds the decisions carried into the
// bitplane's first code on entry (the reference's in/out decoded buffer).
// other: bitplanes of the other code length decoded at the same time.
static int decode_group(dvc_ctx *c, int N, int n, dvc_ldpca_item *items, int sequential, int other, hipStream_t s) {
  Ladder *L = c->ladder(N);
  const int C = L->numCodes, nb = N / 8;
  const bool mode1 = c->bp_mode == 1;
  const bool perCode = sequential && mode1;
  const SlotPlan slots = slot_plan(n, C, c->bp_mode);
  const LdpcaLayout o = ldpca_layout(n, N, C, slots.total, mode1);
  dvc_ctx::LdWork &work = c->ld[N == 6336];
  int rc = ldpca_workspace(work, o.total, o.outEnd);
  if (rc) return rc;
  uint8_t *dev = (uint8_t *)work.dev, *host = (uint8_t *)work.host;
  float *dLR = (float *)(dev + o.lr), *dLLR = (float *)(dev + o.llr);
  uint8_t *dAcc = dev + o.acc, *dCarry = dev + o.carry, *dSlots = dev + o.slots, *dOut = dev + o.out;
  PlaneDesc *dPlanes = (PlaneDesc *)(dev + o.planes);
  PlaneState *dState = (PlaneState *)(dev + o.state);
  int4 *dRec = (int4 *)(dev + o.rec);
  int *dCounters = (int *)(dev + o.counters);  // [0] queue head, [1] slot count, [2] bitplanes to resume
  int *dBcase = (int *)(dev + o.bcase);
  PlaneDesc *hPlanes = (PlaneDesc *)(host + o.planes);
  PlaneState *hState = (PlaneState *)(host + o.state);
  int4 *hRec = (int4 *)(host + o.rec);
  int *hCounters = (int *)(host + o.counters);
  for (int i = 0; i < n; i++) {
    DVC_CHECK(items[i].LR && items[i].acc && items[i].decoded, DVC_EINVAL, "dvc_ldpca: NULL item pointer");
    const int st0 = items[i].start_level;
    DVC_CHECK(st0 < C, DVC_EINVAL, "dvc_ldpca: start_level beyond the ladder");
    memcpy(host + o.lr + sizeof(float) * i * N, items[i].LR, sizeof(float) * N);
    memcpy(host + o.acc + (size_t)i * nb, items[i].acc, nb);
    if (mode1) memcpy(host + o.carry + (size_t)i * N, items[i].decoded, N);
    hPlanes[i] = PlaneDesc{N, dLR + (size_t)i * N, dLLR + (size_t)i * N, dAcc + (size_t)i * nb,
                           (uint32_t)items[i].crc, dState + i, dRec + (size_t)i * C,
                           mode1 ? dCarry + (size_t)i * N : nullptr, mode1 ? dBcase + (size_t)i * C : nullptr};
    hState[i] = PlaneState{st0 >= 0 ? st0 : -1, C - 1, 0.0f, 0, 0};
    for (int l = 0; l < C; l++) hRec[(size_t)i * C + l] = make_int4(0, REC_NOT_RUN, -1, 0);
  }
  DVC_HIP(hipMemcpyAsync(dev, host, o.inEnd, hipMemcpyHostToDevice, s));
  uint32_t *area = N == 6336 ? (uint32_t *)(dev + o.area) : nullptr;
  TIMED(c, "ce_llr", s, launch_ce_llr(dPlanes, n, 1, c->lad1584, c->lad6336, dCounters, area, s));
  std::vector<PlaneState> state(n);
  if (perCode) {
    DVC_HIP(hipMemcpyAsync(state.data(), dState, sizeof(PlaneState) * n, hipMemcpyDeviceToHost, s));
    DVC_HIP(hipStreamSynchronize(s));
  }

  LadderDev ld = ladder_dev(*L);
  std::vector<int4> rec((size_t)n * C);
  if (perCode) {
    // one code per launch, each with the decisions the previous code left
    for (int i = 0; i < n; i++) {
      int level = state[i].start;
      int4 r;
      for (; level < C - 1; level++) {
        PlaneState ps{state[i].start, C - 1, state[i].entropy, level, state[i].taint};
        int zero[3] = {0, 0, 0};
        DVC_HIP(hipMemcpyAsync(dState + i, &ps, sizeof(ps), hipMemcpyHostToDevice, s));
        DVC_HIP(hipMemcpyAsync(dCounters, zero, sizeof(zero), hipMemcpyHostToDevice, s));
        BpArgs a{ld, dPlanes + i, 1, dCounters, 1, 1, c->max_iter, dSlots, dCounters + 1, slots.bp, c->bp_poll,
                 c->bp_mode, c->rate_step};
        a.area = area;
        TIMED(c, N == 6336 ? "bp_6336" : "bp_1584", s, launch_bp(c, N, 1, 0, 1, true, a, s));
        DVC_HIP(hipMemcpyAsync(&r, dRec + (size_t)i * C + level, sizeof(r), hipMemcpyDeviceToHost, s));
        DVC_HIP(hipStreamSynchronize(s));
        if (r.y == REC_ACCEPTED) {
          DVC_HIP(hipMemcpy(items[i].decoded, dSlots + (size_t)r.z * N, N, hipMemcpyDeviceToHost));
          break;
        }
        DVC_CHECK(r.z >= 0 && r.z < slots.bp, DVC_ESTATE, "dvc_ldpca: missing decisions of a failed code");
        DVC_HIP(hipMemcpyAsync(dCarry + (size_t)i * N, dSlots + (size_t)r.z * N, N, hipMemcpyDeviceToDevice, s));
      }
      if (level == C - 1) {
        PlaneState ps{state[i].start, C - 1, state[i].entropy, C, state[i].taint};
        DVC_HIP(hipMemcpyAsync(dState + i, &ps, sizeof(ps), hipMemcpyHostToDevice, s));
        TIMED(c, "invh", s, launch_invh(dPlanes + i, 1, ld, dSlots, slots.bp, s));
        DVC_HIP(hipMemcpyAsync(&r, dRec + (size_t)i * C + (C - 1), sizeof(r), hipMemcpyDeviceToHost, s));
        DVC_HIP(hipStreamSynchronize(s));
        DVC_HIP(hipMemcpy(items[i].decoded, dSlots + (size_t)r.z * N, N, hipMemcpyDeviceToHost));
      }
    }
    DVC_HIP(hipMemcpy(rec.data(), dRec, sizeof(int4) * rec.size(), hipMemcpyDeviceToHost));
  } else {
    const int maxOff = C - 1;
    BpArgs a{ld, dPlanes, n, dCounters, n * maxOff, maxOff, c->max_iter, dSlots, dCounters + 1, slots.bp,
             c->bp_poll, c->bp_mode, c->rate_step};
    a.area = area;
    a.area_clear = 1;
    TIMED(c, N == 6336 ? "bp_6336" : "bp_1584", s, launch_bp(c, N, n, other, 1, sequential, a, s));
    a.area_clear = 0;
    for (int round = 0; mode1; round++) {
      // ParallelMode 1: resolve with the carried decisions; resume the
      // bitplanes that reach a code this launch did not finish
      DVC_CHECK(round <= C, DVC_ESTATE, "dvc_ldpca: ParallelMode 1 resolution does not settle");
      DVC_HIP(launch_zero_ints(dCounters + 2, 1, s));
      DVC_HIP(launch_mode1_resolve(dPlanes, n, C, N, dSlots, slots.bp, dCounters + 2, s));
      int resume = 0;
      DVC_HIP(hipMemcpyAsync(&resume, dCounters + 2, sizeof(int), hipMemcpyDeviceToHost, s));
      DVC_HIP(hipStreamSynchronize(s));
      DVC_CHECK(resume < (1 << 20), DVC_ENOMEM, "ParallelMode 1: decision slots exhausted");
      if (!resume) break;
      DVC_HIP(launch_zero_ints(dCounters, 1, s));
      TIMED(c, N == 6336 ? "bp_6336" : "bp_1584", s, launch_bp(c, N, n, other, 1, sequential, a, s));
    }
    TIMED(c, "invh", s, launch_invh(dPlanes, n, ld, dSlots, slots.bp, s));
    // every bitplane's accepted decisions to dOut, then states, records,
    // counters and decisions back in one copy
    DVC_HIP(launch_gather_accepted(dPlanes, n, N, dSlots, slots.total, dOut, s));
    DVC_HIP(hipMemcpyAsync(host + o.state, dev + o.state, o.outEnd - o.state, hipMemcpyDeviceToHost, s));
    DVC_HIP(hipStreamSynchronize(s));
    DVC_CHECK(hCounters[1] <= slots.bp, DVC_ENOMEM, "dvc_ldpca_decode_batch: decision slots exhausted");
    memcpy(state.data(), hState, sizeof(PlaneState) * n);
    memcpy(rec.data(), hRec, sizeof(int4) * rec.size());
    for (int i = 0; i < n; i++) {
      const int best = state[i].best;
      DVC_CHECK(best >= 0 && best < C, DVC_ESTATE, "dvc_ldpca_decode_batch: bad accepted code");
      const int4 r = rec[(size_t)i * C + best];
      DVC_CHECK(r.y == REC_ACCEPTED && r.z >= 0 && r.z < slots.total, DVC_ESTATE,
                "dvc_ldpca_decode_batch: missing accepted record");
      DVC_CHECK(unfinished_code(&rec[(size_t)i * C], std::max(state[i].start, 0), best, c->rate_step) < 0, DVC_ESTATE,
                "dvc_ldpca: a code below the accepted one did not finish");
      memcpy(items[i].decoded, host + o.out + (size_t)i * N, N);
    }
  }
  // Stats as the sequential search reports them.
  for (int i = 0; i < n; i++) {
    dvc_bp_stats &st = items[i].stats;
    memset(&st, 0, sizeof(st));
    st.start_level = state[i].start;
    st.entropy = state[i].entropy;
    int lvl = -1;
    for (int l = st.start_level; l < C; l++) {
      const int4 r = rec[(size_t)i * C + l];
      if (r.y == REC_ACCEPTED) { lvl = l; break; }
      st.iterations += r.x;
    }
    DVC_CHECK(lvl >= 0, DVC_ESTATE, "dvc_ldpca: no accepted code");
    st.level = lvl;
    st.iterations += rec[(size_t)i * C + lvl].x;
    st.rate = L->syndLength[lvl] + 8;
    st.requests = lvl - st.start_level + 1;
    if (c->rate_step) {
      // codes tried: the DYNAMICSTEP offsets below lvl, then lvl itself
      st.requests = 1;
      for (int off = 0; st.start_level + off < lvl; off = dynstep_next(off)) st.requests++;
    }
    st.used_inverse = rec[(size_t)i * C + lvl].w;
    for (int l = 0; l < C; l++) {
      const int4 r = rec[(size_t)i * C + l];
      if (r.y != REC_NOT_RUN) st.iterations_run += r.x;
    }
  }
  return DVC_OK;
}

int dvc_ldpca_decode(dvc_ctx *c, int N, const float *LR, const uint8_t *acc, uint8_t crc, int start_level,
                     uint8_t *decoded, dvc_bp_stats *stats) {
  DVC_CHECK(c, DVC_EINVAL, "dvc_ldpca_decode: NULL context");
  DVC_CHECK(c->ladder(N), DVC_EINVAL, "dvc_ldpca_decode: N must be 1584 or 6336");
  DVC_HIP(hipSetDevice(c->device));
  dvc_ldpca_item it{N, LR, acc, crc, start_level, decoded, {}};
  int rc = decode_group(c, N, 1, &it, 1, 0, c->stream);
  if (rc == DVC_OK && stats) *stats = it.stats;
  return rc;
}

int dvc_ldpca_decode_batch(dvc_ctx *c, int n, dvc_ldpca_item *items) {
  DVC_CHECK(c, DVC_EINVAL, "dvc_ldpca_decode_batch: NULL context");
  DVC_CHECK(n >= 0 && (n == 0 || items), DVC_EINVAL, "dvc_ldpca_decode_batch: bad item list");
  DVC_HIP(hipSetDevice(c->device));
  std::vector<dvc_ldpca_item> g[2];
  std::vector<int> gi[2];
  for (int i = 0; i < n; i++) {
    DVC_CHECK(items[i].N == 1584 || items[i].N == 6336, DVC_EINVAL, "dvc_ldpca_decode_batch: N must be 1584 or 6336");
    int k = items[i].N == 6336;
    g[k].push_back(items[i]);
    gi[k].push_back(i);
  }
  // both code lengths at once, each on its own stream and host thread: one after
  // the other, the second waited for the last codes of the first (see bp_grid)
  // (the second stream is made when a batch first needs it: a queue taken by one
  // that never runs is missing to an engine's lanes)
  bool both = !g[0].empty() && !g[1].empty();
  if (both && !c->stream2) both = create_stream_beside(&c->stream, 1, &c->stream2, nullptr) == hipSuccess;
  int rcs[2] = {DVC_OK, DVC_OK};
  std::string err[2];
  auto part = [&](int k, hipStream_t s) -> int {
    DVC_HIP(hipSetDevice(c->device));
    return decode_group(c, k ? 6336 : 1584, (int)g[k].size(), g[k].data(), 0, both ? (int)g[1 - k].size() : 0, s);
  };
  auto told = [&](int k, hipStream_t s) -> int {  // its error text is the thread's
    const int rc = part(k, s);
    if (rc) err[k] = dvc_last_error();
    return rc;
  };
  if (both) {
    run_pair([&] { return told(0, c->stream2); }, [&] { return told(1, c->stream); }, DVC_ENOMEM, rcs, err);
    // what a part that failed left on its stream still reads the staging
    if (rcs[0]) (void)hipStreamSynchronize(c->stream2);
    if (rcs[1]) (void)hipStreamSynchronize(c->stream);
  } else {
    for (int k = 0; k < 2; k++)
      if (!g[k].empty()) rcs[k] = told(k, c->stream);
  }
  for (int k = 0; k < 2; k++) {
    if (rcs[k]) {
      set_error(err[k]);
      return rcs[k];
    }
    for (size_t j = 0; j < g[k].size(); j++) items[gi[k][j]].stats = g[k][j].stats;
  }
  return DVC_OK;
}

}  // extern "C"
