// band.hip -- the per-band entry points of include/dvc_accel.h: the calls a
// decoder that keeps its own per-frame loop makes per band, on the
// reference's data layouts (SMF, SearchInfo, Trans, MV of global.h), run by
// the same kernels the batched frame decoder launches (frame_kernels.hip) on
// a one-frame descriptor held in the context.
#include <string.h>
#include <algorithm>
#include <utility>
#include <vector>
#include "dvc_internal.h"
#include "frame_kernels.h"

namespace dvc {

// One WZ frame's device state for the per-band calls, and a second set of
// buffers for dvc_forward_me (which runs before the frame's set-up).
struct BandState {
  int W = 0, H = 0, N = 0, qindex = 0;
  bool ready = false;
  uint8_t *mem = nullptr;  // one block: frame buffers, descriptor and list
  size_t bytes = 0;
  float *dist = nullptr;   // the band's noise distribution, N * stride floats
  size_t distBytes = 0;
  int distIndex = -1, distRange = -1;  // band of the distribution in `dist`
  int nsir = 0;                        // SIR entries (WZ 4x4 blocks)
  std::vector<int> blk;                // blkIdx of each SIR entry
  int *d_blk = nullptr;                // the same on the device
  uint8_t *gat = nullptr;              // the distribution in noiseDistribution's SIR-entry layout
  size_t gatBytes = 0;
  FrameDev fd{};
  FrameDev *d_fd = nullptr;
  int *d_list = nullptr;
  uint8_t *fmeMem = nullptr;  // dvc_forward_me's block
  size_t fmeBytes = 0;
};

void band_free(dvc_ctx *c) {
  if (!c->band) return;
  if (c->band->mem) (void)hipFree(c->band->mem);
  if (c->band->dist) (void)hipFree(c->band->dist);
  if (c->band->fmeMem) (void)hipFree(c->band->fmeMem);
  if (c->band->gat) (void)hipFree(c->band->gat);
  delete c->band;
  c->band = nullptr;
}

static size_t al(size_t v) { return (v + 255) & ~(size_t)255; }

// Device block of at least `bytes` in *p (grown, contents dropped).
static int grow(uint8_t **p, size_t *have, size_t bytes) {
  if (*have >= bytes) return DVC_OK;
  if (*p) DVC_HIP(hipFree(*p));
  *p = nullptr;
  *have = 0;
  DVC_HIP(hipMalloc((void **)p, bytes));
  *have = bytes;
  return DVC_OK;
}

static bool valid_size(int W, int H) { return (W == 176 && H == 144) || (W == 352 && H == 288); }

// The block-major distribution to noiseDistribution's layout: SIR entry i's
// `stride` values at i * stride.
__global__ void k_dist_gather(const float *src, float *dst, int n, const int *blk, int stride) {
  const int i = blockIdx.y, k = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || k >= stride) return;
  dst[(size_t)i * stride + k] = src[(size_t)blk[i] * stride + k];
}

// Staging of one call: buffers that go to the device, each through its part of
// the context's pinned block, and parts that results come back through.
struct Stage {
  dvc_ctx *c;
  size_t used = 0;
  std::vector<HostCopy> copies;
  std::vector<std::pair<void *, std::pair<size_t, size_t>>> ups;  // device, (offset, bytes)
  int reserve(size_t bytes) { return pinned_grow(&c->si_host, &c->si_host_bytes, bytes); }
  // The next `bytes` of the block (the calls reserve what they take).
  uint8_t *part(size_t bytes) {
    uint8_t *p = c->si_host + used;
    used = al(used + bytes);
    return p;
  }
  // Queues the upload of a part that the caller fills, or of a host buffer.
  uint8_t *up(void *dev, size_t bytes, const void *src = nullptr) {
    const size_t o = used;
    uint8_t *p = part(bytes);
    if (src) copies.push_back(HostCopy{p, src, bytes});
    ups.push_back({dev, {o, bytes}});
    return p;
  }
  int send(hipStream_t s) {
    host_copy(c, copies);
    for (const auto &u : ups)
      DVC_HIP(hipMemcpyAsync(u.first, c->si_host + u.second.first, u.second.second, hipMemcpyHostToDevice, s));
    return DVC_OK;
  }
};

// Window positions of block b (initSMF's searchWidth x searchHeight).
static int smf_len(const BandState *B, int b) {
  const int bw = B->W / 4, top = (b / bw) * 4, left = (b % bw) * 4;
  return (std::min(B->W - 4, left + 4) - std::max(0, left - 4) + 1) *
         (std::min(B->H - 4, top + 4) - std::max(0, top - 4) + 1);
}

static int need_frame(dvc_ctx *c, const char *who) {
  DVC_CHECK(c, DVC_EINVAL, std::string(who) + ": NULL context");
  DVC_CHECK(c->band && c->band->ready, DVC_ESTATE, std::string(who) + ": call dvc_band_frame_init first");
  DVC_HIP(hipSetDevice(c->device));
  return DVC_OK;
}

}  // namespace dvc

using namespace dvc;

extern "C" int dvc_band_frame_init(dvc_ctx *c, int W, int H, int qindex, const uint8_t *past, const uint8_t *fut,
                                   int past_idx, int cur_idx, int fut_idx, const dvc_search_info *sir, int nsir) {
  DVC_CHECK(c, DVC_EINVAL, "dvc_band_frame_init: NULL context");
  DVC_CHECK(valid_size(W, H), DVC_EINVAL, "dvc_band_frame_init: size must be QCIF or CIF");
  DVC_CHECK(qindex >= 1 && qindex <= 8, DVC_EINVAL, "dvc_band_frame_init: qindex must be 1..8");
  DVC_CHECK(past && fut, DVC_EINVAL, "dvc_band_frame_init: NULL key frame");
  DVC_CHECK(past_idx < cur_idx && cur_idx < fut_idx, DVC_EINVAL, "dvc_band_frame_init: need past_idx < cur_idx < fut_idx");
  const int N = W * H / 16, bw = W / 4, n8 = N / 4;
  // initSIR (sideInfoCreation.cpp:554-596) lists the 4x4 blocks of the WZ 8x8
  // blocks in raster order; the blocks it leaves out (skip and intra) are
  // marked non-WZ in an 8x8 mode map, which every per-block kernel tests
  std::vector<int> blk;
  std::vector<uint8_t> mode;
  if (sir) {
    DVC_CHECK(nsir >= 0 && nsir <= N, DVC_EINVAL, "dvc_band_frame_init: more SIR entries than blocks");
    mode.assign(n8, 2);
    std::vector<int> per8(n8, 0);
    for (int i = 0; i < nsir; i++) {
      const int b = sir[i].blkIdx;
      DVC_CHECK(b >= 0 && b < N && (i == 0 || b > sir[i - 1].blkIdx) && sir[i].top == (b / bw) * 4 &&
                    sir[i].left == (b % bw) * 4,
                DVC_EINVAL, "dvc_band_frame_init: the SIR must list 4x4 blocks in raster order (blkIdx, top, left)");
      const int b8 = (b / bw / 2) * (bw / 2) + (b % bw) / 2;
      mode[b8] = 0;
      per8[b8]++;
      blk.push_back(b);
    }
    for (int k = 0; k < n8; k++)
      DVC_CHECK(per8[k] == 0 || per8[k] == 4, DVC_EINVAL,
                "dvc_band_frame_init: the SIR lists part of an 8x8 block (block modes are per 8x8 block)");
  } else {
    nsir = N;
  }
  if (blk.empty() && nsir == N)
    for (int b = 0; b < N; b++) blk.push_back(b);
  if (nsir == N) mode.clear();  // every block is WZ
  DVC_HIP(hipSetDevice(c->device));
  int rc = ensure_cost_tables(c);
  if (rc) return rc;
  if (!c->band) c->band = new BandState();
  BandState *B = c->band;
  B->ready = false;
  const size_t FS = (size_t)W * H;
  size_t off = 0;
  auto take = [&off](size_t b) { const size_t o = off; off = al(off + b); return o; };
  const size_t oPast = take(FS), oFut = take(FS), oPlp = take(FS), oFlp = take(FS), oPh = take(4 * FS),
               oFh = take(4 * FS), oSi = take(FS), oRec = take(FS), oRt = take(4 * FS), oAl = take(4 * FS),
               oOb = take((size_t)4 * (W - 3) * (H - 3)), oSmf = take((size_t)4 * 81 * N), oLR = take(4 * (size_t)N), oFd = take(sizeof(FrameDev)),
               oSpan = take(sizeof(int2) * (size_t)N), oList = take(sizeof(int)), oBlk = take(sizeof(int) * (size_t)N), oMode = take((size_t)n8);
  if ((rc = grow(&B->mem, &B->bytes, off))) return rc;
  uint8_t *m = B->mem;
  FrameDev &f = B->fd;
  memset(&f, 0, sizeof(f));
  f.W = W; f.H = H; f.N = N; f.qindex = qindex;
  f.iPC = (double)(cur_idx - past_idx) / (double)(fut_idx - past_idx);
  f.iFC = (double)(fut_idx - cur_idx) / (double)(fut_idx - past_idx);
  f.past = m + oPast; f.fut = m + oFut; f.past_lp = m + oPlp; f.fut_lp = m + oFlp;
  f.past_half = m + oPh; f.fut_half = m + oFh;
  f.si = m + oSi; f.recons = m + oRec; f.reconsTrans = (int *)(m + oRt); f.alpha = (float *)(m + oAl);
  f.octBand = (int *)(m + oOb); f.smf = (float *)(m + oSmf); f.LR = (float *)(m + oLR);
  f.distSpan = (int2 *)(m + oSpan);
  B->d_blk = (int *)(m + oBlk);
  B->nsir = nsir;
  B->blk.swap(blk);
  f.mode = mode.empty() ? nullptr : m + oMode;
  B->d_fd = (FrameDev *)(m + oFd);
  B->d_list = (int *)(m + oList);
  B->W = W; B->H = H; B->N = N; B->qindex = qindex;
  B->distIndex = B->distRange = -1;
  hipStream_t s = c->stream;
  Stage st{c};
  if ((rc = st.reserve(2 * FS + sizeof(int) * (size_t)N + n8 + sizeof(FrameDev) + 6 * 256))) return rc;
  memset(st.up(B->d_list, sizeof(int)), 0, sizeof(int));
  if (nsir > 0) st.up(B->d_blk, sizeof(int) * (size_t)nsir, B->blk.data());
  if (!mode.empty()) st.up((void *)f.mode, (size_t)n8, mode.data());
  st.up((void *)f.past, FS, past);
  st.up((void *)f.fut, FS, fut);
  st.up(B->d_fd, sizeof(FrameDev), &f);
  if ((rc = st.send(s))) return rc;
  DVC_HIP(launch_keyframe_filters(f.past, (uint8_t *)f.past_lp, (uint8_t *)f.past_half, W, H, s));
  DVC_HIP(launch_keyframe_filters(f.fut, (uint8_t *)f.fut_lp, (uint8_t *)f.fut_half, W, H, s));
  DVC_HIP(hipStreamSynchronize(s));
  B->ready = true;
  return DVC_OK;
}

extern "C" int dvc_noise_distribution(dvc_ctx *c, int range, int index, const float *alpha, const dvc_smf *smf,
                                      const int *oct, float *dist) {
  int rc = need_frame(c, "dvc_noise_distribution");
  if (rc) return rc;
  DVC_CHECK(index >= 0 && index < 16 && range > 0 && alpha && smf && oct, DVC_EINVAL,
            "dvc_noise_distribution: bad argument");
  BandState *B = c->band;
  FrameDev &f = B->fd;
  const int W = B->W, H = B->H, N = B->N, stride = index ? 2 * range + 1 : range;
  hipStream_t s = c->stream;
  const size_t need = sizeof(float) * (size_t)N * stride;
  B->distIndex = B->distRange = -1;
  if ((rc = grow((uint8_t **)&B->dist, &B->distBytes, need))) return rc;
  // The kernel reads one coefficient per position of the over-complete transform
  // and the SMF's probabilities: only those go up, packed on the way into pinned
  // memory.  With the whole records copied from pageable memory (8.6 MB for CIF)
  // and unpacked by a kernel, a CIF band's distribution and the likelihood ratios
  // of its six bits took 1.77 ms; now 1.09.
  const int ns = B->nsir, npos = (W - 3) * (H - 3);
  const size_t bAlpha = sizeof(float) * W * H, bOct = sizeof(int) * (size_t)npos, bSmf = sizeof(float) * 81 * (size_t)N;
  const size_t bOut = dist ? sizeof(float) * (size_t)ns * stride : 0;
  Stage st{c};
  if ((rc = st.reserve(bAlpha + bOct + bSmf + sizeof(FrameDev) + bOut + 5 * 256))) return rc;
  f.index = index; f.range = range; f.distStride = stride; f.dist = B->dist;
  st.up(f.alpha, bAlpha, alpha);
  int *hOct = (int *)st.up(f.octBand, bOct);
  float *hSmf = (float *)st.up(f.smf, bSmf);
  st.up(B->d_fd, sizeof(FrameDev), &f);
  constexpr int kPos = 4096, kEnt = 128;  // positions and SIR entries of one piece of work
  const int po = (npos + kPos - 1) / kPos, pe = (ns + kEnt - 1) / kEnt;
  host_parallel(c, po + pe, 64 * (size_t)npos + sizeof(dvc_smf) * (size_t)ns, [&](size_t piece) {
    if ((int)piece < po) {
      const int a = (int)piece * kPos, b = std::min(npos, a + kPos);
      for (int p = a; p < b; p++) hOct[p] = oct[(size_t)16 * p + index];
      return;
    }
    const int a = ((int)piece - po) * kEnt, b = std::min(ns, a + kEnt);
    for (int i = a; i < b; i++) {
      const int len = std::max(0, std::min(smf[i].probLen, 81));
      float *d = hSmf + (size_t)81 * B->blk[i];
      memcpy(d, smf[i].prob, sizeof(float) * len);
      std::fill(d + len, d + 81, 0.0f);
    }
  });
  if ((rc = st.send(s))) return rc;
  DVC_HIP(launch_noise_dist(B->d_fd, B->d_list, 1, N, 1, s));
  const float *from = B->dist;
  if (dist && ns > 0 && ns < N) {  // SIR entries only, in their order
    if ((rc = grow(&B->gat, &B->gatBytes, bOut))) return rc;
    hipLaunchKernelGGL(k_dist_gather, dim3((stride + 255) / 256, ns), dim3(256), 0, s, B->dist, (float *)B->gat, ns,
                       B->d_blk, stride);
    DVC_HIP(hipGetLastError());
    from = (const float *)B->gat;
  }
  if (bOut && (rc = copy_back(c, s, dist, from, st.part(bOut), bOut))) return rc;
  DVC_HIP(hipStreamSynchronize(s));
  B->distIndex = index;
  B->distRange = range;
  return DVC_OK;
}

extern "C" int dvc_cond_bit_prob(dvc_ctx *c, float *LR, int index, int bit, int step, const int *recons_trans,
                                 int range) {
  int rc = need_frame(c, "dvc_cond_bit_prob");
  if (rc) return rc;
  DVC_CHECK(LR && recons_trans && bit >= 1 && bit <= 30 && step > 0, DVC_EINVAL, "dvc_cond_bit_prob: bad argument");
  BandState *B = c->band;
  DVC_CHECK(B->distIndex == index && B->distRange == range, DVC_ESTATE,
            "dvc_cond_bit_prob: no noise distribution of this band (call dvc_noise_distribution first)");
  FrameDev &f = B->fd;
  hipStream_t s = c->stream;
  f.index = index; f.bit = bit; f.step = step; f.range = range;
  f.levelShift = index ? (qtable_entry(B->qindex, index) - 2) / 2 : 0;
  f.distStride = index ? 2 * range + 1 : range;
  f.dist = B->dist;
  const size_t bRt = sizeof(int) * B->W * B->H, bLR = sizeof(float) * B->N;
  Stage st{c};
  if ((rc = st.reserve(bRt + sizeof(FrameDev) + bLR + 3 * 256))) return rc;
  st.up(f.reconsTrans, bRt, recons_trans);
  st.up(B->d_fd, sizeof(FrameDev), &f);
  if ((rc = st.send(s))) return rc;
  DVC_HIP(launch_condbit(B->d_fd, B->d_list, 1, B->N, s));
  return copy_back(c, s, LR, f.LR, st.part(bLR), bLR);
}

extern "C" int dvc_update_si(dvc_ctx *c, uint8_t *side_info, const uint8_t *recons) {
  int rc = need_frame(c, "dvc_update_si");
  if (rc) return rc;
  DVC_CHECK(side_info && recons, DVC_EINVAL, "dvc_update_si: NULL argument");
  BandState *B = c->band;
  FrameDev &f = B->fd;
  hipStream_t s = c->stream;
  const size_t FS = (size_t)B->W * B->H;
  Stage st{c};
  if ((rc = st.reserve(3 * FS + 3 * 256))) return rc;
  st.up(f.si, FS, side_info);
  st.up(f.recons, FS, recons);
  if ((rc = st.send(s))) return rc;
  DVC_HIP(launch_update_si(B->d_fd, B->d_list, 1, B->N, CostTables{c->d_costFme, c->d_costUsi}, s));
  return copy_back(c, s, side_info, f.si, st.part(FS), FS);
}

extern "C" int dvc_update_smf(dvc_ctx *c, dvc_smf *smf, const uint8_t *recons, const uint8_t *side_info) {
  int rc = need_frame(c, "dvc_update_smf");
  if (rc) return rc;
  DVC_CHECK(smf && recons && side_info, DVC_EINVAL, "dvc_update_smf: NULL argument");
  BandState *B = c->band;
  FrameDev &f = B->fd;
  hipStream_t s = c->stream;
  const size_t FS = (size_t)B->W * B->H;
  const int N = B->N, ns = B->nsir;
  if (ns == 0) return DVC_OK;  // no WZ block: updateSMF's loop is empty
  // every window position's probability is new, so none goes up; they come back
  // block by block and are copied into the caller's records
  const size_t bSmf = sizeof(float) * 81 * (size_t)N;
  Stage st{c};
  if ((rc = st.reserve(2 * FS + bSmf + 3 * 256))) return rc;
  st.up(f.si, FS, side_info);
  st.up(f.recons, FS, recons);
  if ((rc = st.send(s))) return rc;
  DVC_HIP(launch_update_smf(B->d_fd, B->d_list, 1, N, s));
  const float *h = (const float *)st.part(bSmf);
  DVC_HIP(hipMemcpyAsync((void *)h, f.smf, bSmf, hipMemcpyDeviceToHost, s));
  DVC_HIP(hipStreamSynchronize(s));
  constexpr int kEnt = 128;
  host_parallel(c, (ns + kEnt - 1) / kEnt, 2 * sizeof(dvc_smf) * (size_t)ns, [&](size_t piece) {
    const int a = (int)piece * kEnt, b = std::min(ns, a + kEnt);
    for (int i = a; i < b; i++) {
      const int len = std::min(smf[i].probLen, smf_len(B, B->blk[i]));
      if (len > 0) memcpy(smf[i].prob, h + (size_t)81 * B->blk[i], sizeof(float) * len);
    }
  });
  return DVC_OK;
}

extern "C" int dvc_forward_me(dvc_ctx *c, int W, int H, const uint8_t *fut_lp, const uint8_t *past_lp, int past_idx,
                              int cur_idx, int fut_idx, dvc_mv *mb_mv) {
  DVC_CHECK(c, DVC_EINVAL, "dvc_forward_me: NULL context");
  DVC_CHECK(valid_size(W, H) && fut_lp && past_lp && mb_mv, DVC_EINVAL, "dvc_forward_me: bad argument");
  DVC_CHECK(past_idx < cur_idx && cur_idx < fut_idx, DVC_EINVAL, "dvc_forward_me: need past_idx < cur_idx < fut_idx");
  static_assert(sizeof(dvc_mv) == sizeof(MVd), "MV layouts differ");
  DVC_HIP(hipSetDevice(c->device));
  int rc = ensure_cost_tables(c);
  if (rc) return rc;
  if (!c->band) c->band = new BandState();
  BandState *B = c->band;
  const size_t FS = (size_t)W * H, nmb = FS / 256;
  size_t off = 0;
  auto take = [&off](size_t b) { const size_t o = off; off = al(off + b); return o; };
  const size_t oPlp = take(FS), oFlp = take(FS), oFwd = take(sizeof(MVd) * nmb), oMb = take(sizeof(MVd) * nmb),
               oHoles = take(16 * nmb), oFd = take(sizeof(FrameDev)), oList = take(sizeof(int));
  if ((rc = grow(&B->fmeMem, &B->fmeBytes, off))) return rc;
  uint8_t *m = B->fmeMem;
  FrameDev f;
  memset(&f, 0, sizeof(f));
  f.W = W; f.H = H; f.N = (int)(FS / 16);
  f.iPC = (double)(cur_idx - past_idx) / (double)(fut_idx - past_idx);
  f.iFC = (double)(fut_idx - cur_idx) / (double)(fut_idx - past_idx);
  f.past_lp = m + oPlp; f.fut_lp = m + oFlp;
  f.fwd = (MVd *)(m + oFwd); f.mbmv = (MVd *)(m + oMb); f.holes = (double *)(m + oHoles);
  hipStream_t s = c->stream;
  const size_t bMv = sizeof(MVd) * nmb;
  Stage st{c};
  if ((rc = st.reserve(2 * FS + sizeof(FrameDev) + bMv + 5 * 256))) return rc;
  memset(st.up(m + oList, sizeof(int)), 0, sizeof(int));
  st.up(m + oFd, sizeof(FrameDev), &f);
  st.up(m + oPlp, FS, past_lp);
  st.up(m + oFlp, FS, fut_lp);
  if ((rc = st.send(s))) return rc;
  DVC_HIP(launch_forward_me((const FrameDev *)(m + oFd), (const int *)(m + oList), 1, (int)nmb,
                            CostTables{c->d_costFme, c->d_costUsi}, s));
  return copy_back(c, s, mb_mv, f.mbmv, st.part(bMv), bMv);
}
