// frame_kernels.hip -- side information, transform, correlation-noise-model,
// motion-learning and reconstruction kernels of the WZ frame decode on gfx950.
//
// Each kernel restates one reference function (file:line of DvcDec/src/) with
// the reference's operand order and precision: integer SADs, FP64 motion
// costs and interpolation weights, FP32 noise-model sums in the reference's
// summation order, and the glibc-identical expf of dvc_math.h.  The results
// are bit-identical to the CPU path.  Work is laid out per frame of a batch:
// blockIdx.y (or .z) selects the frame, the other grid dimensions its blocks.
#include <float.h>
#include <algorithm>
#include "dvc_math.h"
#include "frame_kernels.h"
#include "ldpca_kernels.h"
#include "engine_kernels.h"

#pragma clang fp contract(off)

namespace dvc {

// BlockModeFlag value of a WZ block (defines.h:15)
constexpr uint8_t kWzBlock = 0, kSkipBlock = 2;
// Whether 4x4 block b of f is a WZ block (its 8x8 block's mode, as the
// reference's blk88row + (j >> 1) lookup reads it).
__device__ __forceinline__ bool wz_block(const FrameDev &f, int b) {
  if (!f.mode) return true;
  const int bw = f.W >> 2, i = b / bw, j = b - i * bw;
  return f.mode[(i >> 1) * (f.W >> 3) + (j >> 1)] == kWzBlock;
}

#define DVC_K 0.05f  // defines.h:10, promoted to double where it is used

__device__ __forceinline__ int imin(int a, int b) { return a < b ? a : b; }
__device__ __forceinline__ int imax(int a, int b) { return a > b ? a : b; }

// computeEndPoint (sideInfoCreation.cpp:14-22)
__device__ __forceinline__ int end_point(double st, double vec, double scale, int lower, int upper) {
  int e = (int)((st + vec * scale) + 0.5);
  return e < lower ? lower : (e > upper ? upper : e);
}
// costFunc (sideInfoCreation.cpp:10-12)
__device__ __forceinline__ double cost_func(double mad, double x, double y) {
  return mad * (1.0 + (double)DVC_K * sqrt(x * x + y * y));
}

// op over the wave's 64 values, for min, max and the like (op(x, x) = x), by
// data-parallel moves: within rows of 16 lanes, then across rows to lane 63.
template <class Op>
__device__ __forceinline__ int wave_reduce(int v, Op op) {
  v = op(v, __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, false));   // quad_perm [1, 0, 3, 2]
  v = op(v, __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, false));   // quad_perm [2, 3, 0, 1]
  v = op(v, __builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, false));  // row_half_mirror
  v = op(v, __builtin_amdgcn_mov_dpp(v, 0x140, 0xf, 0xf, false));  // row_mirror
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));  // row_bcast:15 into rows 1 and 3
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));  // row_bcast:31 into rows 2 and 3
  return __builtin_amdgcn_readlane(v, 63);
}

// Lexicographic (cost, index) minimum across a wave: the first candidate in
// scan order among those of least cost, which is what a strict-< raster scan
// returns.
__device__ __forceinline__ void wave_argmin(double &cost, int &idx) {
  for (int o = 32; o > 0; o >>= 1) {
    double c2 = __shfl_xor(cost, o);
    int i2 = __shfl_xor(idx, o);
    if (c2 < cost || (c2 == cost && i2 < idx)) { cost = c2; idx = i2; }
  }
}

// ------------------------------------------------------------ key frames
// lowPassFilter (filter.cpp:214-233): sum/9 in double equals integer division.
// FIR_filter (filter.cpp:55-117): the 6-tap (1,-5,20,20,-5,1)/32 half-pel
// filter; its dyadic coefficients make (int)(sum + 0.5) then the [0,255]
// clip equal to clip((S + 16) >> 5) (1-D) and clip((S + 512) >> 10) (2-D).
// Thread (i, j) of a grid of rows i < rowsY (rowsY >= H) and columns j:
// low-pass sample (i, j) and the half-pel samples of rows i, i + rowsY, ...
// of the 2H x 2W image; with copyTo set it also copies in[i][j] there.
__device__ __forceinline__ void keyframe_filters_at(const uint8_t *in, uint8_t *lp, uint8_t *half, int W, int H,
                                                    int i, int j, int rowsY, uint8_t *copyTo) {
  const int W2 = 2 * W;
  if (j >= W2) return;
  if (copyTo && i < H && j < W) copyTo[i * W + j] = in[i * W + j];
  if (i < H && j < W) {
    int sum = 0;
    for (int m = i - 1; m <= i + 1; m++) {
      if (m < 0 || m >= H) continue;
      for (int n = j - 1; n <= j + 1; n++) {
        if (n < 0 || n >= W) continue;
        sum += in[m * W + n];
      }
    }
    lp[i * W + j] = (uint8_t)(sum / 9);
  }
  for (int ii = i; ii < 2 * H; ii += rowsY) {
    const int sub = (j & 1) + ((ii & 1) << 1), y = ii >> 1, x = j >> 1;
    const int tap[6] = {1, -5, 20, 20, -5, 1};
    int v;
    if (sub == 0) {
      v = in[imin(H - 1, y) * W + imin(W - 1, x)];
    } else if (sub == 1) {
      int s = 0;
      for (int q = 0; q < 6; q++) s += tap[q] * in[y * W + imax(0, imin(W - 1, x - 2 + q))];
      v = (s + 16) >> 5;
    } else if (sub == 2) {
      int s = 0;
      for (int q = 0; q < 6; q++) s += tap[q] * in[imax(0, imin(H - 1, y - 2 + q)) * W + x];
      v = (s + 16) >> 5;
    } else {
      int s = 0;
      for (int a = 0; a < 6; a++) {
        const int row = imax(0, imin(H - 1, y - 2 + a)) * W;
        int r = 0;
        for (int q = 0; q < 6; q++) r += tap[q] * in[row + imax(0, imin(W - 1, x - 2 + q))];
        s += tap[a] * r;
      }
      v = (s + 512) >> 10;
    }
    half[ii * W2 + j] = (uint8_t)imax(0, imin(255, v));
  }
}

__global__ void k_keyframe_filters(const uint8_t *in, uint8_t *lp, uint8_t *half, int W, int H) {
  keyframe_filters_at(in, lp, half, W, H, blockIdx.y, blockIdx.x * blockDim.x + threadIdx.x, gridDim.y, nullptr);
}

// blockIdx.z = key frame; rows and columns span the largest frame.
__global__ void k_keyframe_batch(const KeyFrameJob *jobs) {
  const KeyFrameJob kj = jobs[blockIdx.z];
  const int i = blockIdx.y, j = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 2 * kj.H) return;  // rows in [H, 2H) still own half-pel row i
  keyframe_filters_at(kj.src, kj.lp, kj.half, kj.W, kj.H, i, j, gridDim.y, kj.src != kj.full ? kj.full : nullptr);
}

// ------------------------------------------------------------ forward ME
// forwardME (sideInfoCreation.cpp:61-118): per macroblock of the future
// low-pass frame, exhaustive search of the past low-pass frame over the
// clipped +-32 window; cost SAD*(1 + K*|v|) in double, first minimum in raster
// order.  One workgroup per macroblock.  The window (up to 80 x 80 bytes) is
// staged in LDS as 32-bit words and the macroblock's 64 words sit in scalar
// registers; lane l of every wave takes candidate column l, the four waves
// take every fourth candidate row, and each candidate's SAD is 64 v_sad_u8 on
// window words byte-aligned with v_alignbyte (exact integer SADs, as the
// reference's integer sums are).  The 65th column of a full window is spread
// over the threads afterwards; ties go to the least raster index.
#define FME_LW 21  // staged words per window row: 20 + one zero word
__global__ __launch_bounds__(256) void k_forward_me(const FrameDev *F, const int *list, CostTables ct) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int bw = f.W / 16, nmb = bw * (f.H / 16), mb = blockIdx.x;
  if (mb >= nmb) return;
  const int W = f.W, top = (mb / bw) * 16, left = (mb % bw) * 16;
  const int sT = imax(0, top - 32), sB = imin(f.H - 16, top + 32);
  const int sL = imax(0, left - 32), sR = imin(W - 16, left + 32);  // sL is a multiple of 16
  const int ww = sR - sL + 1, wh = sB - sT + 1, winH = wh + 15, nw = (ww + 15) >> 2;  // nw <= 20
  __shared__ uint32_t win[80 * FME_LW];
  __shared__ uint32_t s_fb[64];
  __shared__ double s_cost[4];
  __shared__ int s_idx[4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (tid < 64) s_fb[tid] = *(const uint32_t *)(f.fut_lp + (size_t)(top + (tid >> 2)) * W + left + 4 * (tid & 3));
  for (int i = tid; i < winH * FME_LW; i += 256) {
    const int r = i / FME_LW, w = i - r * FME_LW;
    win[i] = w < nw ? *(const uint32_t *)(f.past_lp + (size_t)(sT + r) * W + sL + 4 * w) : 0u;
  }
  __syncthreads();
  uint32_t fb[64];
#pragma unroll
  for (int k = 0; k < 64; k++) fb[k] = __builtin_amdgcn_readfirstlane(s_fb[k]);
  auto sad_at = [&](int oy, int ox) -> uint32_t {
    const uint32_t *wr = win + oy * FME_LW + (ox >> 2);
    const int sh = ox & 3;
    uint32_t sad = 0;
#pragma unroll
    for (int m = 0; m < 16; m++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        sad = __builtin_amdgcn_sad_u8(fb[4 * m + q],
                                      __builtin_amdgcn_alignbyte(wr[m * FME_LW + q + 1], wr[m * FME_LW + q], sh), sad);
    return sad;
  };
  double best = DBL_MAX;
  int bidx = 0x7fffffff;
  if (lane < ww) {
    const double *fac = ct.fme + (sL + lane - left + 32);
    for (int oy = wave; oy < wh; oy += 4) {
      const double cost = (double)sad_at(oy, lane) * fac[(sT + oy - top + 32) * 65];
      if (cost < best) { best = cost; bidx = oy * ww + lane; }
    }
  }
  if (ww > 64)
    for (int oy = tid; oy < wh; oy += 256) {
      const double cost = (double)sad_at(oy, 64) * ct.fme[(sT + oy - top + 32) * 65 + sL + 64 - left + 32];
      if (cost < best || (cost == best && oy * ww + 64 < bidx)) { best = cost; bidx = oy * ww + 64; }
    }
  wave_argmin(best, bidx);
  if (lane == 0) { s_cost[wave] = best; s_idx[wave] = bidx; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; w++)
      if (s_cost[w] < best || (s_cost[w] == best && s_idx[w] < bidx)) { best = s_cost[w]; bidx = s_idx[w]; }
    const int px = sL + bidx % ww, py = sT + bidx / ww;
    MVd r;
    r.px = (double)px; r.py = (double)py; r.fx = 0.0; r.fy = 0.0;
    r.vx = (double)(px - left); r.vy = (double)(py - top);
    f.fwd[mb] = r;
    f.holes[2 * mb] = (double)left * f.iPC + (double)px * f.iFC;
    f.holes[2 * mb + 1] = (double)top * f.iPC + (double)py * f.iFC;
  }
}

// ------------------------------------------------------------ bidirectional ME chain
// Sums over the aligned groups of LEN (8 or 16) lanes, the same on each of
// them (quad permutes, then the mirrored half row and row).
template <int LEN>
__device__ __forceinline__ uint32_t group_sum(uint32_t v) {
  v += __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, false);   // quad_perm [1, 0, 3, 2]
  v += __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, false);   // quad_perm [2, 3, 0, 1]
  v += __builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, false);  // row_half_mirror
  if (LEN == 16) v += __builtin_amdgcn_mov_dpp(v, 0x140, 0xf, 0xf, false);  // row_mirror
  return v;
}
// Eight samples two bytes apart (a half-pel row's full-pel samples), packed in
// two words; the 16 bytes read need not be aligned.
__device__ __forceinline__ uint2 even_bytes(const uint8_t *p) {
  uint4 v;
  __builtin_memcpy(&v, p, 16);
  return make_uint2(__builtin_amdgcn_perm(v.y, v.x, 0x06040200), __builtin_amdgcn_perm(v.w, v.z, 0x06040200));
}

// One bidirectional search step of bidirectME (sideInfoCreation.cpp:250-306)
// for block blk, run by one wave; the block's range is bounded by its
// neighbours' current MVs (up/left already refined, down/right not yet).  A
// lane takes one row of one candidate's LEN x LEN samples (two or four 16-byte
// reads), 64 / LEN candidates at a time in raster order.  A lone candidate is taken without its cost, which is below the
// search's limit of 10^7 whatever the pixels (at most 255 * 16 * 16 * (1 +
// 0.05 * 996)).
struct HalfPair {  // a frame's two half-pel key frames, for the sweeps
  const uint8_t *past, *fut;
  int W2, H2;
  double scale;  // iPC / iFC
};
template <int LEN>
__device__ __forceinline__ void bidir_block(const HalfPair &f, MVs *mv, int blk, int i, int j, int bw, int bh,
                                            int lane) {
  constexpr int L2 = 2 * LEN, G = 64 / LEN;
  const int W2 = f.W2, bot = f.H2 - L2, right = W2 - L2, y2 = i * L2, x2 = j * L2;
  const MVs own = mv[blk];
  const int sT = i > 0 ? mv[blk - bw].fy + L2 : own.fy;
  const int sB = i + 1 < bh ? mv[blk + bw].fy - L2 : own.fy;
  const int sL = j > 0 ? mv[blk - 1].fx + L2 : own.fx;
  const int sR = j + 1 < bw ? mv[blk + 1].fx - L2 : own.fx;
  const int nx = sR - sL + 1, ny = sB - sT + 1;
  if (nx <= 0 || ny <= 0) return;
  const int n = nx * ny, row = lane % LEN, g = lane / LEN;
  // c / nx: (c + 0.5) / nx lies at least 0.5 / nx > 7e-4 from an integer and
  // below 576, so the float quotient's error (under 2e-4) never reaches one
  const float rnx = 1.0f / (float)nx;
  auto pos = [&](int c, int &fy, int &fx, int &py, int &px) {
    const int q = (int)(((float)c + 0.5f) * rnx);
    fy = sT + q;
    fx = sL + c - q * nx;
    py = end_point(y2, (double)(y2 - fy), f.scale, 0, bot);
    px = end_point(x2, (double)(x2 - fx), f.scale, 0, right);
  };
  double best = DBL_MAX;
  int bidx = n == 1 ? 0 : 0x7fffffff, fy, fx, py, px;
  if (n > 1) {
    for (int c0 = 0; c0 < n; c0 += G) {
      const int c = imin(c0 + g, n - 1);
      pos(c, fy, fx, py, px);
      const uint8_t *pr = f.past + (size_t)(py + 2 * row) * W2 + px;
      const uint8_t *fr = f.fut + (size_t)(fy + 2 * row) * W2 + fx;
      uint32_t sad = 0;
#pragma unroll
      for (int h = 0; h < LEN; h += 8) {
        const uint2 a = even_bytes(pr + 2 * h), b = even_bytes(fr + 2 * h);
        sad = __builtin_amdgcn_sad_u8(a.x, b.x, sad);
        sad = __builtin_amdgcn_sad_u8(a.y, b.y, sad);
      }
      const double cost = cost_func((double)(int)group_sum<LEN>(sad), (double)(px - fx), (double)(py - fy));
      if (c0 + g < n && cost < 10000000.0 && cost < best) { best = cost; bidx = c; }
    }
#pragma unroll
    for (int o = LEN; o < 64; o <<= 1) {
      const double c2 = __shfl_xor(best, o);
      const int i2 = __shfl_xor(bidx, o);
      if (c2 < best || (c2 == best && i2 < bidx)) { best = c2; bidx = i2; }
    }
  }
  if (lane == 0 && bidx != 0x7fffffff) {
    pos(bidx, fy, fx, py, px);
    mv[blk] = MVs{(short)fx, (short)fy, (short)px, (short)py};
  }
}

// Anti-diagonal sweep: blocks on diagonal d = i + j depend only on diagonal
// d-1 (refined) and d+1 (not yet refined), so this order equals the raster
// order of the in-place reference loop.
template <int LEN>
__device__ __forceinline__ void bidir_sweep(const HalfPair &f, MVs *mv) {
  const int bw = f.W2 / (2 * LEN), bh = f.H2 / (2 * LEN);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nwaves = blockDim.x >> 6;
  for (int d = 0; d <= bw + bh - 2; d++) {
    const int i0 = imax(0, d - (bw - 1)), i1 = imin(bh - 1, d);
    for (int i = i0 + wave; i <= i1; i += nwaves) bidir_block<LEN>(f, mv, i * bw + (d - i), i, d - i, bw, bh, lane);
    __syncthreads();
  }
}

// The serial part of createSideInfo (sideInfoCreation.cpp:119-143, 510-550)
// for one frame per workgroup: each macroblock's nearest hole, the 16x16 and
// the 8x8 bidirectional refinements, with the motion vectors in LDS.  With
// fwdOnly set it stops after forwardME's nearest-hole assignment (:119-143)
// and leaves the macroblock MVs unscaled (forwardME's own output).
// The two sweeps' 118 dependent diagonals (CIF) bound it.  With the vectors in
// global memory, a lane per candidate reading its samples byte by byte, and
// the filter and compensation below in the same single workgroup, this took
// 1930 us for a CIF frame and 550 for QCIF; now 403 and 89, and 8.5 for the
// filter and compensation in a grid of their own.
__global__ __launch_bounds__(1024) void k_si_sweep(const FrameDev *F, const int *list, int fwdOnly) {
  const FrameDev &f = F[list[blockIdx.x]];
  const int tid = threadIdx.x, W = f.W, H = f.H;
  const int bw16 = W / 16, nmb = bw16 * (H / 16), bw8 = W / 8, nb8 = bw8 * (H / 8);
  __shared__ double2 s_hole[22 * 18];
  __shared__ MVs s_mb[22 * 18];
  __shared__ MVs s_blk[44 * 36];
  for (int i = tid; i < nmb; i += 1024) s_hole[i] = make_double2(f.holes[2 * i], f.holes[2 * i + 1]);
  __syncthreads();
  // nearest hole per macroblock (:120-142), the holes split over two lanes,
  // and the x2 half-pel scaling (:511-521); ties go to the lower index
  if (tid < 2 * nmb) {
    const int i = tid >> 1, half = (nmb + 1) >> 1;
    const int top = (i / bw16) * 16, left = (i % bw16) * 16;
    double minDst = W * W + H * H;
    int best = 0;
    for (int jj = (tid & 1) * half; jj < ((tid & 1) ? nmb : half); jj++) {
      const double2 h = s_hole[jj];
      const double dst = (left - h.x) * (left - h.x) + (top - h.y) * (top - h.y);
      if (dst < minDst) { minDst = dst; best = jj; }
    }
    const double d2 = __shfl_xor(minDst, 1);
    const int b2 = __shfl_xor(best, 1);
    if ((tid & 1) == 0) {
      if (d2 < minDst) best = b2;
      const double vx = f.fwd[best].vx, vy = f.fwd[best].vy;
      const int fx = end_point(left, -vx, f.iFC, 0, W - 16), fy = end_point(top, -vy, f.iFC, 0, H - 16);
      const int px = end_point(left, vx, f.iPC, 0, W - 16), py = end_point(top, vy, f.iPC, 0, H - 16);
      s_mb[i] = MVs{(short)(2 * fx), (short)(2 * fy), (short)(2 * px), (short)(2 * py)};
      if (fwdOnly) {
        MVd o;
        o.fx = fx; o.fy = fy; o.px = px; o.py = py;
        o.vx = px - fx; o.vy = py - fy;
        f.mbmv[i] = o;
      }
    }
  }
  if (fwdOnly) return;
  __syncthreads();
  const HalfPair hp = {f.past_half, f.fut_half, 2 * W, 2 * H, f.iPC / f.iFC};
  bidir_sweep<16>(hp, s_mb);
  // 8x8 initial MVs from the 16x16 vectors (:524-545)
  for (int b = tid; b < nb8; b += 1024) {
    const int i = b / bw8, j = b % bw8, y2 = i << 4, x2 = j << 4;
    const MVs m = s_mb[(i >> 1) * bw16 + (j >> 1)];
    const double vx = m.px - m.fx, vy = m.py - m.fy;
    s_blk[b] = MVs{(short)end_point(x2, -vx, f.iFC, 0, (W - 8) << 1), (short)end_point(y2, -vy, f.iFC, 0, (H - 8) << 1),
                   (short)end_point(x2, vx, f.iPC, 0, (W - 8) << 1), (short)end_point(y2, vy, f.iPC, 0, (H - 8) << 1)};
  }
  __syncthreads();
  bidir_sweep<8>(hp, s_blk);
  for (int b = tid; b < nb8; b += 1024) f.bmv[b] = s_blk[b];
}

// motionFilterAndComp (sideInfoCreation.cpp:312-436): weighted vector-median
// filter over the 3x3 neighbourhood of 8x8 blocks, then motion compensation.
// One workgroup per 4x4 tile of 8x8 blocks; the tile's and its border's blocks'
// MSEs first (a lane per row of 8 samples), then 16 lanes per block, one per
// candidate vector, then a lane per four output pixels.
constexpr int SF_T = 4, SF_H = SF_T + 2;  // tile side and its side with the border
__global__ __launch_bounds__(256) void k_si_finish(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int tid = threadIdx.x, W = f.W, H = f.H, W2 = 2 * W, H2 = 2 * H, bw8 = W / 8, bh8 = H / 8;
  const int tw = (bw8 + SF_T - 1) / SF_T, th = (bh8 + SF_T - 1) / SF_T;
  if ((int)blockIdx.x >= tw * th) return;  // uniform over the workgroup
  const int ti = (blockIdx.x / tw) * SF_T, tj = (blockIdx.x % tw) * SF_T;
  __shared__ double s_mse[SF_H * SF_H];
  __shared__ MVs s_mv[SF_H * SF_H], s_new[SF_T * SF_T];
  __shared__ double s_w[SF_T * SF_T][9];
  // MSE per 8x8 block (:324-342): the sum of squared integer differences is
  // exact in double, so it equals the integer sum, formed as sum(a^2) +
  // sum(b^2) - 2 sum(a*b)
  for (int t = tid; t < SF_H * SF_H * 8; t += 256) {
    const int hb = t >> 3, row = t & 7, i = ti - 1 + hb / SF_H, j = tj - 1 + hb % SF_H;
    if (i < 0 || i >= bh8 || j < 0 || j >= bw8) continue;  // uniform over the block's 8 lanes
    const MVs m = f.bmv[i * bw8 + j];
    const uint2 a = even_bytes(f.fut_half + (size_t)(m.fy + 2 * row) * W2 + m.fx);
    const uint2 b = even_bytes(f.past_half + (size_t)(m.py + 2 * row) * W2 + m.px);
    uint32_t sq = __builtin_amdgcn_udot4(a.x, a.x, 0u, false), ab = __builtin_amdgcn_udot4(a.x, b.x, 0u, false);
    sq = __builtin_amdgcn_udot4(a.y, a.y, sq, false);
    sq = __builtin_amdgcn_udot4(b.x, b.x, sq, false);
    sq = __builtin_amdgcn_udot4(b.y, b.y, sq, false);
    ab = __builtin_amdgcn_udot4(a.y, b.y, ab, false);
    const uint32_t sse = group_sum<8>(sq - 2u * ab);
    if (row == 0) {
      s_mse[hb] = (double)(int)sse / 64;
      s_mv[hb] = m;
    }
  }
  __syncthreads();
  const int lb = tid >> 4, c = tid & 15, bi = ti + lb / SF_T, bj = tj + lb % SF_T;
  const bool live = bi < bh8 && bj < bw8;
  // the block's neighbourhood in raster order: rows r0.., ncol columns from q0
  const int r0 = imax(0, bi - 1), q0 = imax(0, bj - 1);
  const int ncol = imin(bw8 - 1, bj + 1) - q0 + 1, cnt = ncol * (imin(bh8 - 1, bi + 1) - r0 + 1);
  auto nbr = [&](int k) { return (r0 + k / ncol - ti + 1) * SF_H + q0 + k % ncol - tj + 1; };
  if (live && c < cnt) {
    const int me = nbr(c);
    const MVs m = s_mv[me];
    const double mse = s_mse[me], vx = m.px - m.fx, vy = m.py - m.fy;
    double w = 0.0;
    for (int k = 0; k < cnt; k++) {
      if (c == k) continue;
      const int o = nbr(k);
      const MVs n = s_mv[o];
      const double dx = vx - (n.px - n.fx), dy = vy - (n.py - n.fy);
      w += mse / s_mse[o] * sqrt(dx * dx + dy * dy);
    }
    s_w[lb][c] = w;
  }
  __syncthreads();
  if (live && c == 0) {
    double minW = s_w[lb][0];
    int best = 0;
    for (int k = 1; k < cnt; k++)
      if (s_w[lb][k] < minW) { minW = s_w[lb][k]; best = k; }
    const MVs m = s_mv[nbr(best)];
    const int y2 = bi << 4, x2 = bj << 4;
    const double vx = m.px - m.fx, vy = m.py - m.fy;
    s_new[lb] = MVs{(short)end_point(x2, -vx, f.iFC, 0, W2 - 16), (short)end_point(y2, -vy, f.iFC, 0, H2 - 16),
                    (short)end_point(x2, vx, f.iPC, 0, W2 - 16), (short)end_point(y2, vy, f.iPC, 0, H2 - 16)};
  }
  __syncthreads();
  if (!live) return;
  // motion compensation (:407-434): pixels 4 * (c & 1) .. of row c >> 1
  const MVs m = s_new[lb];
  const int row = c >> 1, x = 4 * (c & 1);
  uint2 fw, pw;
  __builtin_memcpy(&fw, f.fut_half + (size_t)(m.fy + 2 * row) * W2 + m.fx + 2 * x, 8);
  __builtin_memcpy(&pw, f.past_half + (size_t)(m.py + 2 * row) * W2 + m.px + 2 * x, 8);
  const uint32_t fb = __builtin_amdgcn_perm(fw.y, fw.x, 0x06040200), pb = __builtin_amdgcn_perm(pw.y, pw.x, 0x06040200);
  uint32_t out = 0;
  int res[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int fv = (fb >> (8 * q)) & 0xff, pv = (pb >> (8 * q)) & 0xff;
    out |= (uint32_t)(uint8_t)(int)((double)fv * f.iFC + (double)pv * f.iPC) << (8 * q);
    res[q] = (fv - pv) >> 1;
  }
  const size_t o = (size_t)(8 * bi + row) * W + 8 * bj + x;
  *(uint32_t *)(f.si + o) = out;
  *(int4 *)(f.residue + o) = make_int4(res[0], res[1], res[2], res[3]);
}

// ------------------------------------------------------------ transform helpers
__device__ __forceinline__ int round_d(double x) { return x >= 0.0 ? (int)(x + 0.5) : -(int)(-x + 0.5); }

// forward44 (transform.cpp:63-104) with the double post-scale of initTransform (:12-33).
__device__ void forward44(int *blk) {
  // b = sqrt(0.4) as the host's correctly rounded double (transform.cpp:14)
  const double a2 = 0.25, ab2 = 0.5 * 0x1.43d136248490fp-1 / 2, b24 = 0.4 / 4;
  int t[16];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int x0 = blk[c], x1 = blk[4 + c], x2 = blk[8 + c], x3 = blk[12 + c];
    t[c] = x0 + x1 + x2 + x3;
    t[4 + c] = (x0 << 1) + x1 - x2 - (x3 << 1);
    t[8 + c] = x0 - x1 - x2 + x3;
    t[12 + c] = x0 - (x1 << 1) + (x2 << 1) - x3;
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int x0 = t[4 * r], x1 = t[4 * r + 1], x2 = t[4 * r + 2], x3 = t[4 * r + 3];
    blk[4 * r] = x0 + x1 + x2 + x3;
    blk[4 * r + 1] = (x0 << 1) + x1 - x2 - (x3 << 1);
    blk[4 * r + 2] = x0 - x1 - x2 + x3;
    blk[4 * r + 3] = x0 - (x1 << 1) + (x2 << 1) - x3;
  }
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int r = i >> 2, c = i & 3;
    const double ps = ((r & 1) == 0 && (c & 1) == 0) ? a2 : (((r & 1) && (c & 1)) ? b24 : ab2);
    blk[i] = round_d((double)blk[i] * ps);
  }
}

// inverse44 (transform.cpp:106-151) with preScale*64.
__device__ void inverse44(int *blk) {
  const double a2 = 0.25 * 64.0, ab = 0.5 * 0x1.43d136248490fp-1 * 64.0, b2 = 0.4 * 64.0;
  int t[16];
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int r = i >> 2, c = i & 3;
    const double ps = ((r & 1) == 0 && (c & 1) == 0) ? a2 : (((r & 1) && (c & 1)) ? b2 : ab);
    blk[i] = round_d((double)blk[i] * ps);
  }
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int x0 = blk[c], x1 = blk[4 + c], x2 = blk[8 + c], x3 = blk[12 + c];
    t[c] = x0 + x1 + x2 + (x3 >> 1);
    t[4 + c] = x0 + (x1 >> 1) - x2 - x3;
    t[8 + c] = x0 - (x1 >> 1) - x2 + x3;
    t[12 + c] = x0 - x1 + x2 - (x3 >> 1);
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int x0 = t[4 * r], x1 = t[4 * r + 1], x2 = t[4 * r + 2], x3 = t[4 * r + 3];
    blk[4 * r] = x0 + x1 + x2 + (x3 >> 1);
    blk[4 * r + 1] = x0 + (x1 >> 1) - x2 - x3;
    blk[4 * r + 2] = x0 - (x1 >> 1) - x2 + x3;
    blk[4 * r + 3] = x0 - x1 + x2 - (x3 >> 1);
  }
#pragma unroll
  for (int i = 0; i < 16; i++) blk[i] >>= 6;
}

__constant__ int c_zigzag[16] = {0, 1, 4, 8, 5, 2, 3, 6, 9, 12, 13, 10, 7, 11, 14, 15};
__constant__ int c_qbits[9][16] = {
    {0},
    {4, 3, 0, 0, 3, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0},
    {5, 3, 0, 0, 3, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0},
    {5, 3, 2, 0, 3, 2, 0, 0, 2, 0, 0, 0, 0, 0, 0, 0},
    {5, 4, 3, 2, 4, 3, 2, 0, 3, 2, 0, 0, 2, 0, 0, 0},
    {5, 4, 3, 2, 4, 3, 2, 2, 3, 2, 2, 0, 2, 2, 0, 0},
    {6, 4, 3, 3, 4, 3, 3, 2, 3, 3, 2, 2, 3, 2, 2, 0},
    {6, 5, 4, 3, 5, 4, 3, 2, 4, 3, 2, 2, 3, 2, 2, 0},
    {7, 6, 5, 4, 6, 5, 4, 3, 5, 4, 3, 2, 4, 3, 2, 0}};

// ------------------------------------------------------------ noise parameter
// forwardTransform of the residue (transform.cpp:153-190) and noiseParameter
// (noiseModel.cpp:9-75).  The reference's band means and second moments are
// float sums over all blocks in raster order.  Every term is a non-negative
// integer, so while a total stays at or below 2^24 every partial sum is exact
// and the float sum equals the integer sum in any order: the coefficients, at
// most 512 in magnitude for a residue in [-128, 127], always stay there (6336 *
// 512 < 2^22), their squares do unless the mean square exceeds 2648 (CIF), and
// only then is the sum taken in order.  Three launches: transform and integer
// partial sums per 256 blocks, the bands' moments, alpha.  One workgroup per
// frame with each band's sum on one thread took 955 us for a CIF frame and 205
// for QCIF, a chain of N dependent loads and additions; now 17 and 15.
// Per 256 4x4 blocks: sideTrans and the 16 coefficients' partial sums.
__global__ __launch_bounds__(256) void k_residue_transform(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int tid = threadIdx.x, W = f.W, bw = W / 4, b0 = blockIdx.x * 256;
  if (b0 >= f.N) return;  // uniform over the workgroup
  __shared__ short s_c[256][17];
  __shared__ uint2 s_part[4][16];
  const int b = b0 + tid, top = (b / bw) * 4, left = (b % bw) * 4;
  int blk[16] = {};
  if (b < f.N) {
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const int4 v = *(const int4 *)(f.residue + (size_t)(top + m) * W + left);
      blk[4 * m] = v.x; blk[4 * m + 1] = v.y; blk[4 * m + 2] = v.z; blk[4 * m + 3] = v.w;
    }
    forward44(blk);
#pragma unroll
    for (int m = 0; m < 4; m++)
      *(int4 *)(f.sideTrans + (size_t)(top + m) * W + left) =
          make_int4(blk[4 * m], blk[4 * m + 1], blk[4 * m + 2], blk[4 * m + 3]);
  }
#pragma unroll
  for (int k = 0; k < 16; k++) s_c[tid][k] = (short)abs(blk[k]);
  __syncthreads();
  // thread (part, coefficient) sums 16 blocks, then the 4 parts of a wave and
  // the 4 waves (a workgroup's sums of squares stay below 2^27)
  const int k = tid & 15, part = tid >> 4;
  uint32_t s1 = 0, s2 = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const uint32_t c = s_c[part * 16 + i][k];
    s1 += c;
    s2 += c * c;
  }
  for (int o = 16; o < 64; o <<= 1) {
    s1 += __shfl_xor(s1, o);
    s2 += __shfl_xor(s2, o);
  }
  if ((tid & 63) < 16) s_part[tid >> 6][k] = make_uint2(s1, s2);
  __syncthreads();
  if (tid >= 16) return;
  for (int w = 1; w < 4; w++) {
    s1 += s_part[w][k].x;
    s2 += s_part[w][k].y;
  }
  f.npPart[blockIdx.x * 16 + k] = make_uint2(s1, s2);
}
// One workgroup per (band, frame): mean and variance of the band's magnitudes.
__global__ __launch_bounds__(256) void k_noise_moments(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int tid = threadIdx.x, index = c_zigzag[blockIdx.x], N = f.N, W = f.W, bw = W / 4;
  if (c_qbits[f.qindex][index] <= 0) return;  // uniform: not one of the frame's bands
  __shared__ __align__(16) float s_sq[6336 + 64];
  const int parts = (N + 255) / 256;  // at most 25
  uint2 p = tid < parts ? f.npPart[tid * 16 + index] : make_uint2(0, 0);
  uint32_t sq = p.y;  // the squares total at most 6336 * 512^2 < 2^31
  if (tid < 64)
    for (int o = 32; o > 0; o >>= 1) {
      p.x += __shfl_xor(p.x, o);
      sq += __shfl_xor(sq, o);
    }
  float var = (float)sq;
  // (the first wave holds the totals)
  const int inOrder = __syncthreads_or(tid < 64 && sq > (1u << 24));
  if (inOrder) {
    // the squares past 2^24: their float sum in raster order
    for (int b = tid; b < N; b += 256) {
      const float c = (float)f.sideTrans[((b / bw) * 4 + (index >> 2)) * W + (b % bw) * 4 + (index & 3)];
      s_sq[b] = c * c;
    }
    if (tid < 64) s_sq[N + tid] = 0.0f;  // +0 past the last block leaves the sum as it is
    __syncthreads();
    if (tid >= 64) return;
    var = 0.0f;
    for (int b = 0; b < N; b += 64) {
      const float4 *q = (const float4 *)(s_sq + b);
      float4 a[16];
#pragma unroll
      for (int i = 0; i < 16; i++) a[i] = q[i];
#pragma unroll
      for (int i = 0; i < 16; i++) {
        var += a[i].x;
        var += a[i].y;
        var += a[i].z;
        var += a[i].w;
      }
    }
  }
  if (tid == 0) {
    const float mean = (float)p.x / (float)N;
    f.npMom[index] = make_float2(mean, var / (float)N - mean * mean);
  }
}
// alpha of every block at the frame's bands, 0 at the other coefficients; a
// thread per 4x4 block.
__global__ __launch_bounds__(256) void k_noise_alpha(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int b = blockIdx.x * 256 + threadIdx.x, W = f.W, bw = W / 4;
  if (b >= f.N) return;
  const int top = (b / bw) * 4, left = (b % bw) * 4;
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const size_t o = (size_t)(top + m) * W + left;
    const int4 v = *(const int4 *)(f.sideTrans + o);
    const int c4[4] = {v.x, v.y, v.z, v.w};
    float a4[4];
#pragma unroll
    for (int n = 0; n < 4; n++) {
      a4[n] = 0.0f;
      if (c_qbits[f.qindex][4 * m + n] <= 0) continue;  // uniform
      const float2 mom = f.npMom[4 * m + n];
      const float dst = (float)abs(c4[n]) - mom.x;
      const float dst2 = dst * dst;
      a4[n] = dst2 > mom.y ? sqrtf(2 / dst2) : sqrtf(2 / mom.y);
    }
    *(float4 *)(f.alpha + o) = make_float4(a4[0], a4[1], a4[2], a4[3]);
  }
}

// ------------------------------------------------------------ over-complete transform
// overCompleteTransform (transform.cpp:275-298); with initSideTrans, also
// init_si_ML (motionLearning.cpp:49-68) from the block-aligned positions.
// Each position's coefficient of the band whose noise distribution comes next
// (band 0 at the frame's start, else band + 1) also goes to the octBand plane,
// so that kernel reads 4 contiguous bytes per window position instead of one
// int out of each 64-byte record.
// A workgroup's 256 consecutive positions span at most 3 position rows of a
// frame at least 176 wide, so the side-information rows under them (at most
// 6) are staged in LDS as words with aligned loads, and each position's 4x4
// pixels are taken from there (4 byte alignments) instead of 16 byte loads.
// The 64-byte records of a wave's 64 positions go out through LDS so that each
// store instruction writes 1 KB of consecutive bytes.
#define OCT_ROWS 6
#define OCT_LW 89  // words per staged row: 352 / 4 + one for the byte alignment
__global__ __launch_bounds__(256) void k_oct(const FrameDev *F, const int *list, int initSideTrans) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int ow = f.W - 3, npos = ow * (f.H - 3), W = f.W, nw = W >> 2;
  const int p0 = blockIdx.x * 256;
  if (p0 >= npos) return;  // uniform over the workgroup
  __shared__ uint32_t s_rows[OCT_ROWS * OCT_LW];
  __shared__ int4 s_rec[256 * 4];  // the workgroup's records, position-major
  const int top0 = p0 / ow, rows = imin(f.H, (imin(p0 + 255, npos - 1) / ow) + 4) - top0;  // <= OCT_ROWS
  for (int i = threadIdx.x; i < rows * OCT_LW; i += 256) {
    const int r = i / OCT_LW, w = i - r * OCT_LW;
    s_rows[i] = w < nw ? *(const uint32_t *)(f.si + (size_t)(top0 + r) * W + 4 * w) : 0u;
  }
  __syncthreads();
  const int p = p0 + threadIdx.x;
  const bool valid = p < npos;
  const int top = valid ? p / ow : top0, left = valid ? p % ow : 0, j = left >> 2, sh = left & 3;
  const uint32_t *R = s_rows + (top - top0) * OCT_LW + j;
  int blk[16];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const uint32_t v = __builtin_amdgcn_alignbyte(R[m * OCT_LW + 1], R[m * OCT_LW], sh);
#pragma unroll
    for (int n = 0; n < 4; n++) blk[4 * m + n] = (v >> (8 * n)) & 0xff;
  }
  forward44(blk);
  int4 *rec = s_rec + 4 * threadIdx.x;
  rec[0] = make_int4(blk[0], blk[1], blk[2], blk[3]);
  rec[1] = make_int4(blk[4], blk[5], blk[6], blk[7]);
  rec[2] = make_int4(blk[8], blk[9], blk[10], blk[11]);
  rec[3] = make_int4(blk[12], blk[13], blk[14], blk[15]);
  if (valid) {
    const int nb = initSideTrans ? 0 : f.band + 1;
    if (nb < 16) f.octBand[p] = blk[c_zigzag[nb]];
    if (initSideTrans && (top & 3) == 0 && (left & 3) == 0 && top <= f.H - 4 && left <= f.W - 4)
      for (int m = 0; m < 4; m++)
        for (int n = 0; n < 4; n++) f.sideTrans[(top + m) * W + left + n] = blk[4 * m + n];
  }
  __syncthreads();
  // store i writes the workgroup's 16-byte pieces 256 i + t: position p0 + 64 i + t / 4
  int4 *dst = (int4 *)(f.oct + (size_t)16 * p0);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int piece = 256 * i + threadIdx.x;
    if (p0 + (piece >> 2) < npos) dst[piece] = s_rec[piece];
  }
}

// SMF window of WZ block b (initSMF, motionLearning.cpp:6-47).
struct SmfWin { int top, left, sT, sB, sL, sR, w, len, self; };
__device__ __forceinline__ SmfWin smf_window(const FrameDev &f, int b) {
  SmfWin s;
  const int bw = f.W / 4;
  s.top = (b / bw) * 4; s.left = (b % bw) * 4;
  s.sT = imax(0, s.top - 4); s.sB = imin(f.H - 4, s.top + 4);
  s.sL = imax(0, s.left - 4); s.sR = imin(f.W - 4, s.left + 4);
  s.w = s.sR - s.sL + 1;
  s.len = s.w * (s.sB - s.sT + 1);
  s.self = (s.top - s.sT) * s.w + (s.left - s.sL);
  return s;
}

__global__ void k_smf_init(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= f.N) return;
  const SmfWin s = smf_window(f, b);
  for (int p = 0; p < 81; p++) f.smf[(size_t)81 * b + p] = (p == s.self) ? 1.0f : 0.0f;
}

// ------------------------------------------------------------ noise distribution
// noiseDistribution (noiseModel.cpp:77-132): DC prob[k] = expf(-a*|k - SI_DC|);
// AC prob[k] = sum_m p_m * expf(-a*|k - range - SI_m|), m in window raster
// order.  A window term whose probability is exactly +0 adds +0 to a
// non-negative sum and is skipped when a is finite.  The exponent depends on
// the integer distance d = |k - range - SI_m| only, so each workgroup first
// tabulates expf(-a*(float)d) for the distances its block can reach (the same
// values, bit for bit) and the mixture sums then read the table.  One wave
// per (4x4 block, frame): a block has 2*range+1 <= ~520 values at most
// Qindex 8, and the small workgroup with a 4 KB table lets a CU hold many
// blocks at once to hide the LDS and global latencies of each one's phases.
// A value is +0 where every term's expf underflows, a*d > 104, which for the
// usual a around 1 leaves most of the range zero (a DC row has 1024 values, an
// AC row up to about 1000).  The block's span is the interval outside which
// all values are +0: only it is computed and, for the frame decoder, stored;
// condBitProb's sums are clipped to it, as adding +0 changes none of them.
// With every value computed and stored, a band of 256 CIF frames took 2237 us on
// average (the DC band 3417); now 2124 (2883).  The rest is the sums' products
// and additions, 8 of the 9 VALU instructions per term and four values.
#define ND_TAB 1024  // table entries (4 KB of LDS); larger distances call expf directly
#define ND_T 64      // threads per block distribution (one wave)
// The least distance from which expf(-a * d) is certainly +0 (it is below
// -103.98, and the quotient's and product's roundings stay within the slack),
// or 2^20 where no distance is taken to be.
__device__ __forceinline__ int nd_reach(float a) {
  const float q = 104.0f / a;
  return a > 0.0f && q < 1048000.0f ? (int)q + 2 : 1 << 20;
}
// V values k + i*ND_T (i < V) of one block's distribution: sum over the window
// terms m in order of p_m * tab[value + off_m].  Values at or beyond rmax are
// computed from the table's padding (never from outside it) and not stored.
template <int V>
__device__ __forceinline__ void nd_values(const float *tab, const int2 *ps, int n, int k, int rmax, float *out) {
  float acc[V];
#pragma unroll
  for (int i = 0; i < V; i++) acc[i] = 0.0f;
  for (int m = 0; m < n; m++) {
    const int2 t = ps[m];
    const float pr = __int_as_float(t.x);
    const float *tk = tab + k + t.y;
#pragma unroll
    for (int i = 0; i < V; i++) acc[i] += pr * tk[i * ND_T];
  }
#pragma unroll
  for (int i = 0; i < V; i++)
    if (k + i * ND_T < rmax) out[k + i * ND_T] = acc[i];
}
// fill: also store the zeros outside the span (callers that read whole rows).
__global__ __launch_bounds__(64) void k_noise_dist(const FrameDev *F, const int *list, int fill) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int b = blockIdx.x;
  if (b >= f.N || !wz_block(f, b)) return;  // only SIR candidates have a distribution
  const int tid = threadIdx.x, T = ND_T;
  const int ow = f.W - 3, index = f.index, range = f.range;
  const int rmax = index ? 2 * range + 1 : range;  // values of the row
  const SmfWin s = smf_window(f, b);
  const float a = f.alpha[(s.top + (index >> 2)) * f.W + s.left + (index & 3)];
  float *out = f.dist + (size_t)b * f.distStride;
  int reach = nd_reach(a);
  auto put_span = [&](int lo, int hi) {  // [lo, hi) within [0, rmax], possibly empty
    if (tid == 0) f.distSpan[b] = make_int2(lo, hi);
    if (!fill) return;
    for (int k = tid; k < lo; k += T) out[k] = 0.0f;
    for (int k = hi + tid; k < rmax; k += T) out[k] = 0.0f;
  };
  if (index == 0) {
    const int side = f.octBand[s.top * ow + s.left];
    const int lo = imin(rmax, imax(0, side - reach + 1)), hi = imax(lo, imin(rmax, side + reach));
    put_span(lo, hi);
    for (int k = lo + tid; k < hi; k += T) out[k] = dvc_expf(-a * (float)abs(k - side));
    return;
  }
  __shared__ int2 s_ps[81];  // (probability bits, SI coefficient) of the kept window terms
  // table entries [0, 2D] with 2D + 1 <= ND_TAB, and 3 * ND_T of padding that a
  // lane's values beyond the span (at most 3 * ND_T further on) may read
  __shared__ float s_tab[ND_TAB + 3 * ND_T];
  // compact the window's non-zero terms in raster order
  const bool fin = isfinite(a);
  const float rw = __builtin_amdgcn_rcpf((float)s.w);
  int n = 0, mn = 0x7fffffff, mx = -0x7fffffff;
  bool odd = false;  // some kept probability is not finite: it makes NaN of the zeros
  for (int base = 0; base < s.len; base += 64) {
    const int p = base + tid;
    float pr = 0.0f;
    bool keep = false;
    if (p < s.len) {
      pr = f.smf[(size_t)81 * b + p];
      keep = !(fin && pr == 0.0f);
    }
    const unsigned long long mask = __ballot(keep);
    if (keep) {
      const int pos = n + __popcll(mask & ((1ull << tid) - 1ull));
      const int m = (int)(((float)p + 0.5f) * rw);  // p / s.w, at least 0.5 / 9 from rounding over
      const int sd = f.octBand[(s.sT + m) * ow + s.sL + p - m * s.w];
      s_ps[pos] = make_int2(__float_as_int(pr), sd);
      mn = imin(mn, sd);
      mx = imax(mx, sd);
      odd |= !isfinite(pr);
    }
    n += __popcll(mask);
  }
  mn = wave_reduce(mn, [](int x, int y) { return imin(x, y); });
  mx = wave_reduce(mx, [](int x, int y) { return imax(x, y); });
  if (n == 0) {
    put_span(0, 0);
    return;
  }
  if (__ballot(odd)) reach = 1 << 20;
  const int lo = imin(rmax, imax(0, range + mn - reach + 1)), hi = imax(lo, imin(rmax, range + mx + reach));
  put_span(lo, hi);
  // |k - range - SI_m| for k in the span: within it by reach + (mx - mn), and in
  // any case by range + max|SI_m|
  const int D = imin(range + imax(abs(mn), abs(mx)), reach + mx - mn);
  if (2 * D + 1 <= ND_TAB) {
    // two-sided table s_tab[D + t] = expf(-a*|t|), t in [-D, D]: term m of
    // value k reads s_tab[k + off_m] with off_m = D - range - SI_m
    for (int d = tid; d <= D; d += T) {
      const float v = dvc_expf(-a * (float)d);
      s_tab[D + d] = v;
      s_tab[D - d] = v;
    }
    __syncthreads();
    for (int m = tid; m < n; m += T) s_ps[m].y = D - range - s_ps[m].y;
    __syncthreads();
    // a lane's values k, k + T, ... share each term's offset and carry
    // independent sums; each value still adds its terms in window order.  The
    // number of values per lane is the same on every lane (groups of up to 4).
    int k = lo + tid, left = (hi - lo + T - 1) / T;
    for (; left >= 4; left -= 4, k += 4 * T) nd_values<4>(s_tab, s_ps, n, k, hi, out);
    if (left == 3) nd_values<3>(s_tab, s_ps, n, k, hi, out);
    else if (left == 2) nd_values<2>(s_tab, s_ps, n, k, hi, out);
    else if (left == 1) nd_values<1>(s_tab, s_ps, n, k, hi, out);
  } else {
    const int need = D + 1;
    const int tl = imin(need, ND_TAB);
    for (int d = tid; d < tl; d += T) s_tab[d] = dvc_expf(-a * (float)d);
    __syncthreads();
    for (int k = lo + tid; k < hi; k += T) {
      const int pc = k - range;
      float sum = 0.0f;
      for (int m = 0; m < n; m++) {
        const int2 ps = s_ps[m];
        const int d = abs(pc - ps.y);
        const float e = d < tl ? s_tab[d] : dvc_expf(-a * (float)d);
        sum += __int_as_float(ps.x) * e;
      }
      out[k] = sum;
    }
  }
}

// ------------------------------------------------------------ conditional bit probability
// condBitProb (noiseModel.cpp:191-310): interval sums in ascending k, p0/(p0+p1),
// clipped likelihood ratio.  Two lanes per block, one per interval, each adding
// its own interval's values in ascending k, as the reference's loops do, clipped
// to the block's span (the values outside are +0).  The wave stages the 64
// intervals through LDS in chunks of C values (each load a contiguous piece of
// two intervals), the next chunk's loads issued before this chunk is summed.
// HBM bounds a large batch, the chain of chunks a single frame: with a lane per
// block adding both intervals of the whole row, a launch for one CIF frame took
// 21 us on average and up to 128, for 256 frames 199; now 9.5, 37 and 172.
template <int C>
__device__ __forceinline__ float interval_sum(const float *dist, size_t stride, const int2 *iv, float *v, int lane,
                                              int span) {
  constexpr int R = 64 / C, LD = C + 4;  // rows per load; row length in LDS, 16-byte aligned
  const int i = lane % C, jr = lane / C;
  float nxt[C];
  auto fetch = [&](int c0) {
#pragma unroll
    for (int l = 0; l < C; l++) {
      const int j = l * R + jr;
      const int2 r = iv[j];
      const int k = r.x + c0 + i;
      nxt[l] = k < r.y ? dist[(size_t)(j >> 1) * stride + k] : 0.0f;
    }
  };
  float sum = 0.0f;
  if (span > 0) fetch(0);
  for (int c0 = 0; c0 < span; c0 += C) {
#pragma unroll
    for (int l = 0; l < C; l++) v[(l * R + jr) * LD + i] = nxt[l];
    __syncthreads();
    if (c0 + C < span) fetch(c0 + C);
    const float4 *q = (const float4 *)(v + lane * LD);
#pragma unroll
    for (int t = 0; t < C / 4; t++) {
      // past the interval's end the values are +0, which changes no sum
      const float4 x = q[t];
      sum += x.x;
      sum += x.y;
      sum += x.z;
      sum += x.w;
    }
    __syncthreads();
  }
  return sum;
}
__global__ __launch_bounds__(64) void k_condbit(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int lane = threadIdx.x;
  const int b0 = blockIdx.x * 32;
  if (b0 >= f.N) return;  // uniform over the wave
  __shared__ __align__(16) float s_v[64 * 36];
  __shared__ int2 s_iv[64];
  const int b = b0 + (lane >> 1), one = lane & 1;
  const bool valid = b < f.N;
  const bool wz = valid && wz_block(f, b);  // condBitProb walks the SIR's WZ blocks
  int lo = 0, hi = 0;
  if (wz) {
    const int bw = f.W / 4, top = (b / bw) * 4, left = (b % bw) * 4;
    const int index = f.index, bit = f.bit, step = f.step, range = f.range;
    const int iq = (1 << (bit - 1)) - 1;
    const int rc = f.reconsTrans[(top + (index >> 2)) * f.W + left + (index & 3)];
    // the quantisation indices of bit value `one`
    int ql = one ? ((rc << 1) + 1) << (bit - 1) : rc << bit;
    if (index == 0) {
      lo = ql * step;
      hi = (ql + iq + 1) * step;
    } else {
      const int ls = f.levelShift;
      ql -= ls;
      int qu = ql + iq;
      if (one && qu > ls) qu = ls;
      lo = ((ql <= 0) ? (ql - 1) * step + 1 : ql * step) + range;
      hi = ((qu < 0) ? qu * step + 1 : (qu + 1) * step) + range;
    }
    const int2 sp = f.distSpan[b];  // within [0, values of the row]
    lo = imax(lo, sp.x);
    hi = imin(hi, sp.y);
  }
  s_iv[lane] = make_int2(lo, hi);
  const int span = wave_reduce(imax(0, hi - lo), [](int x, int y) { return imax(x, y); });
  __syncthreads();
  const float *dist = f.dist + (size_t)b0 * f.distStride;
  // short intervals (the lower bits) load in pieces of 16 values
  const float mine = span <= 16 ? interval_sum<16>(dist, f.distStride, s_iv, s_v, lane, span)
                                : interval_sum<32>(dist, f.distStride, s_iv, s_v, lane, span);
  const float other = __shfl_xor(mine, 1);
  if (!valid || one) return;
  if (!wz) {
    // the frame's LR are first set to 0.9999f / 0.0001f when it has skip or
    // intra blocks (DVC_Decoder.cpp:203-207); WZ blocks overwrite theirs
    f.LR[b] = 0.9999f / 0.0001f;
    return;
  }
  const float p0 = mine / (mine + other), p1 = 1 - p0;
  float lr;
  if ((double)p0 <= 0.0001) lr = (float)(0.0001 / 0.9999);
  else if ((double)p0 >= 0.9999) lr = (float)(0.9999 / 0.0001);
  else lr = p0 / p1;
  f.LR[b] = lr;
}

// ------------------------------------------------------------ bitplane -> coefficients
// putBitplaneToCoeff (bitplane.cpp:4-22) with the bits of the code the rate
// search accepted (its record names the decision slot).
__global__ void k_put_bitplane(const FrameDev *F, const int *list, const BpFrameLink *links) {
  const int fi = list[blockIdx.y];
  const FrameDev &f = F[fi];
  const BpFrameLink &lk = links[blockIdx.y];
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= f.N) return;
  const int best = lk.state->best;
  const int slot = (best >= 0 && best < kMaxCodes) ? lk.records[best].z : -1;
  if (slot < 0 || slot >= lk.slot_capacity) return;  // the host reports the missing record
  const uint8_t bitv = lk.slots[(size_t)slot * f.N + b];
  f.decoded[b] = bitv;
  if (lk.carry) lk.carry[b] = bitv;  // ParallelMode 1: the next bitplane starts from these decisions
  if (!wz_block(f, b)) return;      // putBitplaneToCoeff (bitplane.cpp:4-22) skips other blocks
  const int bw = f.W / 4, top = (b / bw) * 4, left = (b % bw) * 4, index = f.index;
  int *p = &f.reconsTrans[(top + (index >> 2)) * f.W + left + (index & 3)];
  *p = (*p << 1) + (int)bitv;
}

// ------------------------------------------------------------ reconstruction
// reconstruction (reconstruction.cpp:184-289).  exp is dvc_exp, the host C
// library's double exp restated bit for bit, and the remaining operations are
// the same IEEE double operations in the same order without contraction, so
// every reconstructed coefficient equals the CPU path's.
__global__ void k_reconstruct(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= f.N || !wz_block(f, b)) return;
  const int bw = f.W / 4, top = (b / bw) * 4, left = (b % bw) * 4, index = f.index, step = f.step;
  const int ci = (top + (index >> 2)) * f.W + left + (index & 3);
  const int side = f.sideTrans[ci];
  const double a = f.alpha[ci];
  int lo, hi;
  if (index == 0) {
    const int q = f.reconsTrans[ci];
    lo = q * step; hi = (q + 1) * step;
  } else {
    const int q = f.reconsTrans[ci] - f.levelShift;
    if (q == 0) { lo = -step + 1; hi = step; }
    else if (q > 0) { lo = q * step; hi = (q + 1) * step; }
    else { lo = (q - 1) * step + 1; hi = q * step + 1; }
  }
  int v;
  if (a <= 0.0001) {
    v = (lo + hi) / 2;
  } else if (side < lo) {
    v = lo + round_d(1.0 / a + (double)step / (1.0 - dvc_exp(a * (double)step)));
  } else if (side >= hi) {
    v = hi - round_d(1.0 / a + (double)step / (1.0 - dvc_exp(a * (double)step)));
  } else {
    const double r = side - lo, d = hi - side;
    const double er = dvc_exp(-a * r), ed = dvc_exp(-a * d);
    v = side + round_d(((r + 1.0 / a) * er - (d + 1.0 / a) * ed) / (2.0 - (er + ed)));
  }
  f.sideTrans[ci] = v;
  if (f.dbFlag) f.dbFlag[ci] = v != side;  // deblockFlag: reconstruction moved the coefficient
}

// inverseTransform (transform.cpp:234-273).
__global__ void k_inverse_transform(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= f.N || !wz_block(f, b)) return;  // the SIR lists WZ blocks only
  const int bw = f.W / 4, top = (b / bw) * 4, left = (b % bw) * 4, W = f.W;
  int blk[16];
  for (int m = 0; m < 4; m++)
    for (int n = 0; n < 4; n++) blk[4 * m + n] = f.sideTrans[(top + m) * W + left + n];
  inverse44(blk);
  for (int m = 0; m < 4; m++)
    for (int n = 0; n < 4; n++) {
      const int c = blk[4 * m + n];
      f.recons[(top + m) * W + left + n] = (uint8_t)(c < 0 ? 0 : (c > 255 ? 255 : c));
    }
}

// ------------------------------------------------------------ SI refresh
// updateSI + subPelRefine (sideInfoCreation.cpp:598-736): per WZ 4x4 block of
// the partially reconstructed frame, separate full-pel argmins on the past
// and future key frames (cost SAD*(1+K*|2v|) in double), 9-position half-pel
// refinement on each interpolated frame, then SI = (int)(P*iPC + F*iFC).
// One wave per block, 4 horizontally adjacent blocks per workgroup (the frame
// width is a multiple of 16, so the 4 share a block row).  The union of their
// search windows (up to 68 rows x 80 bytes of each key frame) is staged in LDS
// as 32-bit words, each wave staging every fourth row of both frames, the two
// frames' rows interleaved so that one address reaches both; lane l
// sweeps candidate column sL+l down the window, forming each candidate's
// 4-pixel rows with v_alignbyte and its SAD with v_sad_u8 (exact integer SADs,
// as the reference's double sums of integer differences are).  A lane keeps
// its best cost only; the rows above the block and the rows from the block down
// run as two loops, so the cost factor's LDS address steps by a constant.  The
// 65th column of a full window is spread over the lanes.  The VALU issue port
// bounds the loop, so the candidate itself is found afterwards: the wave's
// least cost, then the columns that hold it (nearly always one), then, a lane
// per row, the first row of such a column with that cost.  Ties resolve to the
// first candidate in raster order: the least (row, column) key.
// A cost (double)sad * fac is the product of two doubles: the one whose bits
// are the integer sad, which is the subnormal sad * 2^-1074, and fac * 2^1000
// from the table.  The product is sad * fac * 2^-74, far inside the normal
// range, so it has the rounded product's mantissa without a conversion, and all
// costs carry the same scale.
// Tracking the row of each lane's best and forming a cost as fma(2^52 + sad,
// fac, -2^52 * fac), the loop took 19.5 VALU instructions per candidate row of
// both frames, 8 of them SADs; now 14.5 (2421 and 2079 us for 128 CIF frames).
#define USI_LW 21   // staged words per window row: 20 + one zero word
#define USI_ROWS 68
__device__ __forceinline__ uint32_t usi_word(const uint32_t *R, int r, int j, int sh) {
  return __builtin_amdgcn_alignbyte(R[r * 2 * USI_LW + j + 1], R[r * 2 * USI_LW + j], sh);
}
__device__ __forceinline__ uint32_t sad4(const uint32_t *bk, uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3) {
  uint32_t s = __builtin_amdgcn_sad_u8(bk[0], r0, 0u);
  s = __builtin_amdgcn_sad_u8(bk[1], r1, s);
  s = __builtin_amdgcn_sad_u8(bk[2], r2, s);
  return __builtin_amdgcn_sad_u8(bk[3], r3, s);
}
// v_min_f64 of two values known to be numbers (the compiler would otherwise
// canonicalise a loop-carried operand first)
__device__ __forceinline__ double dmin_num(double a, double b) {
  double r;
  __asm__("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double wave_min(double m) {  // numbers only
  for (int o = 32; o > 0; o >>= 1) m = dmin_num(m, __shfl_xor(m, o));
  return m;
}
__global__ __launch_bounds__(256) void k_update_si(const FrameDev *F, const int *list, CostTables ct) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b0 = blockIdx.x * 4;
  if (b0 >= f.N) return;  // uniform over the workgroup
  const int W = f.W, H = f.H, W2 = 2 * W, H2 = 2 * H, bw = W / 4;
  __shared__ uint32_t s_win[USI_ROWS * 2 * USI_LW];  // [row][past, future][word]
  __shared__ double s_fac[33 * 33];  // by (|dy|, |dx|), times 2^1000
  // union window of the 4 blocks: rows [wT, wB], byte columns [cL, cR]
  const int row0 = (b0 / bw) * 4, left0 = (b0 % bw) * 4;
  const int wT = imax(0, row0 - 32), wB = imin(H - 4, row0 + 32) + 3;
  const int cL = imax(0, left0 - 32) & ~3, cR = imin(W - 4, left0 + 12 + 32) + 3;
  const int nrows = wB - wT + 1, nw = (cR + 1 - cL) >> 2;  // nrows <= 68, nw <= 20
  {
    // lanes 0..20 stage a past-frame row's words, lanes 32..52 the future's
    const int half = lane >> 5, w = lane & 31;
    if (w < USI_LW) {
      const uint8_t *src = half ? f.fut : f.past;
      uint32_t *dst = s_win + half * USI_LW;
      for (int r = wave; r < nrows; r += 4)
        dst[r * 2 * USI_LW + w] = w < nw ? *(const uint32_t *)(src + (size_t)(wT + r) * W + cL + 4 * w) : 0u;
    }
    for (int dy = wave; dy < 33; dy += 4)
      if (lane < 33) s_fac[dy * 33 + lane] = ct.usi[(dy + 32) * 65 + lane + 32] * 0x1p1000;
  }
  __syncthreads();
  const int b = b0 + wave;
  if (b >= f.N || !wz_block(f, b)) return;  // updateSI walks the SIR's WZ blocks
  const int top = row0, left = (b % bw) * 4;
  const int sT = imax(0, top - 32), sB = imin(H - 4, top + 32), sL = imax(0, left - 32), sR = imin(W - 4, left + 32);
  const int ww = sR - sL + 1, nr = sB - sT + 1;
  uint32_t bk[4];
#pragma unroll
  for (int m = 0; m < 4; m++) bk[m] = *(const uint32_t *)(f.recons + (size_t)(top + m) * W + left);
  const uint32_t *P = s_win, *Fu = s_win + USI_LW;
  double pBest = DBL_MAX, fBest = DBL_MAX;
  if (lane < ww) {
    const int x = sL + lane, xo = x - cL, j = xo >> 2, sh = xo & 3;
    const double *facCol = s_fac + abs(x - left);
    int r = sT - wT;
    uint32_t p0 = usi_word(P, r, j, sh), p1 = usi_word(P, r + 1, j, sh), p2 = usi_word(P, r + 2, j, sh);
    uint32_t f0 = usi_word(Fu, r, j, sh), f1 = usi_word(Fu, r + 1, j, sh), f2 = usi_word(Fu, r + 2, j, sh);
    // the zero high words of the SADs' doubles, one register per frame so that
    // each SAD can land in the low half of its own pair
    int hiP = 0, hiF = 0;
    __asm__ volatile("" : "+v"(hiP));
    __asm__ volatile("" : "+v"(hiF));
    auto step = [&](double fac) {
      const uint32_t p3 = usi_word(P, r + 3, j, sh), f3 = usi_word(Fu, r + 3, j, sh);
      const uint32_t ps = sad4(bk, p0, p1, p2, p3), fs = sad4(bk, f0, f1, f2, f3);
      pBest = dmin_num(pBest, __hiloint2double(hiP, (int)ps) * fac);
      fBest = dmin_num(fBest, __hiloint2double(hiF, (int)fs) * fac);
      p0 = p1; p1 = p2; p2 = p3;
      f0 = f1; f1 = f2; f2 = f3;
      r++;
    };
    int y = sT;
    // rows above the block: |y - top| falls, so four rows at a time read the
    // table upwards from the lowest of their entries (LDS offsets are positive)
    const double *lo = facCol + 33 * (top - sT - 3);
    for (; y + 4 <= top; y += 4, lo -= 4 * 33) {
      step(lo[99]);
      step(lo[66]);
      step(lo[33]);
      step(lo[0]);
    }
    for (; y < top; y++) step(facCol[33 * (top - y)]);
    const double *fp = facCol;  // rows from the block down: |y - top| rises
    for (; y + 4 <= sB + 1; y += 4, fp += 4 * 33) {
      step(fp[0]);
      step(fp[33]);
      step(fp[66]);
      step(fp[99]);
    }
    for (; y <= sB; y++, fp += 33) step(*fp);
  }
  // the cost of candidate (row, column) relative to (sT, sL) on frame R
  auto cost_at = [&](const uint32_t *R, int row, int col) {
    const int x = sL + col, xo = x - cL, j = xo >> 2, sh = xo & 3, r = sT + row - wT;
    const uint32_t sad = sad4(bk, usi_word(R, r, j, sh), usi_word(R, r + 1, j, sh), usi_word(R, r + 2, j, sh),
                              usi_word(R, r + 3, j, sh));
    return __hiloint2double(0, (int)sad) * s_fac[33 * abs(sT + row - top) + abs(x - left)];
  };
  // column sL+64 of a full window: row `lane`, and row 64 on lane 0
  double pCol[2] = {DBL_MAX, DBL_MAX}, fCol[2] = {DBL_MAX, DBL_MAX};
  if (ww > 64) {
#pragma unroll
    for (int h = 0; h < 2; h++)
      if (lane + 64 * h < nr) {
        pCol[h] = cost_at(P, lane + 64 * h, 64);
        fCol[h] = cost_at(Fu, lane + 64 * h, 64);
      }
  }
  // first candidate in raster order of the wave's least cost: (row << 7) + column
  auto locate = [&](const uint32_t *R, double best, const double *col64) -> int {
    const double m = wave_min(dmin_num(best, dmin_num(col64[0], col64[1])));
    int key = 0x7fffffff;
    const uint64_t e0 = __ballot(col64[0] == m), e1 = __ballot(col64[1] == m);
    if (e0 | e1) key = ((e0 ? __builtin_ctzll(e0) : 64) << 7) + 64;
    uint64_t cols = __ballot(best == m);
    if (__popcll(cols) <= 4) {
      // a lane per row of each column; row 64 only when no earlier row matches
      for (; cols; cols &= cols - 1) {
        const int col = __builtin_ctzll(cols);
        const uint64_t rows = __ballot(lane < nr && cost_at(R, imin(lane, nr - 1), col) == m);
        key = imin(key, ((rows ? __builtin_ctzll(rows) : 64) << 7) + col);
      }
    } else {
      // many columns (flat contents): each looks down its own rows, and the
      // first row that any of them matches holds the least key
      const bool mine = best == m;
      for (int row = 0; row < nr && (row << 7) < key; row++) {
        const uint64_t hit = __ballot(mine && cost_at(R, row, imin(lane, ww - 1)) == m);
        if (hit) {
          key = imin(key, (row << 7) + __builtin_ctzll(hit));
          break;
        }
      }
    }
    return key;
  };
  const int pKey = locate(P, pBest, pCol), fKey = locate(Fu, fBest, fCol);
  const int pbx = sL + (pKey & 127), pby = sT + (pKey >> 7), fbx = sL + (fKey & 127), fby = sT + (fKey >> 7);
  // subPelRefine: lanes 0-8 evaluate the 9 positions of the past frame, 16-24 the future
  const int which = lane >> 4, pos = lane & 15;
  double cost = DBL_MAX;
  int cidx = 0x7fffffff;
  if (which < 2 && pos < 9) {
    const int bx = which ? fbx : pbx, by = which ? fby : pby;
    const uint8_t *ref = which ? f.fut_half : f.past_half;
    const int t = 2 * by + pos / 3 - 1, l = 2 * bx + pos % 3 - 1;
    if (t >= 0 && t <= H2 - 8 && l >= 0 && l <= W2 - 8) {
      // the 4 samples of block row m sit 2 bytes apart in the half-pel frame
      uint32_t s = 0;
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const uint8_t *rp = ref + (size_t)(t + 2 * m) * W2 + l;
        const uint32_t row = (uint32_t)rp[0] | (uint32_t)rp[2] << 8 | (uint32_t)rp[4] << 16 | (uint32_t)rp[6] << 24;
        s = __builtin_amdgcn_sad_u8(bk[m], row, s);
      }
      cost = (double)s;
      cidx = pos;
    }
  }
  // argmin within each 16-lane group (first minimum in (i, j) order)
  for (int o = 8; o > 0; o >>= 1) {
    const double c2 = __shfl_xor(cost, o);
    const int i2 = __shfl_xor(cidx, o);
    if (c2 < cost || (c2 == cost && i2 < cidx)) { cost = c2; cidx = i2; }
  }
  const int pSub = __shfl(cidx, 0), fSub = __shfl(cidx, 16);
  const int phx = 2 * pbx + pSub % 3 - 1, phy = 2 * pby + pSub / 3 - 1;
  const int fhx = 2 * fbx + fSub % 3 - 1, fhy = 2 * fby + fSub / 3 - 1;
  if (lane < 16) {
    const int m = lane >> 2, n = lane & 3;
    const int pv = f.past_half[(phy + 2 * m) * W2 + phx + 2 * n];
    const int fv = f.fut_half[(fhy + 2 * m) * W2 + fhx + 2 * n];
    f.si[(top + m) * W + left + n] = (uint8_t)(int)((double)pv * f.iPC + (double)fv * f.iFC);
  }
}

// ------------------------------------------------------------ motion learning
// updateSMF (motionLearning.cpp:70-127): p = expf(-MU*SSE) over the +-4
// window, normalised by the float sum in raster order.  One wave per 4x4
// block.  Every pixel difference is an integer of magnitude at most 255 and
// every partial SSE stays below 2^24, so the reference's float SSE is exact in
// any order and equals the integer sum of squares; it is formed here as
// sum(a^2) + sum(b^2) - 2 sum(a*b) with v_dot4_u32_u8 on 4-pixel rows (a the
// reconstructed block, b the side information under the window position),
// reading b from the block's side-information window (at most 12 rows x 12
// bytes) staged in LDS as words.  Lane l evaluates window positions l and
// l+64; the wave then adds the probabilities in raster order from LDS.
#define SMF_WORDS 5  // staged words per window row: 4 + one for the byte alignment
__global__ __launch_bounds__(256) void k_update_smf(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = blockIdx.x * 4 + wave;
  __shared__ uint32_t s_si[4][12 * SMF_WORDS];
  __shared__ __align__(16) float s_v[4][84];  // rows of 336 bytes: float4 reads stay aligned
  // updateSMF walks the SIR's WZ blocks; the barrier below is reached by all
  const bool on = b < f.N && wz_block(f, b);
  const int W = f.W;
  const SmfWin s = smf_window(f, on ? b : 0);
  const int cL = s.sL & ~3;
  if (on && lane < 12 * SMF_WORDS) {
    const int r = lane / SMF_WORDS, w = lane - r * SMF_WORDS, x = cL + 4 * w;
    s_si[wave][lane] = s.sT + r <= s.sB + 3 && x + 3 < W ? *(const uint32_t *)(f.si + (size_t)(s.sT + r) * W + x) : 0u;
  }
  uint32_t aw[4];
  uint32_t a2 = 0;
#pragma unroll
  for (int m = 0; m < 4; m++) {
    aw[m] = on ? *(const uint32_t *)(f.recons + (size_t)(s.top + m) * W + s.left) : 0u;
    a2 = __builtin_amdgcn_udot4(aw[m], aw[m], a2, false);
  }
  __syncthreads();
  float v[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int p = lane + 64 * h;
    v[h] = 0.0f;
    if (on && p < s.len) {
      const int pr = p / s.w, xo = s.sL + (p - pr * s.w) - cL, j = xo >> 2, sh = xo & 3;
      const uint32_t *R = s_si[wave] + pr * SMF_WORDS + j;
      uint32_t bb = 0, ab = 0;
#pragma unroll
      for (int ii = 0; ii < 4; ii++) {
        const uint32_t bw = __builtin_amdgcn_alignbyte(R[ii * SMF_WORDS + 1], R[ii * SMF_WORDS], sh);
        bb = __builtin_amdgcn_udot4(bw, bw, bb, false);
        ab = __builtin_amdgcn_udot4(aw[ii], bw, ab, false);
      }
      const float sse = (float)(a2 + bb - 2u * ab);
      v[h] = dvc_expf(-0.01f * sse);
      s_v[wave][p] = v[h];
    }
  }
  __syncthreads();
  if (!on) return;
  // the sum in raster order, the same on every lane (LDS broadcast reads)
  const int len = s.len;
  const float *V = s_v[wave];
  float sum = 0.0f;
  int p = 0;
  for (; p + 4 <= len; p += 4) {
    const float4 q = *(const float4 *)(V + p);
    sum += q.x;
    sum += q.y;
    sum += q.z;
    sum += q.w;
  }
  for (; p < len; p++) sum += V[p];
  float *pr = f.smf + (size_t)81 * b;
  const bool norm = (double)sum > 0.0;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int q = lane + 64 * h;
    if (q < s.len) pr[q] = norm ? v[h] / sum : (q == s.self ? 1.0f : v[h]);
  }
}

// update_si_ML (motionLearning.cpp:129-160): SMF-weighted over-complete
// coefficients for the bands after the frame's current band, accumulated in
// window raster order and truncated.  A wave owns ML_ROWS block rows of 16
// adjacent block columns; lane 4c + g owns row g (coefficients 4g..4g+3) of
// block column c and reads it from each window position's 64-byte record with
// one 16-byte load.  The wave streams down the over-complete rows its blocks'
// windows cover, reading each row once: the windows of block rows R-1, R and
// R+1 share position row 4R, so while position rows 4j..4j+3 stream by, block
// row j-1 takes its last row (at 4j), block row j its rows 5-8 and block row
// j+1 its rows 1-4, each in its own accumulators.  Every coefficient's sum
// still runs over its block's window in raster order; coefficients of bands
// already decoded are summed too but not stored.  A window row's weights are
// loaded three per lane by the four lanes of a block column and passed
// between them with quad permutes.
#define ML_COLS 16  // block columns per wave
template <int L>
__device__ __forceinline__ float quad_bcast(float v) {
  // quad_perm [L, L, L, L]: every lane of a quad takes the quad's lane L
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), L * 0x55, 0xf, 0xf, false));
}
__device__ __forceinline__ float quad_bcast(float v, int l) {  // l is a constant after unrolling
  switch (l) {
    case 0: return quad_bcast<0>(v);
    case 1: return quad_bcast<1>(v);
    case 2: return quad_bcast<2>(v);
    default: return quad_bcast<3>(v);
  }
}
template <int ML_ROWS>
__global__ __launch_bounds__(256) void k_update_si_ml(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  const int bandStart = f.band + 1;  // update_si_ML(..., band+1, ...) (DVC_Decoder.cpp:369)
  if (bandStart >= 16) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int W = f.W, H = f.H, bw = W / 4, bh = H / 4, ow = W - 3;
  const int colTiles = (bw + ML_COLS - 1) / ML_COLS, rowTiles = (bh + ML_ROWS - 1) / ML_ROWS;
  const int tile = blockIdx.x * 4 + wave;
  if (tile >= colTiles * rowTiles) return;  // uniform over the wave
  const int ty = tile / colTiles, tx = tile - ty * colTiles;
  const int c = lane >> 2, g = lane & 3, bc = tx * ML_COLS + c;
  const bool live = bc < bw;
  int need = 0;  // coefficients 4g + jj still to predict
  for (int k = bandStart; k < 16; k++)
    if ((c_zigzag[k] >> 2) == g) need |= 1 << (c_zigzag[k] & 3);
  const int left = 4 * (live ? bc : 0), sL = imax(0, left - 4), w = imin(W - 4, left + 4) - sL + 1;
  const int R0 = ty * ML_ROWS, R1 = imin(bh, R0 + ML_ROWS);
  const int mS = imax(0, 4 * R0 - 4), mE = imin(H - 4, 4 * (R1 - 1) + 4);
  // one position row m for block row R (R0 <= R < R1): acc[jj] += p_q * o_q[jj]
  // over the row.  Positions past a narrow window's edge (q >= w) have p and o
  // zero: adding their +0 products leaves every sum's value unchanged (the
  // reference never adds them; a zero's sign cannot survive the truncation).
  auto rowTerms = [&](float *acc, int R, int m, const float (*o)[4]) {
    const float *pr = f.smf + (size_t)81 * (live ? R * bw + bc : 0) + (m - imax(0, 4 * R - 4)) * w;
    // lane g holds the weights q = g, g + 4, g + 8 of its block column's row
    float wv[3];
#pragma unroll
    for (int i = 0; i < 3; i++) wv[i] = live && g + 4 * i < w ? pr[g + 4 * i] : 0.0f;
#pragma unroll
    for (int q = 0; q < 9; q++) {
      const float p = quad_bcast(wv[q >> 2], q & 3);
#pragma unroll
      for (int jj = 0; jj < 4; jj++) acc[jj] += p * o[q][jj];
    }
  };
  auto finish = [&](const float *acc, int R) {
    const int b = R * bw + bc;
    if (live && wz_block(f, b)) {
      int *dst = f.sideTrans + (4 * R + g) * W + left;
#pragma unroll
      for (int jj = 0; jj < 4; jj++)
        if (need >> jj & 1) dst[jj] = (int)acc[jj];
    }
  };
  float accP[4] = {}, accQ[4] = {};  // block rows j-1 and j, carried into chunk j
  for (int j = mS >> 2; 4 * j <= mE; j++) {
    float accN[4] = {};  // block row j+1, whose window starts at position row 4j
    for (int t = 0; t < 4; t++) {
      const int m = 4 * j + t;
      if (m < mS || m > mE) continue;  // uniform
      float o[9][4];
      const int4 *op = (const int4 *)(f.oct + (size_t)16 * ((size_t)m * ow + sL)) + g;
#pragma unroll
      for (int q = 0; q < 9; q++) {
        const int4 v = live && q < w ? op[4 * q] : make_int4(0, 0, 0, 0);
        o[q][0] = (float)v.x; o[q][1] = (float)v.y; o[q][2] = (float)v.z; o[q][3] = (float)v.w;
      }
      if (t == 0 && j - 1 >= R0) {  // the last row of block row j-1
        rowTerms(accP, j - 1, m, o);
        finish(accP, j - 1);
      }
      if (j >= R0 && j < R1) {
        rowTerms(accQ, j, m, o);
        if (m == H - 4) finish(accQ, j);  // the bottom block row's window ends at H-4
      }
      if (j + 1 < R1) rowTerms(accN, j + 1, m, o);
    }
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
      accP[jj] = accQ[jj];
      accQ[jj] = accN[jj];
    }
  }
}

// ------------------------------------------------------------ launchers
hipError_t launch_keyframe_filters(const uint8_t *in, uint8_t *lp, uint8_t *half, int W, int H, hipStream_t s) {
  hipLaunchKernelGGL(k_keyframe_filters, dim3((2 * W + 127) / 128, H), dim3(128), 0, s, in, lp, half, W, H);
  return hipGetLastError();
}
hipError_t launch_keyframe_batch(const KeyFrameJob *jobs, int n, int maxW, int maxH, hipStream_t s) {
  constexpr int kMost = 32768;  // a side-information batch has two per pair, whose grids take 65535
  for (int k = 0; k < n; k += kMost) {
    hipLaunchKernelGGL(k_keyframe_batch, dim3((2 * maxW + 127) / 128, maxH, n - k < kMost ? n - k : kMost), dim3(128), 0, s,
                       jobs + k);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}
hipError_t launch_create_si(const FrameDev *F, const int *list, int n, int maxMB, CostTables ct, hipStream_t s) {
  // 4x4 tiles of 8x8 blocks: a CIF frame's 11 x 9, more than a QCIF frame's 6 x 5
  const int tiles = 99;
  hipLaunchKernelGGL(k_forward_me, dim3(maxMB, n), dim3(256), 0, s, F, list, ct);
  hipLaunchKernelGGL(k_si_sweep, dim3(n), dim3(1024), 0, s, F, list, 0);
  hipLaunchKernelGGL(k_si_finish, dim3(tiles, n), dim3(256), 0, s, F, list);
  return hipGetLastError();
}
hipError_t launch_forward_me(const FrameDev *F, const int *list, int n, int maxMB, CostTables ct, hipStream_t s) {
  hipLaunchKernelGGL(k_forward_me, dim3(maxMB, n), dim3(256), 0, s, F, list, ct);
  hipLaunchKernelGGL(k_si_sweep, dim3(n), dim3(1024), 0, s, F, list, 1);
  return hipGetLastError();
}
hipError_t launch_noise_param(const FrameDev *F, const int *list, int n, int maxN, hipStream_t s) {
  hipLaunchKernelGGL(k_residue_transform, dim3((maxN + 255) / 256, n), dim3(256), 0, s, F, list);
  hipLaunchKernelGGL(k_noise_moments, dim3(16, n), dim3(256), 0, s, F, list);
  hipLaunchKernelGGL(k_noise_alpha, dim3((maxN + 255) / 256, n), dim3(256), 0, s, F, list);
  return hipGetLastError();
}
hipError_t launch_oct(const FrameDev *F, const int *list, int n, int maxPos, int initSideTrans, hipStream_t s) {
  hipLaunchKernelGGL(k_oct, dim3((maxPos + 255) / 256, n), dim3(256), 0, s, F, list, initSideTrans);
  return hipGetLastError();
}
// copySkipBlkToRecons (skipBlock.cpp:3-22): one thread per 8x8 block.
__global__ void k_skip_copy(const FrameDev *F, const int *list) {
  const FrameDev &f = F[list[blockIdx.y]];
  if (!f.mode) return;
  const int w8 = f.W >> 3, n8 = w8 * (f.H >> 3);
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n8 || f.mode[k] != kSkipBlock) return;
  const int top = (k / w8) * 8, left = (k % w8) * 8;
  for (int m = 0; m < 8; m++) {
    const size_t o = (size_t)(top + m) * f.W + left;
    for (int n = 0; n < 8; n++) f.recons[o + n] = f.past[o + n];  // caller buffers need not be aligned
  }
}
hipError_t launch_skip_copy(const FrameDev *F, const int *list, int n, int maxBlk88, hipStream_t s) {
  hipLaunchKernelGGL(k_skip_copy, dim3((maxBlk88 + 255) / 256, n), dim3(256), 0, s, F, list);
  return hipGetLastError();
}
hipError_t launch_noise_dist(const FrameDev *F, const int *list, int n, int maxN, int fill, hipStream_t s) {
  hipLaunchKernelGGL(k_noise_dist, dim3(maxN, n), dim3(ND_T), 0, s, F, list, fill);
  return hipGetLastError();
}
hipError_t launch_condbit(const FrameDev *F, const int *list, int n, int maxN, hipStream_t s) {
  hipLaunchKernelGGL(k_condbit, dim3((maxN + 31) / 32, n), dim3(64), 0, s, F, list);
  return hipGetLastError();
}
hipError_t launch_put_bitplane(const FrameDev *F, const int *list, const BpFrameLink *links, int n, int maxN,
                               hipStream_t s) {
  hipLaunchKernelGGL(k_put_bitplane, dim3((maxN + 255) / 256, n), dim3(256), 0, s, F, list, links);
  return hipGetLastError();
}
hipError_t launch_reconstruct(const FrameDev *F, const int *list, int n, int maxN, hipStream_t s) {
  hipLaunchKernelGGL(k_reconstruct, dim3((maxN + 255) / 256, n), dim3(256), 0, s, F, list);
  return hipGetLastError();
}
hipError_t launch_inverse_transform(const FrameDev *F, const int *list, int n, int maxN, hipStream_t s) {
  hipLaunchKernelGGL(k_inverse_transform, dim3((maxN + 255) / 256, n), dim3(256), 0, s, F, list);
  return hipGetLastError();
}
hipError_t launch_update_si(const FrameDev *F, const int *list, int n, int maxN, CostTables ct, hipStream_t s) {
  hipLaunchKernelGGL(k_update_si, dim3((maxN + 3) / 4, n), dim3(256), 0, s, F, list, ct);
  return hipGetLastError();
}
hipError_t launch_smf_init(const FrameDev *F, const int *list, int n, int maxN, hipStream_t s) {
  hipLaunchKernelGGL(k_smf_init, dim3((maxN + 255) / 256, n), dim3(256), 0, s, F, list);
  return hipGetLastError();
}
hipError_t launch_update_smf(const FrameDev *F, const int *list, int n, int maxN, hipStream_t s) {
  hipLaunchKernelGGL(k_update_smf, dim3((maxN + 3) / 4, n), dim3(256), 0, s, F, list);
  return hipGetLastError();
}
template <int ML_ROWS>
static void launch_ml(const FrameDev *F, const int *list, int n, int colTiles, int maxBh, hipStream_t s) {
  const int tiles = colTiles * ((maxBh + ML_ROWS - 1) / ML_ROWS);
  hipLaunchKernelGGL((k_update_si_ml<ML_ROWS>), dim3((tiles + 3) / 4, n), dim3(256), 0, s, F, list);
}
hipError_t launch_update_si_ml(const FrameDev *F, const int *list, int n, int maxBw, int maxBh, hipStream_t s) {
  // Block rows per wave: eight read the least (4.6 position rows per block row,
  // against 5.3 for four and 9 for one), but a wave walks its 37 rows one after
  // another, so while eight-row waves do not fill the chip's 1024 SIMDs shorter
  // walks win.  us for 1, 8, 24, 64 and 128 CIF frames (54 eight-row waves each):
  // one row 24, 35, 111, 307, 596; four 59, 62, 95, 257, 490; eight 105, 108,
  // 143, 238, 463.
  const int colTiles = (maxBw + ML_COLS - 1) / ML_COLS, waves8 = n * colTiles * ((maxBh + 7) / 8);
  if (waves8 <= 1024) launch_ml<1>(F, list, n, colTiles, maxBh, s);
  else if (waves8 <= 2560) launch_ml<4>(F, list, n, colTiles, maxBh, s);
  else launch_ml<8>(F, list, n, colTiles, maxBh, s);
  return hipGetLastError();
}

}  // namespace dvc
