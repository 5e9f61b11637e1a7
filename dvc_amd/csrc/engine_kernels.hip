// engine_kernels.hip -- batched frame set-up and result gathering for the
// serving engine (declarations and layouts in engine_kernels.h).
#include "engine_kernels.h"

namespace dvc {

// blockIdx.y = frame; the x blocks stride over each of its buffers.
__global__ __launch_bounds__(256) void k_job_init(const JobInitDev *items) {
  const JobInitDev it = items[blockIdx.y];
  const int t = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  for (int i = t; i < it.fs; i += stride) it.reconsTrans[i] = 0;
  for (int i = t; i < it.N; i += stride) it.carry[i] = 0xAA;
  for (int i = t; i < it.nbp; i += stride) it.state[i] = PlaneState{-1, it.numCodes - 1, 0.0f, 0, 0};
  for (int i = t; i < kMaxCodes * it.nbp; i += stride) it.rec[i] = make_int4(0, REC_NOT_RUN, -1, 0);
  if (it.accSrc)
    for (int i = t; i < it.accBytes; i += stride) it.accDst[i] = it.accSrc[i];
}

// blockIdx.y = segment.
__global__ __launch_bounds__(256) void k_copy_segments(const CopySeg *segs) {
  const CopySeg sg = segs[blockIdx.y];
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = t; i < sg.bytes; i += stride) sg.dst[i] = sg.src[i];
}

// Copies the ring's next block.  turn[0] counts the blocks taken, turn[1] this
// launch's workgroups that have read it; the last of them moves on.
__global__ __launch_bounds__(256) void k_take_block(const uint4 *ring, int blocks, int quads, uint4 *dst, unsigned *turn) {
  __shared__ unsigned s_turn;
  if (threadIdx.x == 0) {
    s_turn = __hip_atomic_load(&turn[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // (acq_rel: the read of turn[0] comes before the count)
    if (__hip_atomic_fetch_add(&turn[1], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
      __hip_atomic_store(&turn[1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&turn[0], s_turn + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  __syncthreads();
  const uint4 *src = ring + (size_t)(s_turn % (unsigned)blocks) * quads;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < quads; i += gridDim.x * 256) dst[i] = src[i];
}

hipError_t launch_take_block(const void *ring, int blocks, size_t bytes, void *dst, unsigned *turn, hipStream_t s) {
  const int quads = (int)(bytes / 16);
  if (bytes % 16 || quads < 1 || blocks < 1) return hipErrorInvalidValue;
  const int grid = quads < 64 * 256 ? (quads + 255) / 256 : 64;
  hipLaunchKernelGGL(k_take_block, dim3(grid), dim3(256), 0, s, (const uint4 *)ring, blocks, quads, (uint4 *)dst, turn);
  return hipGetLastError();
}

hipError_t launch_job_init(const JobInitDev *items, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_job_init, dim3(32, n), dim3(256), 0, s, items);
  return hipGetLastError();
}

hipError_t launch_copy_segments(const CopySeg *segs, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_copy_segments, dim3(64, n), dim3(256), 0, s, segs);
  return hipGetLastError();
}

}  // namespace dvc
