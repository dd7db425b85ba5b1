// gpe_misc.hip -- reductions and pointwise kernels, and the dispatch over
// the stage-kernel variants.  Built with -ffp-contract=off.
#include "batch_ctl.hpp"
#include "launch.h"
#include "pointwise.hpp"

namespace gpe {

hipError_t launch_stage(int prec_bytes, int vid, int kind, int radius, bool comp, const StageArgs &A,
                        hipStream_t s, int *resident) {
  if (prec_bytes == 16) {
    switch (vid) {
      case 0: return launch_stage_f64_v0(kind, radius, comp, A, s, resident);
      case 1: return launch_stage_f64_v1(kind, radius, comp, A, s, resident);
      case 2: return launch_stage_f64_v2(kind, radius, comp, A, s, resident);
      case 3: return launch_stage_f64_v3(kind, radius, comp, A, s, resident);
      case 4: return launch_stage_f64_v4(kind, radius, comp, A, s, resident);
    }
  } else {
    switch (vid) {
      case 0: return launch_stage_f32_v0(kind, radius, comp, A, s, resident);
      case 1: return launch_stage_f32_v1(kind, radius, comp, A, s, resident);
      case 2: return launch_stage_f32_v2(kind, radius, comp, A, s, resident);
      case 3: return launch_stage_f32_v3(kind, radius, comp, A, s, resident);
      case 4: return launch_stage_f32_v4(kind, radius, comp, A, s, resident);
    }
  }
  return hipErrorInvalidValue;
}

hipError_t launch_stage_batched(int prec_bytes, int vid, int kind, int radius, bool comp, const BatchLaunch &B,
                                hipStream_t s) {
  if (prec_bytes == 16) {
    switch (vid) {
      case 0: return launch_batched_f64_v0(kind, radius, comp, B, s);
      case 1: return launch_batched_f64_v1(kind, radius, comp, B, s);
      case 2: return launch_batched_f64_v2(kind, radius, comp, B, s);
      case 3: return launch_batched_f64_v3(kind, radius, comp, B, s);
      case 4: return launch_batched_f64_v4(kind, radius, comp, B, s);
    }
  } else {
    switch (vid) {
      case 0: return launch_batched_f32_v0(kind, radius, comp, B, s);
      case 1: return launch_batched_f32_v1(kind, radius, comp, B, s);
      case 2: return launch_batched_f32_v2(kind, radius, comp, B, s);
      case 3: return launch_batched_f32_v3(kind, radius, comp, B, s);
      case 4: return launch_batched_f32_v4(kind, radius, comp, B, s);
    }
  }
  return hipErrorInvalidValue;
}

hipError_t launch_pair(int prec_bytes, int vid, int pair, int radius, bool comp, const StageArgs &A,
                       const StageArgs &B, hipStream_t s) {
  if (prec_bytes != 16) {
    switch (vid) {
      case 0: return launch_pair_f32_v0(pair, radius, comp, A, B, s);
      case 1: return launch_pair_f32_v1(pair, radius, comp, A, B, s);
      case 2: return launch_pair_f32_v2(pair, radius, comp, A, B, s);
    }
  }
  return hipErrorInvalidValue;
}

hipError_t launch_pair_batched(int prec_bytes, int vid, int pair, int radius, bool comp, const PairBatchLaunch &L,
                               hipStream_t s) {
  if (prec_bytes != 16) {
    switch (vid) {
      case 0: return launch_pair_batched_f32_v0(pair, radius, comp, L, s);
      case 1: return launch_pair_batched_f32_v1(pair, radius, comp, L, s);
      case 2: return launch_pair_batched_f32_v2(pair, radius, comp, L, s);
    }
  }
  return hipErrorInvalidValue;
}

hipError_t launch_batch_control(InstCtl *ctl, StageArgs *args, int cap, int *active, const int *range,
                                const double *pn, const double *pe, hipStream_t s) {
  if (cap <= 0) return hipSuccess;
  hipLaunchKernelGGL(batch_control, dim3(cap), dim3(64), 0, s, ctl, args, cap, active, range, pn, pe);
  return hipGetLastError();
}

namespace {

// Sum / max of a sweep's partials in a fixed order by one workgroup; thread 0
// gets the results.
constexpr int kReduceThreads = 256;
__device__ __forceinline__ void reduce_all(const double *pn, const double *pe, const double *pen, int n, double &sum,
                                           double &top, double &energy) {
  __shared__ double s0[kReduceThreads], s1[kReduceThreads], s2[kReduceThreads];
  double a = 0.0, m = 0.0, c = 0.0;
  for (int i = threadIdx.x; i < n; i += kReduceThreads) {
    if (pn) a += pn[i];
    if (pe) m = (pe[i] > m || pe[i] != pe[i]) ? pe[i] : m;
    if (pen) c += pen[i];
  }
  s0[threadIdx.x] = a;
  s1[threadIdx.x] = m;
  s2[threadIdx.x] = c;
  __syncthreads();
  for (int w = kReduceThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      s0[threadIdx.x] += s0[threadIdx.x + w];
      const double o = s1[threadIdx.x + w];
      s1[threadIdx.x] = (o > s1[threadIdx.x] || o != o) ? o : s1[threadIdx.x];
      s2[threadIdx.x] += s2[threadIdx.x + w];
    }
    __syncthreads();
  }
  sum = s0[0];
  top = s1[0];
  energy = s2[0];
}

// out[0] = sum(pn) * scale_norm, out[1] = max(pe) / eps (maxval(...)/eps,
// solve.f90:184), out[2] = sum(pen) * scale_energy; hist (if set) gets out[0].
// out may be host memory: with ticket != 0 the host reads out[0..2] once
// out[3] holds the ticket, without a copy or a wait for the stream.
__global__ void __launch_bounds__(kReduceThreads)
    reduce_partials(const double *pn, const double *pe, const double *pen, int n, double scale_norm, double eps,
                    double scale_energy, double *out, double *hist, double ticket) {
  double a, m, c;
  reduce_all(pn, pe, pen, n, a, m, c);
  if (threadIdx.x == 0) {
    out[0] = a * scale_norm;
    out[1] = m / eps;
    out[2] = c * scale_energy;
    if (hist) *hist = a * scale_norm;
    if (ticket != 0.0) {
      __threadfence_system();
      __hip_atomic_store(out + 3, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// The norms of several steps, one workgroup each: step b's partials start at
// pn + b*stride.
__global__ void __launch_bounds__(kReduceThreads)
    reduce_norms(const double *pn, size_t stride, int n, double scale_norm, double *hist) {
  double a, m, c;
  reduce_all(pn + blockIdx.x * stride, nullptr, nullptr, n, a, m, c);
  if (threadIdx.x == 0) hist[blockIdx.x] = a * scale_norm;
}

}  // namespace

hipError_t launch_reduce(const double *pn, const double *pe, const double *pen, int n, double scale_norm,
                         double eps, double scale_energy, double *out, double *hist, double ticket, hipStream_t s) {
  hipLaunchKernelGGL(reduce_partials, dim3(1), dim3(kReduceThreads), 0, s, pn, pe, pen, n, scale_norm, eps,
                     scale_energy, out, hist, ticket);
  return hipGetLastError();
}

hipError_t launch_reduce_norms(const double *pn, size_t stride, int n, int steps, double scale_norm, double *hist,
                               hipStream_t s) {
  hipLaunchKernelGGL(reduce_norms, dim3(steps), dim3(kReduceThreads), 0, s, pn, stride, n, scale_norm, hist);
  return hipGetLastError();
}

hipError_t launch_norm_f64(const void *psi, int nx, int ny, int nz, int weighted, double w1, double w2, double w3,
                           double *part, hipStream_t s) {
  hipLaunchKernelGGL((norm_kernel<double, false>), dim3(PW_BLOCKS), dim3(256), 0, s, psi, nullptr, nx, ny, nz,
                     weighted, w1, w2, w3, part);
  return hipGetLastError();
}

hipError_t launch_moments(int prec, const void *psi, const void *lo, const StageArgs &A, double *p2, double *p4,
                          double *pv, hipStream_t s) {
  if (prec == 0)
    hipLaunchKernelGGL((moments_kernel<double, false>), dim3(PW_BLOCKS), dim3(256), 0, s, psi, nullptr, A.nx, A.ny,
                       A.nz, A.xl, A.yl, A.zl, A.dx, A.dy, A.dz, A.ox2, A.oy2, A.oz2, p2, p4, pv);
  else if (lo)
    hipLaunchKernelGGL((moments_kernel<float, true>), dim3(PW_BLOCKS), dim3(256), 0, s, psi, lo, A.nx, A.ny, A.nz,
                       A.xl, A.yl, A.zl, A.dx, A.dy, A.dz, A.ox2, A.oy2, A.oz2, p2, p4, pv);
  else
    hipLaunchKernelGGL((moments_kernel<float, false>), dim3(PW_BLOCKS), dim3(256), 0, s, psi, nullptr, A.nx, A.ny,
                       A.nz, A.xl, A.yl, A.zl, A.dx, A.dy, A.dz, A.ox2, A.oy2, A.oz2, p2, p4, pv);
  return hipGetLastError();
}

hipError_t launch_norm_f32(const void *psi, const void *lo, int nx, int ny, int nz, int weighted, double w1,
                           double w2, double w3, double *part, hipStream_t s) {
  if (lo)
    hipLaunchKernelGGL((norm_kernel<float, true>), dim3(PW_BLOCKS), dim3(256), 0, s, psi, lo, nx, ny, nz, weighted,
                       w1, w2, w3, part);
  else
    hipLaunchKernelGGL((norm_kernel<float, false>), dim3(PW_BLOCKS), dim3(256), 0, s, psi, nullptr, nx, ny, nz,
                       weighted, w1, w2, w3, part);
  return hipGetLastError();
}

hipError_t launch_renorm_f64(void *psi, size_t n, double a, DivC b, hipStream_t s) {
  hipLaunchKernelGGL(renorm_kernel_f64, dim3(PW_BLOCKS), dim3(256), 0, s, psi, n, a, b);
  return hipGetLastError();
}

hipError_t launch_renorm_f32(void *psi, void *lo, size_t n, double a, double b, hipStream_t s) {
  if (lo)
    hipLaunchKernelGGL(renorm_kernel_f32<true>, dim3(PW_BLOCKS), dim3(256), 0, s, psi, lo, n, a, b);
  else
    hipLaunchKernelGGL(renorm_kernel_f32<false>, dim3(PW_BLOCKS), dim3(256), 0, s, psi, nullptr, n, a, b);
  return hipGetLastError();
}

hipError_t launch_imprint(int prec, void *psi, void *lo, const LineArgs &L, hipStream_t s) {
  if (prec == 0)  // GPE_FP64
    hipLaunchKernelGGL((imprint_kernel<double, 0>), dim3(PW_BLOCKS), dim3(256), 0, s, psi, nullptr, L);
  else if (prec == 1)  // GPE_FP32: the reference built in single precision
    hipLaunchKernelGGL((imprint_kernel<float, 1>), dim3(PW_BLOCKS), dim3(256), 0, s, psi, nullptr, L);
  else
    hipLaunchKernelGGL((imprint_kernel<double, 2>), dim3(PW_BLOCKS), dim3(256), 0, s, psi, lo, L);
  return hipGetLastError();
}

// HBM bandwidth probes: read, write and copy of float4 arrays, grid-stride.
static __global__ void __launch_bounds__(256) bw_read(const float4 *__restrict__ a, size_t n, float *sink) {
  float acc = 0.f;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    float4 v = a[i];
    acc += (v.x + v.y) + (v.z + v.w);
  }
  if (acc == 1.2345e-30f) sink[0] = acc;  // keeps the loads live
}
static __global__ void __launch_bounds__(256) bw_write(float4 *__restrict__ b, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    b[i] = make_float4(0.f, 1.f, 2.f, 3.f);
}
static __global__ void __launch_bounds__(256) bw_copy(const float4 *__restrict__ a, float4 *__restrict__ b,
                                                      size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    b[i] = a[i];
}

hipError_t probe_bandwidth(size_t bytes, int reps, double *gbs) {
  const size_t n = bytes / 16;
  float4 *a = nullptr, *b = nullptr;
  float *sink = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t e = hipMalloc((void **)&a, n * 16);
  if (e == hipSuccess) e = hipMalloc((void **)&b, n * 16);
  if (e == hipSuccess) e = hipMalloc((void **)&sink, 64);
  if (e == hipSuccess) e = hipMemset(a, 0, n * 16);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  // many workgroups (65536 x 256 threads): fewer leave the write and copy
  // kernels short of outstanding requests (measured: write 4.2 TB/s at
  // 8192 workgroups, 5.9 TB/s at 65536)
  const int grid = 65536;
  for (int which = 0; which < 3 && e == hipSuccess; ++which) {
    for (int r = -1; r < reps && e == hipSuccess; ++r) {
      if (r == 0) hipEventRecord(e0, 0);
      if (which == 0) hipLaunchKernelGGL(bw_read, dim3(grid), dim3(256), 0, 0, a, n, sink);
      if (which == 1) hipLaunchKernelGGL(bw_write, dim3(grid), dim3(256), 0, 0, b, n);
      if (which == 2) hipLaunchKernelGGL(bw_copy, dim3(grid), dim3(256), 0, 0, a, b, n);
      e = hipGetLastError();
    }
    if (e != hipSuccess) break;
    hipEventRecord(e1, 0);
    e = hipEventSynchronize(e1);
    float ms = 0.f;
    hipEventElapsedTime(&ms, e0, e1);
    const double moved = (double)n * 16 * (which == 2 ? 2.0 : 1.0) * reps;
    gbs[which] = moved / (ms / 1e3) / 1e9;
  }
  if (e0) hipEventDestroy(e0);
  if (e1) hipEventDestroy(e1);
  if (a) hipFree(a);
  if (b) hipFree(b);
  if (sink) hipFree(sink);
  return e;
}

}  // namespace gpe
