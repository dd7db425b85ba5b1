// gpe_brick.hip -- the brick sweeps (brick.hpp) of one precision, built like
// the stage kernels of gpe_stage.hip.
#include "brick.hpp"
#include "launch.h"

#ifdef GPE_F64
#define GPE_REAL double
#define GPE_BRICK launch_brick_f64
#define GPE_BRICK_B launch_brick_batched_f64
#else
#define GPE_REAL float
#define GPE_BRICK launch_brick_f32
#define GPE_BRICK_B launch_brick_batched_f32
#endif

namespace gpe {

namespace {
template <int R, int KIND, bool COMP>
hipError_t launch_one(int planes, const StageArgs &A, hipStream_t s) {
#ifdef GPE_F64
  // bricks of 4 planes: only the kinds brick_planes gives them to
  if constexpr (stage_reads(KIND) <= 2 && KIND != K_ENERGY)
    if (planes == 4) {
      hipLaunchKernelGGL((brick_kernel<GPE_REAL, R, kBrickWaves, 4, KIND, COMP>), dim3(A.nblocks),
                         dim3(64 * kBrickWaves), 0, s, A);
      return hipGetLastError();
    }
#endif
  if (planes != 2) return hipErrorInvalidValue;
  hipLaunchKernelGGL((brick_kernel<GPE_REAL, R, kBrickWaves, 2, KIND, COMP>), dim3(A.nblocks), dim3(64 * kBrickWaves),
                     0, s, A);
  return hipGetLastError();
}

template <int R, int KIND, bool COMP>
hipError_t launch_one_b(int planes, const BatchLaunch &B, hipStream_t s) {
#ifdef GPE_F64
  if constexpr (stage_reads(KIND) <= 2)
    if (planes == 4) {
      hipLaunchKernelGGL((brick_kernel_batched<GPE_REAL, R, kBrickWaves, 4, KIND, COMP>), dim3(B.grid),
                         dim3(64 * kBrickWaves), 0, s, B.insts, B.work, B.nwork, B.active, B.pn, B.pe);
      return hipGetLastError();
    }
#endif
  if (planes != 2) return hipErrorInvalidValue;
  hipLaunchKernelGGL((brick_kernel_batched<GPE_REAL, R, kBrickWaves, 2, KIND, COMP>), dim3(B.grid),
                     dim3(64 * kBrickWaves), 0, s, B.insts, B.work, B.nwork, B.active, B.pn, B.pe);
  return hipGetLastError();
}

template <int R, bool COMP>
hipError_t launch_rb(int planes, int kind, const BatchLaunch &B, hipStream_t s) {
  switch (kind) {
    case K_EULER: return launch_one_b<R, K_EULER, COMP>(planes, B, s);
    case K_RK2_1: return launch_one_b<R, K_RK2_1, false>(planes, B, s);
    case K_RK2_2: return launch_one_b<R, K_RK2_2, COMP>(planes, B, s);
    case K_RK4_1: return launch_one_b<R, K_RK4_1, false>(planes, B, s);
    case K_RK4_2: return launch_one_b<R, K_RK4_2, false>(planes, B, s);
    case K_RK4_3: return launch_one_b<R, K_RK4_3, false>(planes, B, s);
    case K_RK4_4: return launch_one_b<R, K_RK4_4, COMP>(planes, B, s);
    case K_CK_1: return launch_one_b<R, K_CK_1, COMP>(planes, B, s);
    case K_CK_2: return launch_one_b<R, K_CK_2, COMP>(planes, B, s);
    case K_CK_3: return launch_one_b<R, K_CK_3, COMP>(planes, B, s);
    case K_CK_4: return launch_one_b<R, K_CK_4, COMP>(planes, B, s);
    case K_CK_5: return launch_one_b<R, K_CK_5, COMP>(planes, B, s);
    case K_CK_6: return launch_one_b<R, K_CK_6, COMP>(planes, B, s);
    default: return hipErrorInvalidValue;
  }
}

template <int R, bool COMP>
hipError_t launch_r(int planes, int kind, const StageArgs &A, hipStream_t s) {
  switch (kind) {
    case K_RHS: return launch_one<R, K_RHS, false>(planes, A, s);
    case K_EULER: return launch_one<R, K_EULER, COMP>(planes, A, s);
    case K_RK2_1: return launch_one<R, K_RK2_1, false>(planes, A, s);
    case K_RK2_2: return launch_one<R, K_RK2_2, COMP>(planes, A, s);
    case K_RK4_1: return launch_one<R, K_RK4_1, false>(planes, A, s);
    case K_RK4_2: return launch_one<R, K_RK4_2, false>(planes, A, s);
    case K_RK4_3: return launch_one<R, K_RK4_3, false>(planes, A, s);
    case K_RK4_4: return launch_one<R, K_RK4_4, COMP>(planes, A, s);
    case K_CK_1: return launch_one<R, K_CK_1, COMP>(planes, A, s);
    case K_CK_2: return launch_one<R, K_CK_2, COMP>(planes, A, s);
    case K_CK_3: return launch_one<R, K_CK_3, COMP>(planes, A, s);
    case K_CK_4: return launch_one<R, K_CK_4, COMP>(planes, A, s);
    case K_CK_5: return launch_one<R, K_CK_5, COMP>(planes, A, s);
    case K_CK_6: return launch_one<R, K_CK_6, COMP>(planes, A, s);
    case K_ENERGY: return launch_one<R, K_ENERGY, false>(planes, A, s);
    default: return hipErrorInvalidValue;
  }
}
}  // namespace

hipError_t GPE_BRICK(int planes, int kind, int radius, bool comp, const StageArgs &A, hipStream_t s) {
#ifdef GPE_F64
  (void)comp;
  return radius == 1 ? launch_r<1, false>(planes, kind, A, s) : launch_r<2, false>(planes, kind, A, s);
#else
  if (radius == 1) return comp ? launch_r<1, true>(planes, kind, A, s) : launch_r<1, false>(planes, kind, A, s);
  return comp ? launch_r<2, true>(planes, kind, A, s) : launch_r<2, false>(planes, kind, A, s);
#endif
}

hipError_t GPE_BRICK_B(int planes, int kind, int radius, bool comp, const BatchLaunch &B, hipStream_t s) {
#ifdef GPE_F64
  (void)comp;
  return radius == 1 ? launch_rb<1, false>(planes, kind, B, s) : launch_rb<2, false>(planes, kind, B, s);
#else
  if (radius == 1) return comp ? launch_rb<1, true>(planes, kind, B, s) : launch_rb<1, false>(planes, kind, B, s);
  return comp ? launch_rb<2, true>(planes, kind, B, s) : launch_rb<2, false>(planes, kind, B, s);
#endif
}

}  // namespace gpe
