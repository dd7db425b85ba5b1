// gpe_diag.h -- vortex diagnostics of a device field (gpe_diag.hip, diag.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "host_common.h"

namespace gpe {

// Device memory of the diagnostic passes, grown on demand and kept with its
// owner.
struct DiagWork {
  enum { kMarks, kCounts, kList, kPoints, kKinds, kParts, kOut, kBuffers };
  struct Buffer {
    void *p = nullptr;
    size_t bytes = 0;
  } buf[kBuffers];
  ~DiagWork();
};

// linelength (variables.f90:896-1162) of a field in storage form prec (lo: the
// compensated form's low word or null) on stream s.
int diag_linelength(DiagWork &w, int prec, const void *psi, const void *lo, int nx, int ny, int nz, double dx,
                    double *length, hipStream_t s);
// Vortex-core points (gpe_sim_zeros): *count points found, the first
// min(*count, cap) of them, in file order, in out.
int diag_zeros(DiagWork &w, int prec, const void *psi, const void *lo, int nx, int ny, int nz, const double *xyzl,
               const double *dxyz, int which, ZeroPoint *out, long long cap, long long *count, hipStream_t s);

}  // namespace gpe
