// host_common.cpp -- host helpers shared by the single-simulation and the
// batch entry points: the launch descriptor's constant part (field transfers
// are in transfer.hip, error reporting in errors.cpp).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <string>
#include <vector>

#include "host_common.h"

namespace gpe {

void fill_base(const gpe_params *params, int prec, StageArgs &A) {
  const int R = params->order / 2;

  A.nx = params->nx;
  A.ny = params->ny;
  A.nz = params->nz;
  A.periodic = params->bcs == 1;
  A.eqn = params->eqn;
  A.use_diss = params->diss_amp != 0.0;
  A.use_urhs = params->urhs != 0.0;
  A.scale_real = params->real_time ? 1 : 0;
  A.xl = params->xl;
  A.yl = params->yl;
  A.zl = params->zl;
  A.dx = params->dx;
  A.dy = params->dy;
  A.dz = params->dz;
  A.g = params->g;
  A.mu = params->mu;
  A.ox2 = params->omx * params->omx;
  A.oy2 = params->omy * params->omy;
  A.oz2 = params->omz * params->omz;
  A.urhs = params->urhs;
  A.diss_amp = params->diss_amp;
  // a = x(nx-3) etc. (solve.f90:397-399)
  A.a_diss = params->xl + (double)(params->nx - 3) * params->dx;
  A.b_diss = params->yl + (double)(params->ny - 3) * params->dy;
  A.c_diss = params->zl + (double)(params->nz - 3) * params->dz;
  const double dx2 = params->dx * params->dx, dy2 = params->dy * params->dy, dz2 = params->dz * params->dz;
  const double sxx = R == 1 ? dx2 : 12.0 * dx2;
  const double syy = R == 1 ? dy2 : 12.0 * dy2;
  const double szz = R == 1 ? dz2 : 12.0 * dz2;
  const double sx = R == 1 ? 2.0 * params->dx : 12.0 * params->dx;
  if (prec == GPE_FP32) {
    // the reference built with pr = single forms these in single precision
    const float fdx = (float)params->dx, fdy = (float)params->dy, fdz = (float)params->dz;
    const float fx2 = fdx * fdx, fy2 = fdy * fdy, fz2 = fdz * fdz;
    A.inv_xx = 1.0 / (double)(R == 1 ? fx2 : 12.0f * fx2);
    A.inv_yy = 1.0 / (double)(R == 1 ? fy2 : 12.0f * fy2);
    A.inv_zz = 1.0 / (double)(R == 1 ? fz2 : 12.0f * fz2);
    A.inv_x = 1.0 / (double)(R == 1 ? 2.0f * fdx : 12.0f * fdx);
  } else {
    A.inv_xx = 1.0 / sxx;
    A.inv_yy = 1.0 / syy;
    A.inv_zz = 1.0 / szz;
    A.inv_x = 1.0 / sx;
  }
  A.d_xx = make_divc(sxx);
  A.d_yy = make_divc(syy);
  A.d_zz = make_divc(szz);
  A.d_x = make_divc(sx);
  A.d6 = make_divc(6.0);
  A.d3 = make_divc(3.0);
  A.w1 = 3.0 / 8.0;
  A.w2 = 7.0 / 6.0;
  A.w3 = 23.0 / 24.0;
  }

}  // namespace gpe
