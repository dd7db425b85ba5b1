// brick.hpp -- a stage sweep in bricks of 64 x NW x ZB sites.
//
// The z march (stencil.hpp) reads every field once, but a workgroup walks its
// planes one after another, each with a barrier and the latency of its loads
// and of the right-hand side's dependent operations behind it.  A grid that
// gives few tiles to march at once spends its time on that chain.  A brick is
// short in z: each thread loads its whole column (ZB sites and R neighbours on
// either side) and its share of the ghost cells together, one barrier hands
// the stage inputs over in LDS, and the ZB sites are then independent of one
// another.  A field value is read about (ZB + 2R)/ZB + 2R/NW times, from L2 or
// the Infinity Cache for all but the first.  Every value comes from the same
// expressions as in the march, so the fields are the same bits.
#pragma once
#include "stencil.hpp"

namespace gpe {

// Sites (64 tx .. , NW ty .. , z0 .. z0+ZB-1) of one stage sweep; partial sums
// as stage_tile.
template <typename T, int R, int NW, int ZB, int KIND, bool COMP>
__device__ __forceinline__ void brick_tile(Args<T> &A, const int tx, const int ty, const int z0, const int slot,
                                           double *pn, double *pe, double *pen) {
  constexpr int TX = 64, LX = TX + 2 * R, LY = NW + 2 * R, NT = 64 * NW;
  constexpr int NC = ZB + 2 * R;  // planes of a column
  constexpr int NF = FifoInfo<KIND, COMP>::nf, NFA = NF > 0 ? NF : 1;
  constexpr int NO = OutInfo<KIND, COMP>::no, NOA = NO > 0 ? NO : 1;
  constexpr int NYH = 2 * R * TX, NH = NYH + 2 * R * NW;  // ghost cells of a plane
  constexpr int HPT = (NH * ZB + NT - 1) / NT;
  using V = vec2_t<T>;
  __shared__ V lds[ZB][LY * LX];
  __shared__ double red[3][NW];

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nx = A.nx, ny = A.ny, nz = A.nz, per = A.periodic;
  const size_t plane = (size_t)nx * (size_t)ny;
  const int gi = tx * TX + lane, gj = ty * NW + wave;
  // loads at the boundary-mapped offset (always in range), stores inside the grid
  const int gim = bcmap(min(gi, nx - 1 + R), nx, per), gjm = bcmap(min(gj, ny - 1 + R), ny, per);
  const int off = gjm * nx + gim;
  auto zplane = [&](int k) { return (size_t)bcmap(min(k, nz - 1 + R), nz, per) * plane; };

  const cx<T> H = stage_coef<T, KIND>(A);
  cx<T> u[NC], F[ZB][NFA], o[ZB][NOA];
#pragma unroll
  for (int m = 0; m < NC; ++m) {
    Raw<T, KIND> r;
    const bool own = m >= R && m < R + ZB;
    load_raw<T, KIND>(A, zplane(z0 - R + m) + off, r, own);
    u[m] = stage_input<T, KIND, COMP>(H, r);
    if (own) {
      out_terms<T, KIND, COMP>(A, r, F[m - R]);
      load_out<T, KIND, COMP>(A, zplane(z0 - R + m) + off, o[m - R]);
    }
  }
#pragma unroll
  for (int i = 0; i < HPT; ++i) {
    const int h = threadIdx.x + i * NT;
    if (h < NH * ZB) {
      const int b = h / NH, g = h - b * NH;
      int lr, lc;
      if (g < NYH) {
        const int rs = g / TX;
        lr = rs < R ? rs : NW + rs;
        lc = g - rs * TX + R;
      } else {
        const int rs = (g - NYH) / (2 * R), cs = (g - NYH) - rs * (2 * R);
        lr = rs + R;
        lc = cs < R ? cs : TX + cs;
      }
      const int hi = bcmap(min(tx * TX + lc - R, nx - 1 + R), nx, per);
      const int hj = bcmap(min(ty * NW + lr - R, ny - 1 + R), ny, per);
      Raw<T, KIND> r;
      load_raw<T, KIND>(A, zplane(z0 + b) + (hj * nx + hi), r, false);
      const cx<T> w = stage_input<T, KIND, COMP>(H, r);
      V v;
      v.x = w.re;
      v.y = w.im;
      lds[b][lr * LX + lc] = v;
    }
  }
  const int c = (wave + R) * LX + lane + R;
#pragma unroll
  for (int b = 0; b < ZB; ++b) {
    V v;
    v.x = u[b + R].re;
    v.y = u[b + R].im;
    lds[b][c] = v;
  }
  lds_barrier();

  const double wxy = nweight(gi, nx, A.w1, A.w2, A.w3) * nweight(gj, ny, A.w1, A.w2, A.w3);
  Sums<T> sum;
#pragma unroll
  for (int b = 0; b < ZB; ++b) {
    auto at = [&](int d) {
      const V v = lds[b][c + d];
      return mk<T>(v.x, v.y);
    };
    const cx<T> c0 = u[b + R];
    const cx<T> xm1 = at(-1), xp1 = at(1), ym1 = at(-LX), yp1 = at(LX), zm1 = u[b + R - 1], zp1 = u[b + R + 1];
    cx<T> xm2 = xm1, xp2 = xp1, ym2 = ym1, yp2 = yp1;
    if constexpr (R == 2) {
      xm2 = at(-2);
      xp2 = at(2);
      ym2 = at(-2 * LX);
      yp2 = at(2 * LX);
    }
    const cx<T> dxx = d2<T, R>(xm2, xm1, c0, xp1, xp2, div_of(A.d_xx), A.inv_xx);
    const cx<T> dyy = d2<T, R>(ym2, ym1, c0, yp1, yp2, div_of(A.d_yy), A.inv_yy);
    const cx<T> dzz = d2<T, R>(u[b], zm1, c0, zp1, u[b + 2 * R], div_of(A.d_zz), A.inv_zz);
    const int k = z0 + b;
    emit_site<T, R, KIND, COMP>(A, gi < nx && gj < ny && k < nz, (size_t)k * plane + (size_t)gj * nx + gi, gi, gj, k,
                                c0, (dxx + dyy) + dzz, xm2, xm1, xp1, xp2, F[b], o[b],
                                wxy * nweight(k, nz, A.w1, A.w2, A.w3), sum);
  }
  block_sums<T, KIND, COMP, NW>(sum, red, slot, pn, pe, pen);
}

// One workgroup per brick, contiguous ranges of bricks per XCD (as stage_kernel).
template <typename T, int R, int NW, int ZB, int KIND, bool COMP>
__global__ void __launch_bounds__(64 * NW) brick_kernel(const StageArgs D) {
  Args<T> &A = only_argument<T>(D);
  const int nb = A.nblocks, b = blockIdx.x;
  const int xcd = b & 7, q8 = nb >> 3, r8 = nb & 7;
  const int L = xcd * q8 + (xcd < r8 ? xcd : r8) + (b >> 3);
  const int tx = L % A.ntx, rest = L / A.ntx;
  brick_tile<T, R, NW, ZB, KIND, COMP>(A, tx, rest % A.nty, rest / A.nty * ZB, b, A.part_norm, A.part_emax,
                                       A.part_energy);
}

// Many simulations: the work table holds the bricks of every instance in
// order; each XCD's workgroups walk one contiguous part of it (gridDim.x is a
// multiple of 8).
template <typename T, int R, int NW, int ZB, int KIND, bool COMP>
__global__ void __launch_bounds__(64 * NW)
    brick_kernel_batched(const StageArgs *__restrict__ insts, const WorkItem *__restrict__ work, int nwork,
                         const int *__restrict__ active, double *pn, double *pe) {
  const int xcd = blockIdx.x & 7, q8 = nwork >> 3, r8 = nwork & 7;
  const int first = xcd * q8 + min(xcd, r8), end = first + q8 + (xcd < r8);
  for (int w = first + (blockIdx.x >> 3); w < end; w += gridDim.x >> 3) {
    const WorkItem it = work[w];
    if (active[it.inst])
      brick_tile<T, R, NW, ZB, KIND, COMP>(args_at<T>(insts + it.inst), it.tx, it.ty, it.z0, it.slot, pn, pe, nullptr);
    __syncthreads();  // the next item reuses the LDS bricks
  }
}

}  // namespace gpe
