// diag.hpp -- vortex diagnostics of a resident field: the vortex-line
// length (linelength, variables.f90:896-1162) and the vortex-core points
// (get_zeros, get_extra_zeros and get_re_im_zeros, io.f90:886-1393).
//
// Line length.
// Every interior cell (corners i..i+1, j..j+1, k..k+1, 1 <= i,j,k <= n-2)
// is independent except for one thing: the reference keeps its point arrays
// from cell to cell, so a cell that finds only one zero point measures the
// segment to the SECOND point of the most recent earlier cell (x-fastest
// order) that stored one.  Arithmetic is in T (double for FP64 and the
// compensated form, float for plain FP32), one rounding per operation, in the
// reference's order.
//
// Passes.  A cell on whose 8 corners Re or Im keeps one strict sign holds no
// point of either pass (a vortex cell needs both to change sign or vanish),
// and that is all but some 2% of the cells of a dense tangle, scattered so
// that nearly every wave holds one.  So one streaming pass marks the cells
// that may hold something (one bit each), a prefix sum over the marks lists
// them in cell order, and the per-cell arithmetic, which is long and
// divergent, runs over the dense list.  Whatever follows keeps the list's
// order by prefix sums: each one-point cell finds the latest earlier second
// point, and each core point its place in the file.  (One pass over all
// cells, atomically appended lists and sorting on the host took 1.9 + 2 x 1.0
// ms of kernels and 14 ms of host at 256^3; these passes take 0.3 ms, see
// gpe_diag.hip.)
#pragma once
#include <hip/hip_runtime.h>

#include "stage_args.h"

namespace gpe {

template <typename T>
struct LLFace {
  // Edge crossings of one component w[1..5] (w[5] = w[1]) of a face in face
  // coordinates; returns the reference's count index.
  __device__ static int crossings(const T w[6], T *xs, T *ys) {
    int l = 1;
#pragma unroll
    for (int q = 1; q <= 4; ++q) {
      if (w[q] == (T)0) {
        // a zero corner is recorded without advancing the index
        xs[l] = (q == 2 || q == 3) ? (T)1 : (T)0;
        ys[l] = (q >= 3) ? (T)1 : (T)0;
      } else if (w[q] * w[q + 1] < (T)0) {
        if (q == 1) {
          xs[l] = fabs(w[1] / (w[1] - w[2]));
          ys[l] = (T)0;
        } else if (q == 2) {
          xs[l] = (T)1;
          ys[l] = fabs(w[2] / (w[2] - w[3]));
        } else if (q == 3) {
          xs[l] = fabs(w[4] / (w[3] - w[4]));
          ys[l] = (T)1;
        } else {
          xs[l] = (T)0;
          ys[l] = fabs(w[5] / (w[4] - w[5]));
        }
        if (l == 1 || xs[l] != xs[l - 1] || ys[l] != ys[l - 1]) ++l;
      }
    }
    return l;
  }
};

template <typename T>
__device__ __forceinline__ bool ll_in01(T v) {
  return v == (T)0 || v == (T)1;
}

template <typename T>
__device__ __forceinline__ T ll_segment(T x1, T y1, T z1, T x2, T y2, T z2) {
  T a = (T)1;
  const bool ex = x1 == x2 && ll_in01(x1);
  const bool ey = y1 == y2 && ll_in01(y1);
  const bool ez = z1 == z2 && ll_in01(z1);
  if (ex || ey) {  // the reference tests y twice and z never here
    a = a * (T)0.5;
    if ((ex && ey) || (ey && ez)) a = a * (T)0.5;
  }
  return a * sqrt((x1 - x2) * (x1 - x2) + (y1 - y2) * (y1 - y2) + (z1 - z2) * (z1 - z2));
}

// Corners of cell c (x fastest over the interior cells), as indices and offset.
struct Cell {
  int i, j, k;
  size_t at;  // of the lower corner
};
__device__ __forceinline__ Cell cell_of(long long c, int nx, int ny) {
  const long long cx = nx - 2, cy = ny - 2;
  const long long r = c / cx;
  Cell q;
  q.i = 1 + (int)(c - r * cx);
  q.k = 1 + (int)(r / cy);
  q.j = 1 + (int)(r % cy);
  q.at = ((size_t)q.k * ny + q.j) * nx + q.i;
  return q;
}

// The 8 corners, (di, dj, dk) = bits (0, 1, 2) of the index.  S: stored real
// type; T: arithmetic type; lo: low word of the compensated form (or null).
template <typename S, typename T>
__device__ __forceinline__ void corners(const S *__restrict__ f, const S *__restrict__ lo, const Cell &q, int nx, int ny,
                                        T *cu, T *cv) {
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const size_t s = q.at + (b & 1) + (size_t)((b >> 1) & 1) * nx + (size_t)((b >> 2) & 1) * nx * ny;
    if (lo) {
      cu[b] = (T)((double)f[2 * s] + (double)lo[2 * s]);
      cv[b] = (T)((double)f[2 * s + 1] + (double)lo[2 * s + 1]);
    } else {
      cu[b] = (T)f[2 * s];
      cv[b] = (T)f[2 * s + 1];
    }
  }
}

// The cells that may hold a point, as one bit each: kCellsPerBlock cells per
// workgroup, a 64-bit word per wave and step, and the number set per
// workgroup.  which: 0 both components, 1 Re only, 2 Im only.  The compensated
// form's high word alone tells the sign: the low word is at most half its ulp.
constexpr int kCellThreads = 256, kCellSteps = 16, kCellsPerBlock = kCellThreads * kCellSteps;
template <typename S>
__global__ void __launch_bounds__(kCellThreads)
    mark_cells(const S *__restrict__ f, int nx, int ny, long long ncell, int which,
               unsigned long long *__restrict__ marks, long long *__restrict__ counts) {
  typedef S v2 __attribute__((ext_vector_type(2)));
  const v2 *g = reinterpret_cast<const v2 *>(f);
  const int cx = nx - 2, cy = ny - 2;
  const size_t plane = (size_t)nx * ny;
  long long c = (long long)blockIdx.x * kCellsPerBlock + threadIdx.x;
  Cell q = cell_of(c < ncell ? c : 0, nx, ny);
  int found = 0;
  for (int t = 0; t < kCellSteps; ++t, c += kCellThreads) {
    bool may = false;
    if (c < ncell) {
      bool up = true, dn = true, iup = true, idn = true;
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const v2 v = g[q.at + (b & 1) + (size_t)((b >> 1) & 1) * nx + (size_t)((b >> 2) & 1) * plane];
        up = up && v.x > (S)0;
        dn = dn && v.x < (S)0;
        iup = iup && v.y > (S)0;
        idn = idn && v.y < (S)0;
      }
      const bool re = !(up || dn), im = !(iup || idn);
      may = which == 0 ? re && im : which == 1 ? re : im;
    }
    const unsigned long long m = __ballot(may);
    if ((threadIdx.x & 63) == 0) marks[((size_t)blockIdx.x * kCellSteps + t) * (kCellThreads / 64) + (threadIdx.x >> 6)] = m;
    found += may;
    // the thread's next cell, without a division
    q.i += kCellThreads;
    while (q.i > cx) {
      q.i -= cx;
      if (++q.j > cy) {
        q.j = 1;
        ++q.k;
      }
    }
    q.at = (size_t)q.k * plane + (size_t)q.j * nx + q.i;
  }
  __shared__ int red[kCellThreads / 64];
  for (int o = 32; o > 0; o >>= 1) found += __shfl_xor(found, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = found;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// In place: the exclusive prefix sums of v[0 .. n-1] and, in v[n], the total
// (one workgroup).
constexpr int kScanThreads = 1024;
static __global__ void __launch_bounds__(kScanThreads) prefix_sums(long long *v, int n) {
  __shared__ long long sh[kScanThreads];
  const int per = (n + kScanThreads - 1) / kScanThreads;
  const int a = min(n, (int)threadIdx.x * per), b = min(n, a + per);
  long long sum = 0;
  for (int i = a; i < b; ++i) sum += v[i];
  sh[threadIdx.x] = sum;
  __syncthreads();
  for (int o = 1; o < kScanThreads; o <<= 1) {
    const long long add = (int)threadIdx.x >= o ? sh[threadIdx.x - o] : 0;
    __syncthreads();
    sh[threadIdx.x] += add;
    __syncthreads();
  }
  long long run = threadIdx.x ? sh[threadIdx.x - 1] : 0;
  for (int i = a; i < b; ++i) {
    const long long x = v[i];
    v[i] = run;
    run += x;
  }
  if (threadIdx.x == kScanThreads - 1) v[n] = sh[kScanThreads - 1];
}

// The marked cells in cell order: workgroup b's from base[b] on.
static __global__ void __launch_bounds__(kCellThreads)
    list_cells(const unsigned long long *__restrict__ marks, const long long *__restrict__ base,
               long long *__restrict__ list) {
  constexpr int W = kCellSteps * (kCellThreads / 64);  // words of a workgroup's cells
  static_assert(W == 64, "one word per lane");
  const unsigned long long *m = marks + (size_t)blockIdx.x * W;
  const int lane = threadIdx.x & 63;
  // every wave: prefix of the words' populations, then its own quarter of them
  const unsigned long long mine = m[lane];
  int pre = __popcll(mine);
  for (int o = 1; o < 64; o <<= 1) {
    const int up = __shfl_up(pre, o);
    if (lane >= o) pre += up;
  }
  pre -= __popcll(mine);
  for (int w = threadIdx.x >> 6; w < W; w += kCellThreads / 64) {
    const unsigned long long word = __shfl(mine, w);
    const int at = __shfl(pre, w);
    if (word >> lane & 1)
      list[base[blockIdx.x] + at + __popcll(word & ((1ull << lane) - 1))] =
          (long long)blockIdx.x * kCellsPerBlock + (long long)w * 64 + lane;
  }
}

// One cell of the line length: the number of points it stored (0, 1: one in
// p1, 2: a second one in p2), with its own share added to acc; `done` cells are
// settled by a face or an edge of zeros.
template <typename T>
__device__ __forceinline__ int ll_cell(const T *cu, const T *cv, T p1[3], T p2[3], double &acc, bool &done) {
  // corners u(1..4) of faces 1..6 (front k, back k+1, right i+1, left i,
  // top j+1, bottom j) as indices into the cube's 8 corners
  constexpr int face[6][4] = {{0, 1, 3, 2}, {4, 5, 7, 6}, {1, 5, 7, 3}, {0, 4, 6, 2}, {2, 3, 7, 6}, {0, 1, 5, 4}};
  int m = 1;
  done = false;
  T px1 = 0, py1 = 0, pz1 = 0, px2 = 0, py2 = 0, pz2 = 0;
  for (int n = 0; n < 6 && !done; ++n) {
    T u[6], v[6];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      u[q + 1] = cu[face[n][q]];
      v[q + 1] = cv[face[n][q]];
    }
    u[5] = u[1];
    v[5] = v[1];
    const bool uz = u[1] == 0 && u[2] == 0 && u[3] == 0 && u[4] == 0;
    const bool vz = v[1] == 0 && v[2] == 0 && v[3] == 0 && v[4] == 0;
    const bool vs = v[1] * v[2] < 0 || v[2] * v[3] < 0 || v[3] * v[4] < 0 || v[4] * v[1] < 0;
    const bool us = u[1] * u[2] < 0 || u[2] * u[3] < 0 || u[3] * u[4] < 0 || u[4] * u[1] < 0;
    if ((uz && vs) || (vz && us)) {  // a face of zeros
      acc += 0.5;
      done = true;
      break;
    }
#pragma unroll
    for (int q = 1; q <= 4; ++q)
      if (!done && u[q] == 0 && u[q + 1] == 0 && v[q] == 0 && v[q + 1] == 0) {  // an edge of zeros
        acc += 0.25;
        done = true;
      }
    if (done) break;
    T xu[7], yu[7], xv[7], yv[7];
    const int lu = LLFace<T>::crossings(u, xu, yu);
    const int lv = LLFace<T>::crossings(v, xv, yv);
    if (lu > 2 && lv > 2) {
      T den = xv[2] * (yu[1] - yu[2]) + xv[1] * (yu[2] - yu[1]) + (xu[1] - xu[2]) * (yv[1] - yv[2]);
      if (den == (T)0) den = den + (T)0.0000001;
      const T xx = (xu[1] * (xv[2] * (yv[1] - yu[2]) + xv[1] * (yu[2] - yv[2])) +
                    xu[2] * (xv[2] * (yu[1] - yv[1]) + xv[1] * (yv[2] - yu[1]))) / den;
      const T yy = (xv[2] * (yu[1] - yu[2]) * yv[1] + xu[1] * yu[2] * yv[1] - xv[1] * yu[1] * yv[2] -
                    xu[1] * yu[2] * yv[2] + xv[1] * yu[2] * yv[2] + xu[2] * yu[1] * (yv[2] - yv[1])) / den;
      if (xx >= 0 && xx <= 1 && yy >= 0 && yy <= 1) {
        T qx, qy, qz;
        switch (n) {
          case 0: qx = xx; qy = yy; qz = 0; break;
          case 1: qx = xx; qy = yy; qz = 1; break;
          case 2: qx = 1; qy = yy; qz = xx; break;
          case 3: qx = 0; qy = yy; qz = xx; break;
          case 4: qx = xx; qy = 1; qz = yy; break;
          default: qx = xx; qy = 0; qz = yy; break;
        }
        if (m == 1) {
          px1 = qx;
          py1 = qy;
          pz1 = qz;
        } else if (m == 2) {
          px2 = qx;
          py2 = qy;
          pz2 = qz;
        }
        ++m;
      }
    }
  }
  p1[0] = px1;
  p1[1] = py1;
  p1[2] = pz1;
  p2[0] = px2;
  p2[1] = py2;
  p2[2] = pz2;
  if (m >= 3 && !done) acc += (double)ll_segment<T>(px1, py1, pz1, px2, py2, pz2);
  return m >= 3 ? 2 : m - 1;
}

__device__ __forceinline__ double block_sum256(double acc, double *red) {
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  return ((red[0] + red[1]) + red[2]) + red[3];
}

// The listed cells' line length but for the one-point cells.  Per list entry
// the kind (0 nothing to match, 1 one-point cell, 2 stored a second point) and
// that point; per workgroup the sum and the last entry of kind 2 (or -1).
template <typename S, typename T>
__global__ void __launch_bounds__(kCellThreads)
    ll_cells(const S *__restrict__ f, const S *__restrict__ lo, int nx, int ny, const long long *__restrict__ list,
             long long n, double *__restrict__ pts, signed char *__restrict__ kind, double *__restrict__ part,
             long long *__restrict__ last) {
  __shared__ double red[4];
  __shared__ int lastw[4];
  const long long t = (long long)blockIdx.x * kCellThreads + threadIdx.x;
  double acc = 0.0;
  int what = 0;
  if (t < n) {
    T cu[8], cv[8], p1[3], p2[3];
    const Cell q = cell_of(list[t], nx, ny);
    corners<S, T>(f, lo, q, nx, ny, cu, cv);
    bool done;
    what = ll_cell<T>(cu, cv, p1, p2, acc, done);
    if (what == 1 && done) what = 0;
    kind[t] = (signed char)what;
    if (what) {
      const T *p = what == 1 ? p1 : p2;
      pts[3 * t] = (double)p[0];
      pts[3 * t + 1] = (double)p[1];
      pts[3 * t + 2] = (double)p[2];
    }
  }
  const unsigned long long w = __ballot(what == 2);
  if ((threadIdx.x & 63) == 0) lastw[threadIdx.x >> 6] = w ? 63 - __clzll(w) : -1;
  const double sum = block_sum256(acc, red);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = sum;
    long long l = -1;
    for (int v = 0; v < 4; ++v)
      if (lastw[v] >= 0) l = (long long)blockIdx.x * kCellThreads + 64 * v + lastw[v];
    last[blockIdx.x] = l;
  }
}

// In place: the largest of v[0 .. i-1] (-1 before any), one workgroup.
static __global__ void __launch_bounds__(kScanThreads) prefix_max(long long *v, int n) {
  __shared__ long long sh[kScanThreads];
  const int per = (n + kScanThreads - 1) / kScanThreads;
  const int a = min(n, (int)threadIdx.x * per), b = min(n, a + per);
  long long top = -1;
  for (int i = a; i < b; ++i) top = max(top, v[i]);
  sh[threadIdx.x] = top;
  __syncthreads();
  for (int o = 1; o < kScanThreads; o <<= 1) {
    const long long u = (int)threadIdx.x >= o ? sh[threadIdx.x - o] : -1;
    __syncthreads();
    sh[threadIdx.x] = max(sh[threadIdx.x], u);
    __syncthreads();
  }
  long long run = threadIdx.x ? sh[threadIdx.x - 1] : -1;
  for (int i = a; i < b; ++i) {
    const long long x = v[i];
    v[i] = run;
    run = max(run, x);
  }
}

// Segments of the one-point cells to the latest earlier second point (the
// origin before any; variables.f90:1140-1153).
template <typename T>
__global__ void __launch_bounds__(kCellThreads)
    ll_one_point(const double *__restrict__ pts, const signed char *__restrict__ kind, long long n,
                 const long long *__restrict__ before, double *__restrict__ part) {
  __shared__ double red[4];
  __shared__ unsigned long long seconds[4];
  const long long first = (long long)blockIdx.x * kCellThreads, t = first + threadIdx.x;
  const int what = t < n ? kind[t] : 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long w = __ballot(what == 2);
  if (lane == 0) seconds[wave] = w;
  __syncthreads();
  double acc = 0.0;
  if (what == 1) {
    long long l = before[blockIdx.x];
    for (int v = 0; v < wave; ++v)
      if (seconds[v]) l = first + 64 * v + 63 - __clzll(seconds[v]);
    const unsigned long long own = w & ((1ull << lane) - 1);
    if (own) l = first + 64 * wave + 63 - __clzll(own);
    T x = 0, y = 0, z = 0;
    if (l >= 0) {
      x = (T)pts[3 * l];
      y = (T)pts[3 * l + 1];
      z = (T)pts[3 * l + 2];
    }
    acc = (double)ll_segment<T>((T)pts[3 * t], (T)pts[3 * t + 1], (T)pts[3 * t + 2], x, y, z);
  }
  const double sum = block_sum256(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = sum;
}

// ---- vortex-core points -----------------------------------------------------
// One thread per interior lower corner (i, j, k), 1 <= i,j,k <= n-2, as the
// reference's loops; every test of one cell is independent of the others.
// The points go to their places in the reference's file order, (section,
// cell): counted per section and workgroup, then written behind prefix sums.
//
// which = 0 (the zeros file): sections 0..2 are the edges in x, y, z on
// which Re and Im both change sign, or vanish at the first corner
// (io.f90:924-931), the point being where the linear interpolant of Re
// vanishes; sections 3..5 are the xy, xz and yz faces around which Re and Im
// change sign on alternate edges (io.f90:1039-1098 and its xz/yz copies),
// the point being the crossing of the line through the two crossings of one
// component with the line through the two crossings of the other, formed
// with the reference's slopes.  which = 1 / 2 (re_zeros / im_zeros): edges
// on which that component vanishes at the first corner or changes sign; in z
// the reference joins the two tests with .and. (io.f90:1304, 1375), kept as
// written.  Arithmetic in T, one rounding per operation, in the reference's
// order (the translation unit is built without contraction).

template <typename T>
__device__ __forceinline__ T zr_interp(T w0, T w1, T a0, T a1, T d) {
  return -(w1 * a0 / d) + w0 * a1 / d;
}

template <typename T>
__device__ __forceinline__ bool zr_edge(T r0, T i0, T r1, T i1) {
  return (r0 == (T)0 && i0 == (T)0) || (r0 == (T)0 && i0 * i1 < (T)0) || (i0 == (T)0 && r0 * r1 < (T)0) ||
         (r0 * r1 < (T)0 && i0 * i1 < (T)0);
}

// corners u[1..4], v[1..4] around a face (a0,b0), (a1,b0), (a1,b1), (a0,b1):
// u changes sign on edges 1-2 and 3-4 only, v on 2-3 and 4-1 only
template <typename T>
__device__ __forceinline__ bool zr_face_pattern(const T *u, const T *v) {
  return (u[1] * u[2] < (T)0 && v[1] * v[2] >= (T)0) && (v[2] * v[3] < (T)0 && u[2] * u[3] >= (T)0) &&
         (u[3] * u[4] < (T)0 && v[3] * v[4] >= (T)0) && (v[4] * v[1] < (T)0 && u[4] * u[1] >= (T)0);
}

template <typename T>
__device__ __forceinline__ void zr_face_point(const T *u, const T *v, T a0, T a1, T b0, T b1, T &ap, T &bp) {
  const T z1 = zr_interp<T>(u[1], u[2], a0, a1, u[1] - u[2]);
  const T z2 = zr_interp<T>(v[2], v[3], b0, b1, v[2] - v[3]);
  const T z3 = zr_interp<T>(u[3], u[4], a1, a0, u[3] - u[4]);
  const T z4 = zr_interp<T>(v[4], v[1], b1, b0, v[4] - v[1]);
  const T m1 = (b0 - b1) / (z1 - z3);
  const T m2 = (z2 - z4) / (a1 - a0);
  const T a = (z4 - a0 * m2 - b0 + z1 * m1) / (m1 - m2);
  ap = a;
  bp = a * m1 + b0 - z1 * m1;
}

// The points of one cell: emit(section, x, y, z) for each, sections ascending.
template <typename T, typename Emit>
__device__ __forceinline__ void zr_cell(const T *re, const T *im, T x0, T x1, T y0, T y1, T z0, T z1, int which,
                                        Emit emit) {
  const int nsec = which == 0 ? 6 : 3;
  for (int sec = 0; sec < nsec; ++sec) {
    T px = x0, py = y0, pz = z0;
    bool hit = false;
    if (sec < 3) {
      const int q1 = 1 << sec;  // the edge's far corner: +x, +y or +z
      T w0, w1;
      bool cond;
      if (which == 0) {
        w0 = re[0];
        w1 = re[q1];
        cond = zr_edge<T>(re[0], im[0], re[q1], im[q1]);
      } else {
        w0 = which == 1 ? re[0] : im[0];
        w1 = which == 1 ? re[q1] : im[q1];
        cond = sec < 2 ? (w0 == (T)0 || w0 * w1 < (T)0) : (w0 == (T)0 && w0 * w1 < (T)0);
      }
      if (cond) {
        const T d = w0 - w1;
        if (d != (T)0) {
          hit = true;
          if (sec == 0) px = zr_interp<T>(w0, w1, x0, x1, d);
          else if (sec == 1) py = zr_interp<T>(w0, w1, y0, y1, d);
          else pz = zr_interp<T>(w0, w1, z0, z1, d);
        }
      }
    } else {
      // c1..c4 as corner indices, and the face axes (a, b)
      int c2, c3, c4;
      T a0, a1, b0, b1;
      if (sec == 3) {         // i,j,k --> i+1,j,k --> i+1,j+1,k --> i,j+1,k
        c2 = 1; c3 = 3; c4 = 2;
        a0 = x0; a1 = x1; b0 = y0; b1 = y1;
      } else if (sec == 4) {  // i,j,k --> i+1,j,k --> i+1,j,k+1 --> i,j,k+1
        c2 = 1; c3 = 5; c4 = 4;
        a0 = x0; a1 = x1; b0 = z0; b1 = z1;
      } else {                // i,j,k --> i,j,k+1 --> i,j+1,k+1 --> i,j+1,k
        c2 = 4; c3 = 6; c4 = 2;
        a0 = z0; a1 = z1; b0 = y0; b1 = y1;
      }
      const T u[5] = {(T)0, re[0], re[c2], re[c3], re[c4]};
      const T v[5] = {(T)0, im[0], im[c2], im[c3], im[c4]};
      T ap = 0, bp = 0;
      if (zr_face_pattern<T>(u, v)) {
        zr_face_point<T>(u, v, a0, a1, b0, b1, ap, bp);
        hit = true;
      } else if (zr_face_pattern<T>(v, u)) {
        zr_face_point<T>(v, u, a0, a1, b0, b1, ap, bp);
        hit = true;
      }
      if (hit) {
        if (sec == 3) { px = ap; py = bp; }
        else if (sec == 4) { px = ap; pz = bp; }
        else { pz = ap; py = bp; }
      }
    }
    if (hit) emit(sec, px, py, pz);
  }
}

struct ZrGrid {
  double xl, yl, zl, dx, dy, dz;
  int nx, ny;
};

// emit(section, cell, x, y, z) for the points of the list's entry t.
template <typename S, typename T, typename Emit>
__device__ __forceinline__ void zr_entry(const S *f, const S *lo, const ZrGrid &g, long long c, int which, Emit emit) {
  const Cell q = cell_of(c, g.nx, g.ny);
  T re[8], im[8];
  corners<S, T>(f, lo, q, g.nx, g.ny, re, im);
  const T txl = (T)g.xl, tyl = (T)g.yl, tzl = (T)g.zl, dx = (T)g.dx, dy = (T)g.dy, dz = (T)g.dz;
  // x(i) = xl + real(i)*dx (ic.f90:53-66)
  zr_cell<T>(re, im, txl + (T)q.i * dx, txl + (T)(q.i + 1) * dx, tyl + (T)q.j * dy, tyl + (T)(q.j + 1) * dy,
             tzl + (T)q.k * dz, tzl + (T)(q.k + 1) * dz, which,
             [&](int sec, T x, T y, T z) { emit(sec, (long long)q.at, (double)x, (double)y, (double)z); });
}

// Points per section and workgroup of the list, counts[section * gridDim.x + b].
template <typename S, typename T>
__global__ void __launch_bounds__(kCellThreads)
    zr_count(const S *__restrict__ f, const S *__restrict__ lo, const ZrGrid g, int which,
             const long long *__restrict__ list, long long n, long long *__restrict__ counts) {
  __shared__ int hits[6];
  if (threadIdx.x < 6) hits[threadIdx.x] = 0;
  __syncthreads();
  const long long t = (long long)blockIdx.x * kCellThreads + threadIdx.x;
  unsigned has = 0;
  if (t < n)
    zr_entry<S, T>(f, lo, g, list[t], which, [&](int sec, long long, double, double, double) { has |= 1u << sec; });
  for (int s = 0; s < 6; ++s) {
    const int m = __popcll(__ballot(has >> s & 1));
    if ((threadIdx.x & 63) == 0 && m) atomicAdd(&hits[s], m);
  }
  __syncthreads();
  const int nsec = which == 0 ? 6 : 3;
  if ((int)threadIdx.x < nsec) counts[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = hits[threadIdx.x];
}

// The points, each at its place (base: prefix sums of zr_count's counts).
template <typename S, typename T>
__global__ void __launch_bounds__(kCellThreads)
    zr_write(const S *__restrict__ f, const S *__restrict__ lo, const ZrGrid g, int which,
             const long long *__restrict__ list, long long n, const long long *__restrict__ base,
             ZeroPoint *__restrict__ out) {
  __shared__ int hits[6][kCellThreads / 64];
  const long long t = (long long)blockIdx.x * kCellThreads + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned has = 0;
  ZeroPoint p[6];
  if (t < n)
    zr_entry<S, T>(f, lo, g, list[t], which, [&](int sec, long long cell, double x, double y, double z) {
#pragma unroll
      for (int s = 0; s < 6; ++s)
        if (s == sec) p[s] = ZeroPoint{sec, 0, cell, x, y, z};
      has |= 1u << sec;
    });
  int rank[6];
#pragma unroll
  for (int s = 0; s < 6; ++s) {
    const unsigned long long m = __ballot(has >> s & 1);
    rank[s] = __popcll(m & ((1ull << lane) - 1));
    if (lane == 0) hits[s][wave] = __popcll(m);
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 6; ++s) {
    if (!(has >> s & 1)) continue;
    long long at = base[(size_t)s * gridDim.x + blockIdx.x] + rank[s];
    for (int v = 0; v < wave; ++v) at += hits[s][v];
    out[at] = p[s];
  }
}

}  // namespace gpe
