// gpe_diag.hip -- the vortex diagnostics' passes (diag.hpp) and their order.
// Built with -ffp-contract=off.
//
// At 256^3, FP32C, a random-phase tangle: marking the cells 53 us (the field's
// high words read once at 2.5 TB/s, the other corners from L1 and L2), listing
// them 14, the segments of the line length 49, the core points 45 to write and
// as much to count.  The line length and the points, with the points' copy to
// the host, the norms, the spectrum and the condensed fraction make a save step
// of 3.1 ms (20.2 ms with one pass per question over all cells and lists
// sorted on the host).
#include "gpe_diag.h"

#include <algorithm>
#include <vector>

#include "diag.hpp"

namespace gpe {

DiagWork::~DiagWork() {
  for (Buffer &b : buf)
    if (b.p) (void)hipFree(b.p);
}

namespace {

// Buffer `which` with room for n values of V (its contents are lost when it
// grows).
template <typename V>
int room(DiagWork &w, int which, size_t n, V **out) {
  DiagWork::Buffer &b = w.buf[which];
  const size_t bytes = std::max<size_t>(256, n * sizeof(V));
  if (b.bytes < bytes) {
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.bytes = 0;
    const size_t want = bytes + bytes / 4;
    if (hipMalloc(&b.p, want) != hipSuccess) return fail(GPE_ENOMEM, "diagnostic lists of %zu bytes", want);
    b.bytes = want;
  }
  *out = static_cast<V *>(b.p);
  return GPE_OK;
}

// Grids have to fit one launch dimension.
int blocks(long long n, int per) { return (int)((n + per - 1) / per); }

int read_back(const long long *dev, long long *host, hipStream_t s) {
  GPE_HIPCHK(hipMemcpyAsync(host, dev, sizeof *host, hipMemcpyDeviceToHost, s));
  GPE_HIPCHK(hipStreamSynchronize(s));
  return GPE_OK;
}

// The cells that may hold a point, in cell order.
int list_of_cells(DiagWork &w, int prec, const void *psi, int nx, int ny, int nz, int which, long long **list,
                  long long *n, hipStream_t s) {
  const long long ncell = (long long)(nx - 2) * (ny - 2) * (nz - 2);
  const int nb = blocks(ncell, kCellsPerBlock);
  unsigned long long *marks;
  long long *counts;
  if (int rc = room(w, DiagWork::kMarks, (size_t)nb * kCellSteps * (kCellThreads / 64), &marks)) return rc;
  if (int rc = room(w, DiagWork::kCounts, (size_t)nb + 1, &counts)) return rc;
  if (prec == GPE_FP64)
    hipLaunchKernelGGL(mark_cells<double>, dim3(nb), dim3(kCellThreads), 0, s, (const double *)psi, nx, ny, ncell, which,
                       marks, counts);
  else
    hipLaunchKernelGGL(mark_cells<float>, dim3(nb), dim3(kCellThreads), 0, s, (const float *)psi, nx, ny, ncell, which,
                       marks, counts);
  hipLaunchKernelGGL(prefix_sums, dim3(1), dim3(kScanThreads), 0, s, counts, nb);
  GPE_HIPCHK(hipGetLastError());
  if (int rc = read_back(counts + nb, n, s)) return rc;
  if (int rc = room(w, DiagWork::kList, (size_t)*n, list)) return rc;
  hipLaunchKernelGGL(list_cells, dim3(nb), dim3(kCellThreads), 0, s, marks, counts, *list);
  GPE_HIPCHK(hipGetLastError());
  return GPE_OK;
}

template <typename S, typename T>
int linelength_sum(DiagWork &w, const void *psi, const void *lo, int nx, int ny, const long long *list, long long n,
                   double *sum, hipStream_t s) {
  const int nb = blocks(n, kCellThreads);
  double *pts, *part;
  signed char *kind;
  long long *last;
  if (int rc = room(w, DiagWork::kPoints, 3 * (size_t)n, &pts)) return rc;
  if (int rc = room(w, DiagWork::kKinds, (size_t)n, &kind)) return rc;
  if (int rc = room(w, DiagWork::kParts, 2 * (size_t)nb, &part)) return rc;
  if (int rc = room(w, DiagWork::kCounts, (size_t)nb, &last)) return rc;
  hipLaunchKernelGGL((ll_cells<S, T>), dim3(nb), dim3(kCellThreads), 0, s, (const S *)psi, (const S *)lo, nx, ny, list,
                     n, pts, kind, part, last);
  hipLaunchKernelGGL(prefix_max, dim3(1), dim3(kScanThreads), 0, s, last, nb);
  hipLaunchKernelGGL(ll_one_point<T>, dim3(nb), dim3(kCellThreads), 0, s, pts, kind, n, last, part + nb);
  GPE_HIPCHK(hipGetLastError());
  std::vector<double> h(2 * (size_t)nb);
  GPE_HIPCHK(hipMemcpyAsync(h.data(), part, sizeof(double) * h.size(), hipMemcpyDeviceToHost, s));
  GPE_HIPCHK(hipStreamSynchronize(s));
  for (double v : h) *sum += v;
  return GPE_OK;
}

template <typename S, typename T>
int zero_points(DiagWork &w, const void *psi, const void *lo, const ZrGrid &g, int which, const long long *list,
                long long n, ZeroPoint *out, long long cap, long long *count, hipStream_t s) {
  const int nb = blocks(n, kCellThreads), nsec = which == 0 ? 6 : 3;
  long long *counts;
  if (int rc = room(w, DiagWork::kCounts, (size_t)nsec * nb + 1, &counts)) return rc;
  hipLaunchKernelGGL((zr_count<S, T>), dim3(nb), dim3(kCellThreads), 0, s, (const S *)psi, (const S *)lo, g, which, list,
                     n, counts);
  hipLaunchKernelGGL(prefix_sums, dim3(1), dim3(kScanThreads), 0, s, counts, nsec * nb);
  GPE_HIPCHK(hipGetLastError());
  if (int rc = read_back(counts + (size_t)nsec * nb, count, s)) return rc;
  const long long take = std::min(cap, *count);
  if (take == 0) return GPE_OK;
  ZeroPoint *pts;
  if (int rc = room(w, DiagWork::kOut, (size_t)*count, &pts)) return rc;
  hipLaunchKernelGGL((zr_write<S, T>), dim3(nb), dim3(kCellThreads), 0, s, (const S *)psi, (const S *)lo, g, which, list,
                     n, counts, pts);
  GPE_HIPCHK(hipGetLastError());
  GPE_HIPCHK(hipStreamSynchronize(s));
  static_assert(sizeof(ZeroPoint) % 8 == 0, "points are moved as 8-byte words");
  return words_download(8, (size_t)take * (sizeof(ZeroPoint) / 8), pts, nullptr, out, GPE_HOST_C64);
}

}  // namespace

int diag_linelength(DiagWork &w, int prec, const void *psi, const void *lo, int nx, int ny, int nz, double dx,
                    double *length, hipStream_t s) {
  long long *list, n = 0;
  if (int rc = list_of_cells(w, prec, psi, nx, ny, nz, 0, &list, &n, s)) return rc;
  double sum = 0.0;
  if (n) {
    const int rc = prec == GPE_FP64   ? linelength_sum<double, double>(w, psi, nullptr, nx, ny, list, n, &sum, s)
                   : prec == GPE_FP32 ? linelength_sum<float, float>(w, psi, nullptr, nx, ny, list, n, &sum, s)
                                      : linelength_sum<float, double>(w, psi, lo, nx, ny, list, n, &sum, s);
    if (rc) return rc;
  }
  *length = prec == GPE_FP32 ? (double)((float)sum * (float)dx) : sum * dx;
  return GPE_OK;
}

int diag_zeros(DiagWork &w, int prec, const void *psi, const void *lo, int nx, int ny, int nz, const double *xyzl,
               const double *dxyz, int which, ZeroPoint *out, long long cap, long long *count, hipStream_t s) {
  *count = 0;
  long long *list, n = 0;
  if (int rc = list_of_cells(w, prec, psi, nx, ny, nz, which, &list, &n, s)) return rc;
  if (!n) return GPE_OK;
  const ZrGrid g{xyzl[0], xyzl[1], xyzl[2], dxyz[0], dxyz[1], dxyz[2], nx, ny};
  return prec == GPE_FP64   ? zero_points<double, double>(w, psi, nullptr, g, which, list, n, out, cap, count, s)
         : prec == GPE_FP32 ? zero_points<float, float>(w, psi, nullptr, g, which, list, n, out, cap, count, s)
                            : zero_points<float, double>(w, psi, lo, g, which, list, n, out, cap, count, s);
}

}  // namespace gpe
