// launch.h -- host-side view of the kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "stage_args.h"

namespace gpe {

// Tile shape of a stage kernel: NW waves, P rows per wave, so TY = NW*P rows
// of 64 x-sites.  Each variant is compiled into its own translation unit
// (gpe_stage.hip with -DGPE_VID) and the host picks one per stage kind
// (defaults below, or the autotuner's choice).
struct Tile {
  int nw, p;
};
constexpr int N_TILE_VARIANTS = 5;
constexpr Tile kTiles[N_TILE_VARIANTS] = {{4, 4}, {8, 2}, {16, 1}, {4, 2}, {8, 1}};

// FP64 Cash-Karp stages do not run the (4,4) and (8,2) tiles.  An earlier
// build gave wrong 4th-order FP64 RKF45 fields with exactly these two
// shapes (every other shape, scheme and precision matched the oracle), and
// no fault in the source was found.  They are the two shapes whose FP64
// 4th-order last-stage instantiation is allocated the full 256 VGPRs and
// still spills to scratch (484 and 292 B per lane in the single-simulation
// kernel, 624 and 372 B batched); (16,1) spills too, but under a 128-VGPR
// budget, and passes.  (8,1) needs no scratch in any stage; the automatic
// march takes it for the last stage, but (16,1) for two of the others in 4th
// order (march_vid).
constexpr int kVidF64Ck = 4;
constexpr bool variant_allowed(bool fp64, int kind, int vid) {
  return vid >= 0 && vid < N_TILE_VARIANTS && !(fp64 && kind >= K_CK_1 && kind <= K_CK_6 && vid <= 1);
}

// The (8,2) tile: the automatic march of the kinds that nothing else serves
// better.
constexpr int kDefaultVid = 1;

// Tiling of one stage sweep over an nx x ny x nz grid with tile variant vid
// and z-chunk zc (0: automatic): sets A.ntx, A.nty, A.zc, A.nzc and
// A.nblocks and returns the number of workgroups.  Automatic chunks give
// enough workgroups to fill 256 CUs several times over, but stay long
// enough that re-reading 2R planes per chunk stays small: at least 32
// planes unless that leaves fewer than 1024 workgroups (small grids, where
// the z march's latency, not its traffic, sets the time).
inline int stage_grid(int nx, int ny, int nz, int vid, int zc, StageArgs &A) {
  const Tile t = kTiles[vid];
  const int TY = t.nw * t.p;
  A.ntx = (nx + 63) / 64;
  A.nty = (ny + TY - 1) / TY;
  const int tiles2d = A.ntx * A.nty;
  if (zc <= 0) {
    int nzc = (2048 + tiles2d - 1) / tiles2d;
    zc = (nz + nzc - 1) / nzc;
    if (zc < 32 && tiles2d * ((nz + 31) / 32) >= 1024) zc = 32;
  }
  if (zc < 8) zc = 8;
  if (zc > nz) zc = nz;
  A.zc = zc;
  A.nzc = (nz + zc - 1) / zc;
  A.nblocks = tiles2d * A.nzc;
  return A.nblocks;
}

// Fields a stage kind reads per site of its sweep.
constexpr int stage_reads(int kind) {
  return kind == K_RK2_2 || kind == K_RK4_2 || kind == K_RK4_3 ? 2
         : kind == K_RK4_4                                     ? 3
         : kind >= K_CK_1 && kind <= K_CK_6                    ? kind - K_CK_1 + 1
                                                               : 1;
}

// A single simulation's sweep: bricks of some planes, or (planes 0) the march
// with a tile variant and z-chunk.
struct Sweep {
  int planes, vid, zc;
};

// The z-chunk of a kind in its automatic configuration, in which every kind
// starts; one that was read (-planes for bricks) sets it too.
constexpr int kAutoChunk = -1;
constexpr bool automatic_chunk(int zc) { return zc == kAutoChunk || zc == -2 || zc == -4; }

// Brick sweeps (brick.hpp): kBrickWaves rows and 2 or 4 planes per workgroup.
constexpr int kBrickWaves = 8;
inline int brick_grid(int nx, int ny, int nz, int planes, StageArgs &A) {
  A.ntx = (nx + 63) / 64;
  A.nty = (ny + kBrickWaves - 1) / kBrickWaves;
  A.zc = planes;
  A.nzc = (nz + planes - 1) / planes;
  A.nblocks = A.ntx * A.nty * A.nzc;
  return A.nblocks;
}

// Planes per brick with which a kind in its automatic configuration sweeps a
// grid, or 0 for the z march.  A brick reads
// each of its fields about three times (2 planes, 4th order) where the march
// reads them once, so it pays while the march's chain of planes takes longer
// than that: up to some number of field values per sweep, more in FP32, whose
// values are half the size.  Measured (MI355X, us per sweep, march / 2 planes):
//   FP64 4th order, ck_1: 48^3 22 / 8, 64^3 23 / 12, 128^3 47 / 35
//   ck_3: 64^3 19 / 10, 96^3 35 / 24, 128^3 42 / 43
//   ck_6: 64^3 32 / 15, 96^3 59 / 60, 128^3 72 / 129
//   FP32C ck_6: 64^3 32 / 12, 96^3 35 / 29, 128^3 43 / 47; ck_3: 128^3 20.5 / 20.6
// The FP64 kinds that read one field, or two on all but the largest grids,
// take bricks of 4 planes beyond that: at 256^3 rk4_1 185 -> 135, rk4_2
// 256 -> 231 (2nd order), ck_1 323 -> 206, ck_2 256 -> 226; at 384^3 rk4_1
// 615 -> 425, but rk4_2 782 -> 866.
inline int brick_planes(bool fp64, int kind, int radius, int nx, int ny, int nz) {
  const long long n = (long long)nx * ny * nz;
  const int reads = stage_reads(kind);
  StageArgs A;
  // 4th order in FP32, one field: the march with (4,2) tiles is ahead earlier
  // (ck_1 at 2.4 M sites 24 -> 21, 225^3 45 -> 35)
  const long long most = fp64 ? 5000000 : reads == 1 && radius == 2 && kind != K_ENERGY ? 2000000 : 8000000;
  if (n * reads <= most) return brick_grid(nx, ny, nz, 2, A) <= 65536 ? 2 : 0;
  if (!fp64 || kind == K_ENERGY || reads > 2) return 0;
  if (kind == K_CK_1) return 4;
  // as above for 4th-order kinds that the march with (4,2) tiles serves well:
  // rk4_1 at 192^3 81 -> 73, 320^3 322 -> 264, rk4_3 103 -> 85 and 445 -> 338,
  // ck_2 101 -> 86 and 547 -> 350
  const bool early = radius == 2 && kind != K_RK4_2 && kind != K_RK2_2;
  if (reads == 1) return early && n > 6000000 ? 0 : 4;
  // rk4_2's march wants whole tiles (256^3 270 -> 219, but 257 x 255 x 258 291 -> 329)
  const bool whole = radius == 2 && kind == K_RK4_2 && nx % 64 == 0;
  return n <= (early || whole ? 6000000 : 20000000) ? 4 : 0;
}

// Tile variant of the z march where a kind's configuration is automatic: the
// fastest of the five over grids of 0.5 .. 134 M sites, each with chunks of
// march_chunk.  FP64 kinds are bound by instructions and by the latency of a
// plane, so the variants with the fewest registers per lane and more
// workgroups win ((4,2) against (8,2), 4th order: 256^3 rk4_4 283 -> 229 us,
// 512^3 rk4_3 1590 -> 1300, ck_2 against (8,1) 2060 -> 1340; (16,1) for ck_3
// and ck_4, 256^3 319 -> 261, though these two spill 36 and 84 B a lane in 4th
// order: spilling is what the shapes that variant_allowed refuses had in
// common, so test_march_gpu.py holds the automatic fields to (8,1)'s bit for
// bit on either side of every line); the FP32 ones keep (8,2) but for those that
// store little or read one field (rk4_1 at 256^3 82 -> 65, rk4_2 157 -> 118).
inline int march_vid(bool fp64, int kind, int radius, long long n) {
  const bool r2 = radius == 2;
  if (kind == K_ENERGY) return kDefaultVid;
  if (!fp64) {
    if (kind == K_EULER) return 1;
    if (stage_reads(kind) == 1) return n < 50000000 ? 3 : 0;
    if (kind == K_RK4_2 && r2) return n < 5000000 ? 3 : 0;
    return kind == K_RK2_2 && r2 ? 4 : 1;
  }
  switch (kind) {
    case K_RK4_2: return r2 ? 0 : 3;
    case K_RK2_2: return r2 ? 1 : 3;
    case K_CK_3:
    case K_CK_4: return r2 ? 2 : 3;
    case K_CK_5: return r2 ? 4 : 3;
    case K_CK_6: return 4;
    default: return 3;
  }
}

// Planes per chunk of the march, automatic: a CU holds `resident` of the
// kind's workgroups, so a sweep takes ceil(workgroups / (CUs x resident))
// rounds of zc + 2R planes each, and the chunk with the smallest product wins:
// long enough that few planes are read twice, and with no round that is nearly
// empty (FP64 ck_6 at 192^3: chunks of 8, 16, 32, 64 planes take 7, 4, 2, 1
// rounds and 250, 243, 223, 208 us).  Against the best of chunks of 8, 16, 32
// and 64 in the same tile (261 kinds: seven grids of 2 .. 134 M sites, FP64 and
// FP32C, both orders, every scheme) it takes 0.99 times as long in the mean, 1.00
// in the median, 0.77 .. 1.14 at the ends and at most 1.045 in nine of ten; the
// worst are FP64 kinds in the small (4,2) tile (256^3 rk4_1 159 us against 139
// in chunks of 32).
constexpr int kCUs = 256;
inline int march_chunk(int nx, int ny, int nz, int vid, int radius, int resident) {
  const Tile t = kTiles[vid];
  const long long tiles2d = (long long)((nx + 63) / 64) * ((ny + t.nw * t.p - 1) / (t.nw * t.p));
  const long long room = (long long)kCUs * (resident > 0 ? resident : 1);
  int best = nz;
  long long least = 0;
  for (int n = 1; n == 1 || (nz + n - 1) / n >= 8; ++n) {
    const int zc = (nz + n - 1) / n;
    const long long groups = tiles2d * ((nz + zc - 1) / zc);
    const long long cost = (groups + room - 1) / room * (zc + 2 * radius);
    if (n == 1 || cost < least) {
      least = cost;
      best = zc;
    }
  }
  return best;
}
hipError_t launch_brick_f64(int planes, int kind, int radius, bool comp, const StageArgs &A, hipStream_t s);
hipError_t launch_brick_f32(int planes, int kind, int radius, bool comp, const StageArgs &A, hipStream_t s);
inline hipError_t launch_brick(int prec_bytes, int planes, int kind, int radius, bool comp, const StageArgs &A,
                               hipStream_t s) {
  return prec_bytes == 16 ? launch_brick_f64(planes, kind, radius, comp, A, s)
                          : launch_brick_f32(planes, kind, radius, comp, A, s);
}

// Launch stage kernel `kind` (radius 1 or 2) over A.nblocks workgroups with
// tile variant `vid`.  comp selects the compensated FP32 form.  With resident,
// nothing is launched: how many of its workgroups a CU holds at once.
hipError_t launch_stage(int prec_bytes, int vid, int kind, int radius, bool comp, const StageArgs &A,
                        hipStream_t s, int *resident = nullptr);

// Fused stage pairs (fused.hpp): pair kinds P_RK4_12 .. P_CK_56 and their
// tile variants.
constexpr int N_PAIR_KINDS = 5;
constexpr int N_PAIR_VARIANTS = 3;
// waves, rows per wave, planes of prefetch
struct PairTile {
  int nw, p, d;
};
constexpr PairTile kPairTiles[N_PAIR_VARIANTS] = {{8, 2, 2}, {16, 1, 2}, {16, 1, 4}};
// FP64 (the parity path) always runs the stages one by one: its fused
// kernels would spill ~1 KB per lane to scratch, gain nothing, and a
// batched 4th-order FP64 build gave results different from the
// stage-by-stage sweeps for reasons not found in the source.
constexpr int N_PAIR_VARIANTS_F64 = 0;
// A: stage A's descriptor, B: stage B's (B carries the grid: ntx/nty over
// the (64-2R) x (TY-2R) interiors, zc, nblocks).
hipError_t launch_pair(int prec_bytes, int vid, int pair, int radius, bool comp, const StageArgs &A,
                       const StageArgs &B, hipStream_t s);

// Batched launch over a work table (see stage_kernel_batched).
struct BatchLaunch {
  const StageArgs *insts;  // this kind's StageArgs of every instance slot
  const WorkItem *work;
  int nwork;
  const int *active;
  double *pn, *pe;  // partial sums of the final stage (null otherwise)
  int grid;
};
hipError_t launch_stage_batched(int prec_bytes, int vid, int kind, int radius, bool comp, const BatchLaunch &B,
                                hipStream_t s);
// B.grid: a multiple of 8
hipError_t launch_brick_batched_f64(int planes, int kind, int radius, bool comp, const BatchLaunch &B, hipStream_t s);
hipError_t launch_brick_batched_f32(int planes, int kind, int radius, bool comp, const BatchLaunch &B, hipStream_t s);
inline hipError_t launch_brick_batched(int prec_bytes, int planes, int kind, int radius, bool comp,
                                       const BatchLaunch &B, hipStream_t s) {
  return prec_bytes == 16 ? launch_brick_batched_f64(planes, kind, radius, comp, B, s)
                          : launch_brick_batched_f32(planes, kind, radius, comp, B, s);
}
struct PairBatchLaunch {
  const StageArgs *instA, *instB;  // stage A's / B's StageArgs of every instance slot
  const WorkItem *work;
  int nwork;
  const int *active;
  double *pn, *pe;
  int grid;
};
hipError_t launch_pair_batched(int prec_bytes, int vid, int pair, int radius, bool comp, const PairBatchLaunch &L,
                               hipStream_t s);

// Per-instance step control after the final stage of a batched iteration.
hipError_t launch_batch_control(InstCtl *ctl, StageArgs *args, int cap, int *active, const int *range,
                                const double *pn, const double *pe, hipStream_t s);

// Reduce per-block partials to out[0..2], device memory or (ticket != 0) mapped
// host memory (see reduce_partials); the norms of several steps at once.
hipError_t launch_reduce(const double *pn, const double *pe, const double *pen, int n, double scale_norm,
                         double eps, double scale_energy, double *out, double *hist, double ticket, hipStream_t s);
hipError_t launch_reduce_norms(const double *pn, size_t stride, int n, int steps, double scale_norm, double *hist,
                               hipStream_t s);

// Pointwise helpers over a whole field.  Partials: one double per block.
constexpr int PW_BLOCKS = 1024;
hipError_t launch_norm_f64(const void *psi, int nx, int ny, int nz, int weighted, double w1, double w2,
                           double w3, double *part, hipStream_t s);
// Block partials (PW_BLOCKS each) of sum |psi|^2, |psi|^4, V |psi|^2 (prec 0: FP64 storage).
hipError_t launch_moments(int prec, const void *psi, const void *lo, const StageArgs &A, double *p2, double *p4,
                          double *pv, hipStream_t s);
hipError_t launch_norm_f32(const void *psi, const void *lo, int nx, int ny, int nz, int weighted, double w1,
                           double w2, double w3, double *part, hipStream_t s);
hipError_t launch_renorm_f64(void *psi, size_t n, double a, DivC b, hipStream_t s);
hipError_t launch_renorm_f32(void *psi, void *lo, size_t n, double a, double b, hipStream_t s);

// imprint_vortex_line over the whole field (pointwise.hpp); prec as
// GPE_FP64 / GPE_FP32 / GPE_FP32C (lo = low word of the compensated form).
hipError_t launch_imprint(int prec, void *psi, void *lo, const LineArgs &L, hipStream_t s);

// HBM read / write / copy bandwidth (GB/s) of float4 arrays of `bytes`.
hipError_t probe_bandwidth(size_t bytes, int reps, double *gbs);

// per-variant entry points (one definition per translation unit)
#define GPE_DECL_VARIANT(P, V) \
  hipError_t launch_stage_##P##_v##V(int kind, int radius, bool comp, const StageArgs &A, hipStream_t s, \
                                     int *resident);
GPE_DECL_VARIANT(f64, 0)
GPE_DECL_VARIANT(f64, 1)
GPE_DECL_VARIANT(f64, 2)
GPE_DECL_VARIANT(f64, 3)
GPE_DECL_VARIANT(f64, 4)
GPE_DECL_VARIANT(f32, 0)
GPE_DECL_VARIANT(f32, 1)
GPE_DECL_VARIANT(f32, 2)
GPE_DECL_VARIANT(f32, 3)
GPE_DECL_VARIANT(f32, 4)
#undef GPE_DECL_VARIANT
#define GPE_DECL_BVARIANT(P, V)                                                                            \
  hipError_t launch_batched_##P##_v##V(int kind, int radius, bool comp, const BatchLaunch &B, hipStream_t s);
GPE_DECL_BVARIANT(f64, 0)
GPE_DECL_BVARIANT(f64, 1)
GPE_DECL_BVARIANT(f64, 2)
GPE_DECL_BVARIANT(f64, 3)
GPE_DECL_BVARIANT(f64, 4)
GPE_DECL_BVARIANT(f32, 0)
GPE_DECL_BVARIANT(f32, 1)
GPE_DECL_BVARIANT(f32, 2)
GPE_DECL_BVARIANT(f32, 3)
GPE_DECL_BVARIANT(f32, 4)
#undef GPE_DECL_BVARIANT
#define GPE_DECL_PVARIANT(P, V)                                                                              \
  hipError_t launch_pair_##P##_v##V(int pair, int radius, bool comp, const StageArgs &A, const StageArgs &B,  \
                                    hipStream_t s);                                                         \
  hipError_t launch_pair_batched_##P##_v##V(int pair, int radius, bool comp, const PairBatchLaunch &L,       \
                                            hipStream_t s);
GPE_DECL_PVARIANT(f32, 0)
GPE_DECL_PVARIANT(f32, 1)
GPE_DECL_PVARIANT(f32, 2)
#undef GPE_DECL_PVARIANT

}  // namespace gpe
