// fv:: operators and CrsEquation algebra on the device.
//
// A phase_hip_equation is FiniteVolumeEquation<T> / CrsEquation
// (src/Math/CrsEquation.cpp, src/2D/Unstructured/FiniteVolume/Equation/
// FiniteVolumeEquation.tpp) held in HBM: rank = ncomp * nCells rows in the
// IndexMap block layout (row = comp * nCells + cell, IndexMap.cpp:31-36), each
// row a list of up to `stride` (column, value) pairs in first-touch order plus
// the stored rhs (A x + rhs = 0).
//
// Operators run one thread per cell and replay the reference's per-cell face
// loop, so every row has the reference's column order and every sum its
// summation order (bit-identical with -ffp-contract=off).  A row is built in
// LDS with CrsEquation::addCoeff's first-touch rule (CrsEquation.cpp:
// 113-131) and the block's rows leave in one contiguous run.  operator+= / -= (CrsEquation.cpp:185-275) rebuilds each row the
// same way: the left rows' non-zero entries, then the right rows' non-zero
// entries accumulated into a matching column or appended.
//
// Field kernels: src::div / src::src (Source.cpp:5-25, 77-95), the face and
// cell gradients (ScalarGradient.cpp:34-74) and face interpolation with the
// boundary rules (FiniteVolumeField.tpp:129-182, VectorFiniteVolumeField.cpp:
// 140-160).  Vector fields are interleaved (x0, y0, x1, y1, ...).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "equation.h"
#include "mesh.h"
#include "solver.h"
#include "solver_kernels.h"

using namespace phase;

namespace {

constexpr int kRowCap = 16;  // most slots of a row: diagonal + 14 neighbours + one cross-component entry

struct MeshDev {
  int nCells;
  bool repeated;  // a cell meets a neighbour over more than one face
  const double *vol, *cc, *fc, *sf;
  const int *iptr, *iface, *inb, *bptr, *bface;  // iface, bface: with kFlip (mesh.h)
  const double *idot, *ims, *bdot, *bms;
};

MeshDev meshDev(const phase_hip_mesh *m) {
  return MeshDev{m->nCells, m->repeated, m->dVol.p, m->dCC.p, m->dFC.p, m->dSf.p, m->dIptr.p, m->dIfaceS.p,
                 m->dInb.p, m->dBptr.p, m->dBfaceS.p, m->dIDot.p, m->dIMs.p, m->dBDot.p, m->dBMs.p};
}

__device__ __forceinline__ Dv2 ld2(const double *a, int i) {
  const dv2_t v = *(const dv2_t *)(a + 2 * (size_t)i);
  return Dv2{v.x, v.y};
}
__device__ __forceinline__ void st2(double *a, int i, double x, double y) { *(dv2_t *)(a + 2 * (size_t)i) = dv2_t{x, y}; }

// The links [beg, end) in order, four at a time: load(q, k) issues link k's
// loads into slot q of the caller's arrays (the last ones again past the end),
// use(q, k) consumes them.  A cell has three or four links, so its loads are
// in flight together instead of one dependent round trip per link.
template <class Load, class Use>
__device__ __forceinline__ void forLinks(int beg, int end, Load &&load, Use &&use) {
  for (int k0 = beg; k0 < end; k0 += 4) {
#pragma unroll
    for (int q = 0; q < 4; ++q) load(q, min(k0 + q, end - 1));
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (k0 + q < end) use(q, k0 + q);
  }
}

// Rows under construction, one per thread of a block of kRowBlock, in LDS.
// CrsEquation::addCoeff semantics: the first touch of a column claims the next
// slot, later touches accumulate in call order.  The diagonal accumulates in a
// register.  A cell's neighbours are distinct, so a neighbour is its column's
// only touch; on meshes where they are not (`repeated`) the staged row is
// searched.  Rows in registers, indexed by the running count, went to scratch
// memory (1.2 KB a thread): at 1M quads, two components, the upwind divergence
// took 858 us, and each slot's store touched every line of the block's rows.
// (kEqDivGrad still keeps 96 B a lane there, its batched links' geometry: 120 us
// against 854 for the same mesh.)
constexpr int kRowBlock = 256;
inline int rowPitch(int stride) { return stride | 1; }  // odd: the threads' rows start in different banks
inline size_t rowLds(int stride) { return (size_t)kRowBlock * rowPitch(stride) * (sizeof(double) + sizeof(int)); }
extern __shared__ __align__(16) char rowStage[];

struct RowS {
  double *val;
  int *col;
  double diag;
  int c, n, pd, stride;
  bool over, repeated;
  __device__ RowS(int cell, int str, bool rep) {
    const int P = str | 1;
    val = (double *)rowStage + threadIdx.x * P;
    col = (int *)((double *)rowStage + kRowBlock * P) + threadIdx.x * P;
    diag = 0.;
    c = cell;
    n = 0;
    pd = -1;
    stride = str;
    over = false;
    repeated = rep;
  }
  __device__ __forceinline__ int claim() {
    if (n >= stride) {
      over = true;
      return -1;
    }
    return n++;
  }
  // column c
  __device__ __forceinline__ void addDiag(double v) {
    if (pd < 0) {
      pd = claim();
      diag = v;
    } else {
      diag += v;
    }
  }
  // a neighbour's column (or another column coded as storeRows takes it);
  // `search`: the row may hold it already
  __device__ __forceinline__ void add(int nb, double v, bool search = false) {
    if (repeated || search) {
      if (nb == c) return addDiag(v);
      for (int j = 0; j < n; ++j)
        if (j != pd && col[j] == nb) {
          val[j] += v;
          return;
        }
    }
    const int p = claim();
    if (p < 0) return;
    col[p] = nb;
    val[p] = v;
  }
  __device__ __forceinline__ void finish() {
    if (pd >= 0) {
      col[pd] = c;
      val[pd] = diag;
    }
    for (int j = n; j < stride; ++j) {
      col[j] = -1;
      val[j] = 0.;
    }
  }
};

// The block's staged rows (cells c0 and up) to component q's rows, in one
// contiguous run.  Staged columns: -1 empty, >= 0 a cell (column q N + cell),
// below -1 the column -2 - value itself.  A row with more columns than slots
// raises err bit 4 and is not written.  Called by every thread of the block.
__device__ __forceinline__ void storeRows(const RowS &r, int q, int N, int c0, int *cols, double *vals, int *cnt,
                                          int *err) {
  const int stride = r.stride, P = stride | 1;
  const int rows = min(kRowBlock, N - c0);
  const double *sv = (const double *)rowStage;
  const int *sc = (const int *)(sv + kRowBlock * P);
  const size_t base = ((size_t)q * N + c0) * stride;
  const bool mine = (int)threadIdx.x < rows;
  auto column = [&](int s) { return s >= 0 ? q * N + s : s == -1 ? -1 : -2 - s; };
  if (__syncthreads_or(mine && r.over)) {
    if (mine && r.over) atomicOr(err, 4);
    if (mine && !r.over)
      for (int j = 0; j < stride; ++j) {
        cols[base + (size_t)threadIdx.x * stride + j] = column(r.col[j]);
        vals[base + (size_t)threadIdx.x * stride + j] = r.val[j];
      }
  } else {
    // idx / stride: the product is at least 0.5 / 16 away from an integer
    const float inv = 1.f / (float)stride;
    for (int idx = threadIdx.x; idx < rows * stride; idx += kRowBlock) {
      const int row = (int)((idx + 0.5f) * inv), at = row * P + idx - row * stride;
      cols[base + idx] = column(sc[at]);
      vals[base + idx] = sv[at];
    }
  }
  if (mine && !r.over) cnt[(size_t)q * N + c0 + threadIdx.x] = r.n;
  __syncthreads();
}

// The operators: one cell per thread, the block's cells in step so that every
// thread reaches storeRows.  Bound by HBM: the links' indices and geometry, the
// face and cell fields once each (neighbouring cells share faces out of L2),
// and the rows written once.  NC: components (1, or 2 for Vector2D, whose rows
// differ in the column offset only except at SYMMETRY faces).

// fv::laplacian, all four forms (Laplacian.h:7-167) and the Vector2D theta
// forms with the SYMMETRY tangential term (Laplacian.cpp:5-120).  Same
// coefficient (gamma * dot(r, Sf)) / |r|^2 as the oracle; err bit 1 =
// unsupported boundary type, bit 2 = missing boundary/old-time input.
// 1M quads, two components: 77 us (430 us with rows in registers).
template <int NC>
__global__ __launch_bounds__(kRowBlock) void kEqLaplacian(MeshDev M, int variant, double gamma,
                                                          const double *__restrict__ gF,
                                                          const double *__restrict__ g0F, double theta,
                                                          const int *__restrict__ bc,
                                                          const double *__restrict__ phiF,
                                                          const double *__restrict__ phi0C,
                                                          const double *__restrict__ phi0F, int stride, int *cols,
                                                          double *vals, int *cnt, double *rhs, int *err) {
  const bool hasTheta = (variant == 0 || variant == 2);
  const bool field = (variant >= 2);
  const int N = M.nCells;
  for (int c0 = blockIdx.x * kRowBlock; c0 < N; c0 += gridDim.x * kRowBlock) {
    const int c = c0 + threadIdx.x;
    RowS row(c, stride, M.repeated);
    double src[NC] = {};
    // SYMMETRY, Vector2D: the components' diagonals part, with a cross entry each
    double diag1 = 0., cross[2] = {0., 0.};
    bool parted = false, hasCross[2] = {false, false};
    if (c < N) {
      double p0[NC];
      if (hasTheta && phi0C)
        for (int q = 0; q < NC; ++q) p0[q] = phi0C[NC * (size_t)c + q];
      int f[4], nb[4];
      double g[4], g0[4], dt[4], ms[4], pn[4][NC];
      forLinks(M.iptr[c], M.iptr[c + 1],
               [&](int q, int k) {
                 nb[q] = M.inb[k];
                 dt[q] = M.idot[k];
                 ms[q] = M.ims[k];
                 f[q] = field ? faceOf(M.iface[k]) : 0;
                 g[q] = field ? gF[f[q]] : gamma;
                 if (hasTheta) {
                   g0[q] = field ? g0F[f[q]] : 0.;
                   if (phi0C)
                     for (int i = 0; i < NC; ++i) pn[q][i] = phi0C[NC * (size_t)nb[q] + i];
                 }
               },
               [&](int q, int) {
                 const double coeff = g[q] * dt[q] / ms[q];
                 if (!hasTheta) {
                   if (!field) {  // Laplacian.h:57-58
                     row.add(nb[q], coeff);
                     row.addDiag(-coeff);
                   } else {  // Laplacian.h:141-142
                     row.addDiag(-coeff);
                     row.add(nb[q], coeff);
                   }
                   return;
                 }
                 if (!phi0C) {
                   atomicOr(err, 2);
                   return;
                 }
                 const double coeff0 = field ? g0[q] * dt[q] / ms[q] : coeff;
                 if (!field) {  // Laplacian.h:17-21
                   row.add(nb[q], theta * coeff);
                   row.addDiag(theta * -coeff);
                 } else {  // Laplacian.h:99-101, Laplacian.cpp:75-77
                   row.addDiag(theta * -coeff);
                   row.add(nb[q], theta * coeff);
                 }
                 for (int i = 0; i < NC; ++i) src[i] += (1. - theta) * coeff0 * (pn[q][i] - p0[i]);
               });
      for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
        const int fb = faceOf(M.bface[k]);
        const int bt = bc ? bc[fb] : PHASE_HIP_BC_NORMAL_GRADIENT;
        const double gb = field ? gF[fb] : gamma;
        const double coeff = gb * M.bdot[k] / M.bms[k];
        if (bt == PHASE_HIP_BC_FIXED) {
          if (!phiF || (hasTheta && (!phi0F || !phi0C))) {
            atomicOr(err, 2);
            continue;
          }
          const double a = hasTheta ? theta * -coeff : -coeff;  // Laplacian.h:31-36, 69-72
          row.addDiag(a);
          if (parted) diag1 += a;
          if (!hasTheta) {
            for (int q = 0; q < NC; ++q) src[q] += coeff * phiF[NC * (size_t)fb + q];
          } else {
            const double coeff0 = field ? g0F[fb] * M.bdot[k] / M.bms[k] : coeff;
            for (int q = 0; q < NC; ++q) src[q] += theta * coeff * phiF[NC * (size_t)fb + q];
            for (int q = 0; q < NC; ++q) src[q] += (1. - theta) * coeff0 * (phi0F[NC * (size_t)fb + q] - p0[q]);
          }
        } else if (bt == PHASE_HIP_BC_NORMAL_GRADIENT) {
        } else if (bt == PHASE_HIP_BC_SYMMETRY) {
          if (NC == 2 && hasTheta) {  // Laplacian.cpp:36-43
            if (!phi0C) {
              atomicOr(err, 2);
              continue;
            }
            const Dv2 sfo = outwardOf(M.bface[k], M.sf);
            const Dv2 tv{-sfo.y, sfo.x};  // Vector2D::tangentVec, Vector2D.h:28
            const double tm = sqrt(tv.x * tv.x + tv.y * tv.y);
            const Dv2 tw{tv.x / tm, tv.y / tm};
            const double coeff0 = field ? g0F[fb] * M.bdot[k] / M.bms[k] : coeff;
            row.addDiag(theta * -coeff);
            diag1 = parted ? diag1 + theta * -coeff : row.diag;
            parted = true;
            const double tc = theta * coeff;
            // add(cell, cell, Tensor2D), VectorFiniteVolumeEquation.cpp:48-66
            const double xx = tc * (tw.x * tw.x), xy = tc * (tw.x * tw.y), yx = tc * (tw.y * tw.x),
                         yy = tc * (tw.y * tw.y);
            row.addDiag(xx);
            diag1 += yy;
            if (xy != 0.) {
              cross[0] = hasCross[0] ? cross[0] + xy : xy;
              hasCross[0] = true;
            }
            if (yx != 0.) {
              cross[1] = hasCross[1] ? cross[1] + yx : yx;
              hasCross[1] = true;
            }
            const double d = p0[0] * tw.x + p0[NC - 1] * tw.y;
            const double w = (1. - theta) * coeff0;
            src[0] += w * (tw.x * d - p0[0]);
            src[NC - 1] += w * (tw.y * d - p0[NC - 1]);
          }
        } else {
          atomicOr(err, 1);
        }
      }
    }
    // the cross entries are the last columns claimed: every other column of the
    // row is an interior link's, or the diagonal, which the same face touches
    // before them
    const int base = row.n;
    const bool over = row.over;
    if (c < N) {
      if (hasCross[0]) row.add(-2 - (N + c), cross[0]);
      row.finish();
      for (int q = 0; q < NC; ++q) rhs[(size_t)q * N + c] = src[q];
    }
    storeRows(row, 0, N, c0, cols, vals, cnt, err);
    if (NC == 2) {
      if (parted) {
        row.n = base;
        row.over = over;
        row.diag = diag1;
        if (hasCross[1]) row.add(-2 - c, cross[1]);
        row.finish();
      }
      storeRows(row, 1, N, c0, cols, vals, cnt, err);
    }
  }
}

// fv::ddt(field, timeStep), TimeDerivative.h:37-48
template <int NC>
__global__ __launch_bounds__(kRowBlock) void kEqDdt(MeshDev M, double dt, const double *__restrict__ phi0C, int stride,
                                                    int *cols, double *vals, int *cnt, double *rhs, int *err) {
  const int N = M.nCells;
  for (int c0 = blockIdx.x * kRowBlock; c0 < N; c0 += gridDim.x * kRowBlock) {
    const int c = c0 + threadIdx.x;
    RowS row(c, stride, false);
    if (c < N) {
      const double v = M.vol[c];
      row.addDiag(v / dt);
      row.finish();
      for (int q = 0; q < NC; ++q) rhs[(size_t)q * N + c] = -v * phi0C[NC * (size_t)c + q] / dt;
    }
    for (int q = 0; q < NC; ++q) storeRows(row, q, N, c0, cols, vals, cnt, err);
  }
}

// fv::ddt with a density: scalar rho (TimeDerivative.h:7-19) or a field rho with
// rho0 for the source (:21-35); mask (optional) keeps the rows of a cell
// group only (:50-62), the others stay empty
template <int NC>
__global__ __launch_bounds__(kRowBlock) void kEqDdtRho(MeshDev M, double dt, double rho,
                                                       const double *__restrict__ rhoC,
                                                       const double *__restrict__ rho0C,
                                                       const double *__restrict__ phi0C, const int *__restrict__ mask,
                                                       int stride, int *cols, double *vals, int *cnt, double *rhs,
                                                       int *err) {
  const int N = M.nCells;
  for (int c0 = blockIdx.x * kRowBlock; c0 < N; c0 += gridDim.x * kRowBlock) {
    const int c = c0 + threadIdx.x;
    RowS row(c, stride, false);
    if (c < N) {
      const bool in = !mask || mask[c];
      const double v = M.vol[c];
      if (in) row.addDiag(rhoC ? rhoC[c] * v / dt : rho * v / dt);
      row.finish();
      const double r0 = !in ? 0. : rhoC ? -rho0C[c] * v : -rho * v;
      for (int q = 0; q < NC; ++q) rhs[(size_t)q * N + c] = in ? r0 * phi0C[NC * (size_t)c + q] / dt : 0.;
    }
    for (int q = 0; q < NC; ++q) storeRows(row, q, N, c0, cols, vals, cnt, err);
  }
}

__device__ __forceinline__ double upMax(double a) { return a < 0. ? 0. : a; }  // std::max(a, 0.)
__device__ __forceinline__ double upMin(double a) { return 0. < a ? 0. : a; }  // std::min(a, 0.)

// fv::div(u, phi, theta), first-order upwind, Divergence.h:7-53.
// 1M quads, two components: 79 us (858 us with rows in registers).
template <int NC>
__global__ __launch_bounds__(kRowBlock) void kEqDiv(MeshDev M, const double *__restrict__ uF, const double *__restrict__ u0F,
                                                    double theta, const int *__restrict__ bc, const double *__restrict__ phiF,
                                                    const double *__restrict__ phi0C, const double *__restrict__ phi0F, int stride,
                                                    int *cols, double *vals, int *cnt, double *rhs, int *err) {
  const int N = M.nCells;
  for (int c0 = blockIdx.x * kRowBlock; c0 < N; c0 += gridDim.x * kRowBlock) {
    const int c = c0 + threadIdx.x;
    RowS row(c, stride, M.repeated);
    if (c < N) {
      double src[NC] = {};
      double p0[NC], pn[4][NC];
      for (int q = 0; q < NC; ++q) p0[q] = phi0C[NC * (size_t)c + q];
      int nb[4];
      Dv2 s[4], u[4], u0[4];
      forLinks(M.iptr[c], M.iptr[c + 1],
               [&](int q, int k) {
                 const int link = M.iface[k], f = faceOf(link);
                 nb[q] = M.inb[k];
                 s[q] = outwardOf(link, M.sf);
                 u[q] = ld2(uF, f);
                 u0[q] = ld2(u0F, f);
                 for (int i = 0; i < NC; ++i) pn[q][i] = phi0C[NC * (size_t)nb[q] + i];
               },
               [&](int q, int) {
                 const double flux = u[q].x * s[q].x + u[q].y * s[q].y;
                 const double flux0 = u0[q].x * s[q].x + u0[q].y * s[q].y;
                 row.addDiag(theta * upMax(flux));
                 row.add(nb[q], theta * upMin(flux));
                 for (int i = 0; i < NC; ++i) src[i] += (1. - theta) * upMax(flux0) * p0[i];
                 for (int i = 0; i < NC; ++i) src[i] += (1. - theta) * upMin(flux0) * pn[q][i];
               });
      for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
        const int link = M.bface[k], f = faceOf(link);
        const Dv2 s = outwardOf(link, M.sf);
        const double flux = uF[2 * f] * s.x + uF[2 * f + 1] * s.y;
        const double flux0 = u0F[2 * f] * s.x + u0F[2 * f + 1] * s.y;
        const int bt = bc ? bc[f] : PHASE_HIP_BC_NORMAL_GRADIENT;
        if (bt == PHASE_HIP_BC_FIXED) {
          if (!phiF || !phi0F) {
            atomicOr(err, 2);
            continue;
          }
          for (int q = 0; q < NC; ++q) src[q] += theta * flux * phiF[NC * (size_t)f + q];
          for (int q = 0; q < NC; ++q) src[q] += (1. - theta) * flux0 * phi0F[NC * (size_t)f + q];
        } else if (bt == PHASE_HIP_BC_NORMAL_GRADIENT) {
          row.addDiag(theta * flux);
          for (int q = 0; q < NC; ++q) src[q] += (1. - theta) * flux0 * p0[q];
        } else if (bt == PHASE_HIP_BC_SYMMETRY) {
        } else {
          atomicOr(err, 1);
        }
      }
      row.finish();
      for (int q = 0; q < NC; ++q) rhs[(size_t)q * N + c] = src[q];
    }
    for (int q = 0; q < NC; ++q) storeRows(row, q, N, c0, cols, vals, cnt, err);
  }
}

// fv::divc(u, phi, theta), central, Divergence.h:55-103 (boundary flux0 from u,
// as the reference computes it)
template <int NC>
__global__ __launch_bounds__(kRowBlock) void kEqDivc(MeshDev M, const double *__restrict__ uF, const double *__restrict__ u0F,
                                                     double theta, const int *__restrict__ bc, const double *__restrict__ phiF,
                                                     const double *__restrict__ phi0C, const double *__restrict__ phi0F, int stride,
                                                     int *cols, double *vals, int *cnt, double *rhs, int *err) {
  const int N = M.nCells;
  for (int c0 = blockIdx.x * kRowBlock; c0 < N; c0 += gridDim.x * kRowBlock) {
    const int c = c0 + threadIdx.x;
    RowS row(c, stride, M.repeated);
    if (c < N) {
      double src[NC] = {};
      const Dv2 pc = ld2(M.cc, c);
      double p0[NC], pn[4][NC];
      for (int q = 0; q < NC; ++q) p0[q] = phi0C[NC * (size_t)c + q];
      int nb[4];
      Dv2 s[4], u[4], u0[4], fc[4], cn[4];
      forLinks(M.iptr[c], M.iptr[c + 1],
               [&](int q, int k) {
                 const int link = M.iface[k], f = faceOf(link);
                 nb[q] = M.inb[k];
                 s[q] = outwardOf(link, M.sf);
                 u[q] = ld2(uF, f);
                 u0[q] = ld2(u0F, f);
                 fc[q] = ld2(M.fc, f);
                 cn[q] = ld2(M.cc, nb[q]);
                 for (int i = 0; i < NC; ++i) pn[q][i] = phi0C[NC * (size_t)nb[q] + i];
               },
               [&](int q, int) {
                 const double flux = theta * (u[q].x * s[q].x + u[q].y * s[q].y);
                 const double flux0 = (1. - theta) * (u0[q].x * s[q].x + u0[q].y * s[q].y);
                 const double ax = fc[q].x - pc.x, ay = fc[q].y - pc.y, bx = fc[q].x - cn[q].x, by = fc[q].y - cn[q].y;
                 const double lc = sqrt(ax * ax + ay * ay), ln = sqrt(bx * bx + by * by);
                 const double g = ln / (lc + ln);
                 row.addDiag(g * flux);
                 row.add(nb[q], (1. - g) * flux);
                 for (int i = 0; i < NC; ++i) src[i] += flux0 * (g * p0[i] + (1. - g) * pn[q][i]);
               });
      for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
        const int link = M.bface[k], f = faceOf(link);
        const Dv2 s = outwardOf(link, M.sf);
        const double fl = uF[2 * f] * s.x + uF[2 * f + 1] * s.y;
        const double flux = theta * fl, flux0 = (1. - theta) * fl;
        const int bt = bc ? bc[f] : PHASE_HIP_BC_NORMAL_GRADIENT;
        if (bt == PHASE_HIP_BC_FIXED) {
          if (!phiF || !phi0F) {
            atomicOr(err, 2);
            continue;
          }
          for (int q = 0; q < NC; ++q) src[q] += flux * phiF[NC * (size_t)f + q];
          for (int q = 0; q < NC; ++q) src[q] += flux0 * phi0F[NC * (size_t)f + q];
        } else if (bt == PHASE_HIP_BC_NORMAL_GRADIENT) {
          row.addDiag(flux);
          for (int q = 0; q < NC; ++q) src[q] += flux0 * p0[q];
        } else if (bt == PHASE_HIP_BC_SYMMETRY) {
        } else {
          atomicOr(err, 1);
        }
      }
      row.finish();
      for (int q = 0; q < NC; ++q) rhs[(size_t)q * N + c] = src[q];
    }
    for (int q = 0; q < NC; ++q) storeRows(row, q, N, c0, cols, vals, cnt, err);
  }
}

// fv::dive(u, phi, theta), ExplicitDivergence.h:7-51: sources only, from
// (u0, phi0) and (u1, phi1); the rows stay empty
template <int NC>
__global__ __launch_bounds__(kRowBlock) void kEqDive(MeshDev M, const double *__restrict__ u0F,
                                                     const double *__restrict__ u1F, double theta,
                                                     const int *__restrict__ bc, const double *__restrict__ phi0C,
                                                     const double *__restrict__ phi1C,
                                                     const double *__restrict__ phi0F,
                                                     const double *__restrict__ phi1F, int stride, int *cols,
                                                     double *vals, int *cnt, double *rhs, int *err) {
  const int N = M.nCells;
  for (int c0 = blockIdx.x * kRowBlock; c0 < N; c0 += gridDim.x * kRowBlock) {
    const int c = c0 + threadIdx.x;
    RowS row(c, stride, false);
    if (c < N) {
      double src[NC] = {};
      double p0[NC], p1[NC], n0[4][NC], n1[4][NC];
      for (int q = 0; q < NC; ++q) {
        p0[q] = phi0C[NC * (size_t)c + q];
        p1[q] = phi1C[NC * (size_t)c + q];
      }
      Dv2 s[4], u0[4], u1[4];
      forLinks(M.iptr[c], M.iptr[c + 1],
               [&](int q, int k) {
                 const int link = M.iface[k], f = faceOf(link), nb = M.inb[k];
                 s[q] = outwardOf(link, M.sf);
                 u0[q] = ld2(u0F, f);
                 u1[q] = ld2(u1F, f);
                 for (int i = 0; i < NC; ++i) {
                   n0[q][i] = phi0C[NC * (size_t)nb + i];
                   n1[q][i] = phi1C[NC * (size_t)nb + i];
                 }
               },
               [&](int q, int) {
                 const double flux0 = u0[q].x * s[q].x + u0[q].y * s[q].y;
                 const double flux1 = u1[q].x * s[q].x + u1[q].y * s[q].y;
                 for (int i = 0; i < NC; ++i) src[i] += theta * upMax(flux0) * p0[i];
                 for (int i = 0; i < NC; ++i) src[i] += theta * upMin(flux0) * n0[q][i];
                 for (int i = 0; i < NC; ++i) src[i] += (1. - theta) * upMax(flux1) * p1[i];
                 for (int i = 0; i < NC; ++i) src[i] += (1. - theta) * upMin(flux1) * n1[q][i];
               });
      for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
        const int link = M.bface[k], f = faceOf(link);
        const Dv2 s = outwardOf(link, M.sf);
        const double flux0 = u0F[2 * f] * s.x + u0F[2 * f + 1] * s.y;
        const double flux1 = u1F[2 * f] * s.x + u1F[2 * f + 1] * s.y;
        const int bt = bc ? bc[f] : PHASE_HIP_BC_NORMAL_GRADIENT;
        if (bt == PHASE_HIP_BC_FIXED || bt == PHASE_HIP_BC_NORMAL_GRADIENT) {
          for (int q = 0; q < NC; ++q) src[q] += theta * flux0 * phi0F[NC * (size_t)f + q];
          for (int q = 0; q < NC; ++q) src[q] += (1. - theta) * flux1 * phi1F[NC * (size_t)f + q];
        } else if (bt == PHASE_HIP_BC_SYMMETRY) {
        } else {
          atomicOr(err, 1);
        }
      }
      row.finish();
      for (int q = 0; q < NC; ++q) rhs[(size_t)q * N + c] = src[q];
    }
    for (int q = 0; q < NC; ++q) storeRows(row, q, N, c0, cols, vals, cnt, err);
  }
}

// fv::div(phiU, gradU, u), Divergence.cpp:3-47 (Vector2D): upwind with the
// upwind cell's Jacobian (xx xy yx yy) carried to the face centroid
__global__ __launch_bounds__(kRowBlock) void kEqDivGrad(MeshDev M, const double *__restrict__ phiUF,
                                                        const double *__restrict__ J, const int *__restrict__ bc,
                                                        const double *__restrict__ uF, int stride, int *cols,
                                                        double *vals, int *cnt, double *rhs, int *err) {
  constexpr int NC = 2;
  const int N = M.nCells;
  for (int c0 = blockIdx.x * kRowBlock; c0 < N; c0 += gridDim.x * kRowBlock) {
    const int c = c0 + threadIdx.x;
    RowS row(c, stride, M.repeated);
    if (c < N) {
      double src[NC] = {};
      auto jsrc = [&](int cell, double rx, double ry, double flux) {
        const double *j = J + 4 * (size_t)cell;
        const double vx = j[0] * rx + j[1] * ry, vy = j[2] * rx + j[3] * ry;
        src[0] += flux * vx;
        src[1] += flux * vy;
      };
      const Dv2 pc = ld2(M.cc, c);
      int nb[4];
      Dv2 s[4], u[4], fc[4], cn[4];
      forLinks(M.iptr[c], M.iptr[c + 1],
               [&](int q, int k) {
                 const int link = M.iface[k], f = faceOf(link);
                 nb[q] = M.inb[k];
                 s[q] = outwardOf(link, M.sf);
                 u[q] = ld2(phiUF, f);
                 fc[q] = ld2(M.fc, f);
                 cn[q] = ld2(M.cc, nb[q]);
               },
               [&](int q, int) {
                 const double flux = u[q].x * s[q].x + u[q].y * s[q].y;
                 if (flux > 0.) {
                   row.addDiag(flux);
                   jsrc(c, fc[q].x - pc.x, fc[q].y - pc.y, flux);
                 } else {
                   row.add(nb[q], flux);
                   jsrc(nb[q], fc[q].x - cn[q].x, fc[q].y - cn[q].y, flux);
                 }
               });
      for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
        const int link = M.bface[k], f = faceOf(link);
        const Dv2 fb = ld2(M.fc, f);
        const Dv2 s = outwardOf(link, M.sf);
        const double flux = phiUF[2 * f] * s.x + phiUF[2 * f + 1] * s.y;
        const int bt = bc ? bc[f] : PHASE_HIP_BC_NORMAL_GRADIENT;
        if (bt == PHASE_HIP_BC_FIXED) {
          if (!uF) {
            atomicOr(err, 2);
            continue;
          }
          src[0] += flux * uF[2 * f];
          src[1] += flux * uF[2 * f + 1];
        } else if (bt == PHASE_HIP_BC_NORMAL_GRADIENT) {
          row.addDiag(flux);
          jsrc(c, fb.x - pc.x, fb.y - pc.y, flux);
        } else if (bt == PHASE_HIP_BC_SYMMETRY) {
        } else {
          atomicOr(err, 1);
        }
      }
      row.finish();
      for (int q = 0; q < NC; ++q) rhs[(size_t)q * N + c] = src[q];
    }
    for (int q = 0; q < NC; ++q) storeRows(row, q, N, c0, cols, vals, cnt, err);
  }
}

// VectorFiniteVolumeField::faceToCell, plain (VectorFiniteVolumeField.cpp:5-26)
// or weighted (:28-51): sum of pointwise(v_f, |S_f|) [/ faceWeight_f] over the
// cell's faces, componentwise over sum |S_f| [times cellWeight]
__global__ __launch_bounds__(256) void kFaceToCell(MeshDev M, const double *__restrict__ fv,
                                                   const double *__restrict__ cw, const double *__restrict__ fw,
                                                   double *__restrict__ out) {
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < M.nCells; c += gridDim.x * blockDim.x) {
    double sx = 0., sy = 0., tx = 0., ty = 0.;
    Dv2 n[4], v[4];
    double w[4];
    auto load = [&](int q, int link) {
      const int f = faceOf(link);
      n[q] = ld2(M.sf, f);
      v[q] = ld2(fv, f);
      w[q] = fw ? fw[f] : 1.;
    };
    auto add = [&](int q, int) {
      const double ax = fabs(n[q].x), ay = fabs(n[q].y);
      double px = v[q].x * ax, py = v[q].y * ay;
      if (fw) {
        px /= w[q];
        py /= w[q];
      }
      tx += px;
      ty += py;
      sx += ax;
      sy += ay;
    };
    forLinks(M.iptr[c], M.iptr[c + 1], [&](int q, int k) { load(q, M.iface[k]); }, add);
    for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
      load(0, M.bface[k]);
      add(0, k);
    }
    double vx = tx / sx, vy = ty / sy;
    if (cw) {
      vx = cw[c] * vx;
      vy = cw[c] * vy;
    }
    st2(out, c, vx, vy);
  }
}

// ---------------------------------------------------------------- VOF (CICSAM)
// std::min / std::max as the reference calls them -- min(a, b) = (b < a) ? b : a,
// max(a, b) = (a < b) ? b : a -- so a NaN first argument passes through
__device__ __forceinline__ double smin(double a, double b) { return (b < a) ? b : a; }
__device__ __forceinline__ double smax(double a, double b) { return (a < b) ? b : a; }
// clamp(v, lo, hi) = max(min(v, hi), lo), Math/Algorithm.h:11-13
__device__ __forceinline__ double sclamp(double v, double lo, double hi) { return smax(smin(v, hi), lo); }
// cicsam::hc and cicsam::uq, Cicsam.cpp:5-18
__device__ __forceinline__ double cicsamHc(double g, double co) { return g >= 0 && g <= 1 ? smin(1., g / co) : g; }
__device__ __forceinline__ double cicsamUq(double g, double co) {
  return g >= 0 && g <= 1 ? smin((8. * co * g + (1. - co) * (6. * g + 3.)) / 8., cicsamHc(g, co)) : g;
}

// Courant number of a cell's outflow over all of its faces, summed in link order
// (the donor's number in Cicsam.cpp:20-66)
__device__ __forceinline__ double courantOf(const MeshDev &M, int c, const double *__restrict__ uF, double dt) {
  const double v = M.vol[c];
  double sum = 0.;
  Dv2 n[4], u[4];
  auto load = [&](int q, int link) {
    n[q] = outwardOf(link, M.sf);
    u[q] = ld2(uF, faceOf(link));
  };
  auto add = [&](int q, int) { sum += smax((u[q].x * n[q].x + u[q].y * n[q].y) / v * dt, 0.); };
  forLinks(M.iptr[c], M.iptr[c + 1], [&](int q, int k) { load(q, M.iface[k]); }, add);
  for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
    load(0, M.bface[k]);
    add(0, k);
  }
  return sum;
}
__global__ __launch_bounds__(256) void kCellCourant(MeshDev M, const double *__restrict__ uF, double dt,
                                                    double *__restrict__ co) {
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < M.nCells; c += gridDim.x * blockDim.x)
    co[c] = courantOf(M, c, uF, dt);
}

// cicsam::faceInterpolationWeights, Cicsam.cpp:20-66 (k = 1), one face per
// thread; boundary faces 0.  cos(2 theta_F) with theta_F = acos(c) is
// evaluated as 2 c^2 - 1 (c > 1 from rounding stays NaN, as acos makes it).
// CELLS: the donors' Courant numbers from kCellCourant, once per cell; else
// formed here, the donor's four faces read again per face.
template <bool CELLS>
__global__ __launch_bounds__(256) void kCicsamWeights(MeshDev M, int nFaces, const int *__restrict__ fl,
                                                      const int *__restrict__ fr, const double *__restrict__ uF,
                                                      const double *__restrict__ gC,
                                                      const double *__restrict__ gradC, double dt,
                                                      const double *__restrict__ co, double *__restrict__ beta) {
  for (int f = blockIdx.x * blockDim.x + threadIdx.x; f < nFaces; f += gridDim.x * blockDim.x) {
    const int l = fl[f], r = fr[f];
    if (r < 0) {
      beta[f] = 0.;
      continue;
    }
    const Dv2 uf = ld2(uF, f);
    const Dv2 s = outward(ld2(M.fc, f), ld2(M.sf, f), ld2(M.cc, l));
    const double flux = uf.x * s.x + uf.y * s.y;
    const int d = flux > 0. ? l : r, a = flux <= 0. ? l : r;
    const Dv2 cd = ld2(M.cc, d), ca = ld2(M.cc, a);
    const Dv2 rc{ca.x - cd.x, ca.y - cd.y};
    const Dv2 gd = ld2(gradC, d);
    const double coD = CELLS ? co[d] : courantOf(M, d, uF, dt);
    const double gD = sclamp(gC[d], 0., 1.), gA = sclamp(gC[a], 0., 1.);
    const double gU = sclamp(gA - 2. * (rc.x * gd.x + rc.y * gd.y), 0., 1.);
    double gDT = (gD - gU) / (gA - gU);
    if (!isfinite(gDT)) gDT = 0.;
    const double mg = sqrt(gd.x * gd.x + gd.y * gd.y), mr = sqrt(rc.x * rc.x + rc.y * rc.y);
    const double c = fabs((gd.x / mg) * (rc.x / mr) + (gd.y / mg) * (rc.y / mr));
    const double cos2 = c > 1. ? __builtin_nan("") : 2. * c * c - 1.;
    const double psiF = smin(1. * (cos2 + 1.) / 2., 1.);
    const double gFT = psiF * cicsamHc(gDT, coD) + (1. - psiF) * cicsamUq(gDT, coD);
    const double b = (gFT - gDT) / (1. - gDT);
    beta[f] = isfinite(b) ? smax(smin(1., b), 0.) : 0.;
  }
}

// cicsam::div(u, gamma, beta, theta), Cicsam.cpp:87-138: per link the donor and
// acceptor coefficients theta (1 - b) F and theta b F in that order, the
// explicit part as a source, boundary links by type (err bit 1: other type)
__global__ __launch_bounds__(kRowBlock) void kEqCicsamDiv(MeshDev M, const double *__restrict__ uF,
                                                          const double *__restrict__ beta, double theta,
                                                          const int *__restrict__ bc, const double *__restrict__ gF,
                                                          const double *__restrict__ g0C,
                                                          const double *__restrict__ g0F, int stride, int *cols,
                                                          double *vals, int *cnt, double *rhs, int *err) {
  constexpr int NC = 1;
  const int N = M.nCells;
  for (int c0 = blockIdx.x * kRowBlock; c0 < N; c0 += gridDim.x * kRowBlock) {
    const int c = c0 + threadIdx.x;
    RowS row(c, stride, M.repeated);
    if (c < N) {
      double src[NC] = {};
      const double p0 = g0C[c];
      int nb[4];
      Dv2 s[4], u[4];
      double b[4], pn[4];
      forLinks(M.iptr[c], M.iptr[c + 1],
               [&](int q, int k) {
                 const int link = M.iface[k], f = faceOf(link);
                 nb[q] = M.inb[k];
                 s[q] = outwardOf(link, M.sf);
                 u[q] = ld2(uF, f);
                 b[q] = beta[f];
                 pn[q] = g0C[nb[q]];
               },
               [&](int q, int) {
                 const double flux = u[q].x * s[q].x + u[q].y * s[q].y;
                 const double cd = theta * (1. - b[q]) * flux, ca = theta * b[q] * flux;
                 // donor, then acceptor; for a NaN flux both are the neighbour
                 if (flux > 0.) row.addDiag(cd);
                 else row.add(nb[q], cd);
                 if (flux <= 0.) row.addDiag(ca);
                 else if (flux > 0.) row.add(nb[q], ca);
                 else row.add(nb[q], ca, true);
                 const double gFace = (1. - b[q]) * (flux > 0. ? p0 : pn[q]) + b[q] * (flux <= 0. ? p0 : pn[q]);
                 src[0] += (1. - theta) * flux * gFace;
               });
      for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
        const int link = M.bface[k], f = faceOf(link);
        const Dv2 s = outwardOf(link, M.sf);
        const double flux = uF[2 * f] * s.x + uF[2 * f + 1] * s.y;
        const int bt = bc ? bc[f] : PHASE_HIP_BC_NORMAL_GRADIENT;
        if (bt == PHASE_HIP_BC_FIXED) {
          if (!gF || !g0F) {
            atomicOr(err, 2);
            continue;
          }
          src[0] += theta * flux * gF[f];
          src[0] += (1. - theta) * flux * g0F[f];
        } else if (bt == PHASE_HIP_BC_NORMAL_GRADIENT) {
          row.addDiag(theta * flux);
          src[0] += (1. - theta) * flux * p0;
        } else if (bt == PHASE_HIP_BC_SYMMETRY) {
        } else {
          atomicOr(err, 1);
        }
      }
      row.finish();
      for (int q = 0; q < NC; ++q) rhs[(size_t)q * N + c] = src[q];
    }
    for (int q = 0; q < NC; ++q) storeRows(row, q, N, c0, cols, vals, cnt, err);
  }
}

// cicsam::computeMomentumFlux, Cicsam.cpp:68-85 (rhoU per face, interleaved)
__global__ void kCicsamMomentumFlux(MeshDev M, int nFaces, const int *__restrict__ fl, const int *__restrict__ fr,
                                    double rho1, double rho2, const double *__restrict__ uF,
                                    const double *__restrict__ gC, const double *__restrict__ gF,
                                    const double *__restrict__ beta, double *__restrict__ rhoU) {
  for (int f = blockIdx.x * blockDim.x + threadIdx.x; f < nFaces; f += gridDim.x * blockDim.x) {
    const int l = fl[f], r = fr[f];
    const Dv2 uf = ld2(uF, f);
    double g;
    if (r >= 0) {
      const Dv2 s = outward(ld2(M.fc, f), ld2(M.sf, f), ld2(M.cc, l));
      const double flux = uf.x * s.x + uf.y * s.y;
      const int d = flux > 0. ? l : r, a = flux <= 0. ? l : r;
      const double b = beta[f];
      g = (1. - b) * gC[d] + b * gC[a];
    } else {
      g = gF[f];
    }
    const double rho = rho1 + sclamp(g, 0., 1.) * (rho2 - rho1);
    rhoU[2 * f] = rho * uf.x;
    rhoU[2 * f + 1] = rho * uf.y;
  }
}

// FractionalStepMultiphase::updateProperties, FractionalStepMultiphase.cpp:175-214:
// density, and dynamic viscosity from the kinematic viscosities, for n values
__global__ void kVofProperties(int n, double rho1, double rho2, double mu1, double mu2, const double *__restrict__ g,
                               double *__restrict__ rho, double *__restrict__ mu) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double gi = sclamp(g[i], 0., 1.);
    const double r = rho1 + gi * (rho2 - rho1);
    rho[i] = r;
    mu[i] = r / (rho1 / mu1 + gi * (rho2 / mu2 - rho1 / mu1));
  }
}

// lhs (+|-)= rhs, CrsEquation.cpp:185-275: the left row's non-zero entries, in
// order, then the right row's accumulated into a matching column or appended.
// Both sides' rows come through LDS in contiguous runs and are merged in place
// there; an entry mostly meets its column at its own index, or one off.  Bound
// by HBM: three rows of `stride` slots moved per row.
// 2M rows of 6 slots: 107 us, 4.0 TB/s (153 us with rows in registers).
constexpr int kMergeBlock = 128;
inline size_t mergeLds(int stride) { return 2 * (size_t)kMergeBlock * rowPitch(stride) * (sizeof(double) + sizeof(int)); }
__global__ __launch_bounds__(kMergeBlock) void kEqMerge(int rank, int stride, int sign, int *lc, double *lv, int *ln,
                                                        double *lr, const int *rc, const double *rv, const int *rn,
                                                        const double *rr, int *err) {
  const int P = stride | 1;
  double *sl = (double *)rowStage, *sr = sl + kMergeBlock * P;
  int *cl = (int *)(sr + kMergeBlock * P), *cr = cl + kMergeBlock * P;
  const float inv = 1.f / (float)stride;
  for (int r0 = blockIdx.x * kMergeBlock; r0 < rank; r0 += gridDim.x * kMergeBlock) {
    const int rows = min(kMergeBlock, rank - r0);
    const size_t base = (size_t)r0 * stride;
    for (int idx = threadIdx.x; idx < rows * stride; idx += kMergeBlock) {
      const int row = (int)((idx + 0.5f) * inv), at = row * P + idx - row * stride;
      cl[at] = lc[base + idx];
      sl[at] = lv[base + idx];
      cr[at] = rc[base + idx];
      sr[at] = rv[base + idx];
    }
    const int row = r0 + threadIdx.x;
    const bool mine = (int)threadIdx.x < rows;
    const int nl = mine ? ln[row] : 0, nr = mine ? rn[row] : 0;
    const double rhsL = mine ? lr[row] : 0., rhsR = mine ? rr[row] : 0.;
    __syncthreads();
    int n = 0;
    bool over = false;
    if (mine) {
      int *c = cl + threadIdx.x * P;
      double *v = sl + threadIdx.x * P;
      const int *oc = cr + threadIdx.x * P;
      const double *ov = sr + threadIdx.x * P;
      for (int j = 0; j < nl; ++j) {
        const int cj = c[j];
        const double vj = v[j];
        if (vj != 0. && cj >= 0) {
          c[n] = cj;
          v[n] = vj;
          ++n;
        }
      }
      for (int j = 0; j < nr; ++j) {
        const double vj = ov[j];
        const int cj = oc[j];
        if (vj == 0. || cj < 0) continue;
        const double w = sign > 0 ? vj : -vj;
        int p = -1;
        if (j < n && c[j] == cj) p = j;
        else
          for (int q = 0; q < n && p < 0; ++q)
            if (c[q] == cj) p = q;
        if (p >= 0) {
          v[p] += w;
        } else if (n < stride) {
          c[n] = cj;
          v[n] = w;
          ++n;
        } else {
          over = true;
        }
      }
      for (int j = n; j < stride; ++j) {
        c[j] = -1;
        v[j] = 0.;
      }
      lr[row] = sign > 0 ? rhsL + rhsR : rhsL - rhsR;
      if (!over) ln[row] = n;
    }
    if (__syncthreads_or(over)) {  // rows with more columns than slots keep what they held
      if (over) atomicOr(err, 4);
      if (mine && !over)
        for (int j = 0; j < stride; ++j) {
          lc[base + (size_t)threadIdx.x * stride + j] = cl[threadIdx.x * P + j];
          lv[base + (size_t)threadIdx.x * stride + j] = sl[threadIdx.x * P + j];
        }
    } else {
      for (int idx = threadIdx.x; idx < rows * stride; idx += kMergeBlock) {
        const int r = (int)((idx + 0.5f) * inv), at = r * P + idx - r * stride;
        lc[base + idx] = cl[at];
        lv[base + idx] = sl[at];
      }
    }
    __syncthreads();
  }
}

// CrsEquation::operator*=(Scalar), CrsEquation.cpp:287-291
__global__ void kEqScale(int rank, int stride, double s, double *vals, double *rhs) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < (size_t)rank * stride;
       i += (size_t)gridDim.x * blockDim.x)
    vals[i] *= s;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rank; i += gridDim.x * blockDim.x) rhs[i] *= s;
}

// operator*(ScalarFiniteVolumeField, equation): every slot and the rhs of row
// r times field[r mod nCells] (scaleRow, CrsEquation.cpp:153-159)
__global__ void kEqScaleCells(int rank, int nCells, int stride, const double *__restrict__ field, double *vals,
                              double *rhs) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < (size_t)rank * stride;
       i += (size_t)gridDim.x * blockDim.x)
    vals[i] *= field[(i / stride) % nCells];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rank; i += gridDim.x * blockDim.x)
    rhs[i] *= field[i % nCells];
}

// remove(cell): the masked cells' rows keep their values but lose their
// columns (-1) and rhs
__global__ void kEqRemoveCells(int rank, int nCells, int stride, const int *__restrict__ mask, int *cols,
                               double *rhs) {
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < rank; r += gridDim.x * blockDim.x) {
    if (!mask[r % nCells]) continue;
    for (int j = 0; j < stride; ++j) cols[(size_t)r * stride + j] = -1;
    rhs[r] = 0.;
  }
}

// rhs -= v (operator-=(Vector) / ==(Vector), CrsEquation.cpp:282-285, 308-311);
// v == nullptr: rhs -= s (operator==(Scalar), :299-303)
__global__ void kEqSubRhs(int rank, const double *__restrict__ v, double s, double *rhs) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rank; i += gridDim.x * blockDim.x)
    rhs[i] -= v ? v[i] : s;
}

// implicit under-relaxation: a_P /= alpha; rhs -= (1 - alpha) * a_P * phi
// (ScalarFiniteVolumeEquation.cpp:45-55, VectorFiniteVolumeEquation.cpp:129-146)
__global__ void kEqRelax(int rank, int stride, double alpha, const double *__restrict__ phi, const int *cols,
                         double *vals, const int *cnt, double *rhs) {
  for (int row = blockIdx.x * blockDim.x + threadIdx.x; row < rank; row += gridDim.x * blockDim.x) {
    const size_t o = (size_t)row * stride;
    for (int j = 0; j < cnt[row]; ++j)
      if (cols[o + j] == row) {
        vals[o + j] /= alpha;
        rhs[row] -= (1. - alpha) * vals[o + j] * phi[row];
        break;
      }
  }
}

// src::div(u), Source.cpp:5-21: sum over the cell's faces of dot(u_f, Sf_out).
// The field kernels are bound by HBM; at 1M triangles (1.5M faces) this one
// takes 23.8 us (47.6 us with the outward test per link and one link at a
// time), the cell gradients 26.3 us (31.6), the face gradients 14.8 us (18.5)
// and the vector face interpolation 15.4 us (29) with their geometry per face.
__global__ __launch_bounds__(256) void kSrcDiv(MeshDev M, const double *__restrict__ uF, double *__restrict__ out) {
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < M.nCells; c += gridDim.x * blockDim.x) {
    double d = 0.;
    Dv2 s[4], u[4];
    auto load = [&](int q, int link) {
      s[q] = outwardOf(link, M.sf);
      u[q] = ld2(uF, faceOf(link));
    };
    auto add = [&](int q, int) { d += u[q].x * s[q].x + u[q].y * s[q].y; };
    forLinks(M.iptr[c], M.iptr[c + 1], [&](int q, int k) { load(q, M.iface[k]); }, add);
    for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
      load(0, M.bface[k]);
      add(0, k);
    }
    out[c] = d;
  }
}

// src::src(field), Source.cpp:77-95: phi * V per row (block layout)
__global__ void kSrcSrc(MeshDev M, int ncomp, const double *__restrict__ phiC, double *out) {
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < M.nCells; c += gridDim.x * blockDim.x)
    for (int q = 0; q < ncomp; ++q) out[(size_t)q * M.nCells + c] = phiC[ncomp * c + q] * M.vol[c];
}

// ScalarGradient::computeFaces, ScalarGradient.cpp:34-52
__global__ __launch_bounds__(256) void kGradFaces(int nFaces, const int *__restrict__ fl, const int *__restrict__ fr,
                                                  const double *__restrict__ faceD, const double *__restrict__ phiC,
                                                  const double *__restrict__ phiF, double *__restrict__ gF) {
  for (int f = blockIdx.x * blockDim.x + threadIdx.x; f < nFaces; f += gridDim.x * blockDim.x) {
    const int l = fl[f], r = fr[f];
    const Dv2 d = ld2(faceD, f);
    const double dphi = (r >= 0 ? phiC[r] : phiF[f]) - phiC[l];
    const double ms = d.x * d.x + d.y * d.y;
    st2(gF, f, d.x * dphi / ms, d.y * dphi / ms);
  }
}

// ScalarGradient::compute(FACE_TO_CELL), ScalarGradient.cpp:54-74:
// componentwise sum_f g_f |Sf_out| / sum_f |Sf_out| over the cell's links
__global__ __launch_bounds__(256) void kGradCells(MeshDev M, const double *__restrict__ gF, double *__restrict__ gC) {
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < M.nCells; c += gridDim.x * blockDim.x) {
    double sx = 0., sy = 0., tx = 0., ty = 0.;
    Dv2 n[4], g[4];
    auto load = [&](int q, int link) {
      n[q] = ld2(M.sf, faceOf(link));
      g[q] = ld2(gF, faceOf(link));
    };
    auto add = [&](int q, int) {
      const double ax = fabs(n[q].x), ay = fabs(n[q].y);
      tx += g[q].x * ax;
      ty += g[q].y * ay;
      sx += ax;
      sy += ay;
    };
    forLinks(M.iptr[c], M.iptr[c + 1], [&](int q, int k) { load(q, M.iface[k]); }, add);
    for (int k = M.bptr[c]; k < M.bptr[c + 1]; ++k) {
      load(0, M.bface[k]);
      add(0, k);
    }
    st2(gC, c, tx / sx, ty / sy);
  }
}

// interpolateFaces(DISTANCE) + setBoundaryFaces, FiniteVolumeField.tpp:129-182
// and VectorFiniteVolumeField.cpp:140-160; FIXED faces keep their value.
template <int NC>
__global__ __launch_bounds__(256) void kInterpFaces(int nFaces, const int *__restrict__ fl, const int *__restrict__ fr,
                                                    const double *__restrict__ faceW, const double *__restrict__ sf,
                                                    const int *__restrict__ bc, const double *__restrict__ phiC,
                                                    double *__restrict__ phiF) {
  for (int f = blockIdx.x * blockDim.x + threadIdx.x; f < nFaces; f += gridDim.x * blockDim.x) {
    const int l = fl[f], r = fr[f];
    if (r >= 0) {
      const double g = faceW[f];
      if (NC == 2) {
        const Dv2 a = ld2(phiC, l), b = ld2(phiC, r);
        st2(phiF, f, g * a.x + (1. - g) * b.x, g * a.y + (1. - g) * b.y);
      } else {
        phiF[f] = g * phiC[l] + (1. - g) * phiC[r];
      }
      continue;
    }
    const int bt = bc ? bc[f] : PHASE_HIP_BC_NORMAL_GRADIENT;
    if (bt == PHASE_HIP_BC_FIXED) continue;
    if (bt == PHASE_HIP_BC_SYMMETRY && NC == 2) {
      const double nx = sf[2 * f], ny = sf[2 * f + 1];
      const double px = phiC[2 * l], py = phiC[2 * l + 1];
      const double d = px * nx + py * ny;
      const double ms = nx * nx + ny * ny;
      phiF[2 * f] = px - nx * d / ms;
      phiF[2 * f + 1] = py - ny * d / ms;
    } else {
      for (int q = 0; q < NC; ++q) phiF[NC * (size_t)f + q] = phiC[NC * (size_t)l + q];
    }
  }
}

// f with the equation's component count as a compile-time constant
template <class F>
void byComponents(int ncomp, F &&f) {
  if (ncomp == 1) f(std::integral_constant<int, 1>());
  else f(std::integral_constant<int, 2>());
}

inline int g256(long n) { return (int)std::max<long>(1, std::min<long>((n + 255) / 256, 8192)); }

template <class F>
int guardedEq(phase_hip_equation *e, F &&f) {
  if (!e) return PHASE_HIP_EINVAL;
  try {
    f();
    return PHASE_HIP_OK;
  } catch (const HipError &x) {
    e->err = x.msg;
    return x.code;
  } catch (const std::exception &x) {
    e->err = x.what();
    return PHASE_HIP_EINVAL;
  }
}

template <class F>
int guardedM(phase_hip_mesh *m, F &&f) {
  if (!m) return PHASE_HIP_EINVAL;
  try {
    f();
    return PHASE_HIP_OK;
  } catch (const HipError &x) {
    m->err = x.msg;
    return x.code;
  } catch (const std::exception &x) {
    m->err = x.what();
    return PHASE_HIP_EINVAL;
  }
}

// Pinned ints for the equations' error bits, one block of 1024 for the process
// (a pinned allocation per equation took longer than the rest of its creation);
// past those, an allocation of its own.
class PinnedSlots {
 public:
  int *take() {
    std::lock_guard<std::mutex> lock(mutex_);
    if (!block_) {
      PH_CHECK(hipHostMalloc((void **)&block_, kSlots * sizeof(int), hipHostMallocPortable));
      for (int i = 0; i < kSlots; ++i) free_.push_back(block_ + i);
    }
    int *p = nullptr;
    if (free_.empty()) {
      PH_CHECK(hipHostMalloc((void **)&p, sizeof(int), hipHostMallocPortable));
    } else {
      p = free_.back();
      free_.pop_back();
    }
    return p;
  }
  void give(int *p) {
    std::lock_guard<std::mutex> lock(mutex_);
    if (p >= block_ && p < block_ + kSlots) free_.push_back(p);
    else (void)hipHostFree(p);
  }

 private:
  static constexpr int kSlots = 1024;
  std::mutex mutex_;
  int *block_ = nullptr;
  std::vector<int *> free_;
};
PinnedSlots &pinnedSlots() {
  static PinnedSlots *s = new PinnedSlots();  // never destroyed: equations may outlive static objects
  return *s;
}

// Device error bits of the last operator: raised as the reference's exceptions.
void checkEq(phase_hip_equation *e, const char *op) {
  PH_CHECK(hipMemcpyAsync(e->hErr, e->dErr.p, sizeof(int), hipMemcpyDeviceToHost, e->mesh->stream));
  PH_CHECK(hipStreamSynchronize(e->mesh->stream));
  const int v = *e->hErr;
  if (!v) return;
  PH_CHECK(hipMemsetAsync(e->dErr.p, 0, sizeof(int), e->mesh->stream));
  if (v & 1) fail(PHASE_HIP_EBOUNDARY, std::string(op) + ": unrecognized or unspecified boundary type.");
  if (v & 2) fail(PHASE_HIP_EINVAL, std::string(op) + ": a boundary or old-time input is missing");
  fail(PHASE_HIP_EINVAL, std::string(op) + ": a row needs more slots than the equation holds");
}

void fresh(phase_hip_equation *e) { e->compact = false; }

}  // namespace

phase_hip_equation::~phase_hip_equation() {
  if (hErr) pinnedSlots().give(hErr);
}

namespace phase {

// Solver side of FiniteVolumeEquation<T>::solve (FiniteVolumeEquation.tpp:64-86):
// A from the equation's rows, b = -rhs.  Defined in solver.hip.  adjPtr /
// adjNb (host, may be NULL): the rows' structural neighbours (for scalar mesh
// equations the face neighbours), the largest pattern the rows can take.
void solverSetFromRows(phase_hip_solver *s, int rank, int stride, const int *dCols, const double *dVals,
                       const double *dRhs, hipStream_t producer, const double *dCellXY, const int *adjPtr,
                       const int *adjNb);

}  // namespace phase

extern "C" {

const char *phase_hip_equation_last_error(const phase_hip_equation *e) { return e ? e->err.c_str() : "null equation"; }

int phase_hip_equation_create(phase_hip_equation **out, phase_hip_mesh *m, int ncomp) {
  if (!out || !m || (ncomp != 1 && ncomp != 2)) return PHASE_HIP_EINVAL;
  *out = nullptr;
  phase_hip_equation *e = new phase_hip_equation();
  e->mesh = m;
  e->ncomp = ncomp;
  e->rank = ncomp * m->nCells;
  // diagonal + neighbours (+ one cross-component column for Vector2D)
  e->stride = std::max(5, 1 + m->maxDeg + (ncomp == 2 ? 1 : 0));
  const int rc = guardedEq(e, [&] {
    if (e->stride > kRowCap) fail(PHASE_HIP_EINVAL, "a cell has more faces than an equation row holds");
    PH_CHECK(hipSetDevice(m->device));
    const size_t slots = (size_t)e->rank * e->stride;
    e->cols.alloc(slots);
    e->vals.alloc(slots);
    e->cnt.alloc(e->rank);
    e->rhs.alloc(e->rank);
    e->dErr.alloc(1);
    e->dErr.zero(m->stream);
    e->hErr = pinnedSlots().take();
    // CrsEquation(N, 5): every slot empty
    PH_CHECK(hipMemsetAsync(e->cols.p, 0xff, slots * sizeof(int), m->stream));
    e->vals.zero(m->stream);
    e->cnt.zero(m->stream);
    e->rhs.zero(m->stream);
    PH_CHECK(hipStreamSynchronize(m->stream));
  });
  if (rc != PHASE_HIP_OK) {
    delete e;
    return rc;
  }
  *out = e;
  return PHASE_HIP_OK;
}

int phase_hip_equation_destroy(phase_hip_equation *e) {
  delete e;
  return PHASE_HIP_OK;
}

int phase_hip_equation_rank(const phase_hip_equation *e) { return e ? e->rank : 0; }

int phase_hip_eq_laplacian(phase_hip_equation *e, int variant, double gamma, const double *gammaFace,
                           const double *gamma0Face, double theta, const int *bcType, const double *phiFace,
                           const double *phi0Cell, const double *phi0Face) {
  return guardedEq(e, [&] {
    if (variant < 0 || variant > 3) fail(PHASE_HIP_EINVAL, "laplacian variant must be 0..3");
    if (variant >= 2 && (!gammaFace || (variant == 2 && !gamma0Face)))
      fail(PHASE_HIP_EINVAL, "face-field laplacian needs gammaFace (and gamma0Face with theta)");
    phase_hip_mesh *m = e->mesh;
    PH_CHECK(hipSetDevice(m->device));
    byComponents(e->ncomp, [&](auto nc) {
      hipLaunchKernelGGL((kEqLaplacian<decltype(nc)::value>), dim3(g256(m->nCells)), dim3(kRowBlock),
                         rowLds(e->stride),
                         m->stream, meshDev(m), variant, gamma, gammaFace, gamma0Face, theta, bcType, phiFace,
                         phi0Cell, phi0Face, e->stride, e->cols.p, e->vals.p, e->cnt.p, e->rhs.p, e->dErr.p);
    });
    PH_CHECK(hipGetLastError());
    fresh(e);
    checkEq(e, "fv::laplacian");
  });
}

int phase_hip_eq_ddt(phase_hip_equation *e, double timeStep, const double *phi0Cell) {
  return guardedEq(e, [&] {
    if (!phi0Cell) fail(PHASE_HIP_EINVAL, "fv::ddt needs the old-time field");
    phase_hip_mesh *m = e->mesh;
    PH_CHECK(hipSetDevice(m->device));
    byComponents(e->ncomp, [&](auto nc) {
      hipLaunchKernelGGL((kEqDdt<decltype(nc)::value>), dim3(g256(m->nCells)), dim3(kRowBlock), rowLds(e->stride),
                         m->stream, meshDev(m), timeStep, phi0Cell, e->stride, e->cols.p, e->vals.p, e->cnt.p,
                         e->rhs.p, e->dErr.p);
    });
    PH_CHECK(hipGetLastError());
    fresh(e);
  });
}

int phase_hip_eq_ddt_rho(phase_hip_equation *e, double timeStep, double rho, const double *rhoCell,
                         const double *rho0Cell, const double *phi0Cell, const int *cellMask) {
  return guardedEq(e, [&] {
    if (!phi0Cell) fail(PHASE_HIP_EINVAL, "fv::ddt needs the old-time field");
    if (!rhoCell != !rho0Cell) fail(PHASE_HIP_EINVAL, "a density field needs its old-time values too");
    phase_hip_mesh *m = e->mesh;
    PH_CHECK(hipSetDevice(m->device));
    byComponents(e->ncomp, [&](auto nc) {
      hipLaunchKernelGGL((kEqDdtRho<decltype(nc)::value>), dim3(g256(m->nCells)), dim3(kRowBlock), rowLds(e->stride),
                         m->stream, meshDev(m), timeStep, rho, rhoCell, rho0Cell, phi0Cell, cellMask, e->stride,
                         e->cols.p, e->vals.p, e->cnt.p, e->rhs.p, e->dErr.p);
    });
    PH_CHECK(hipGetLastError());
    fresh(e);
  });
}

int phase_hip_eq_div(phase_hip_equation *e, const double *uFace, const double *u0Face, double theta,
                     const int *bcType, const double *phiFace, const double *phi0Cell, const double *phi0Face) {
  return guardedEq(e, [&] {
    if (!uFace || !u0Face || !phi0Cell) fail(PHASE_HIP_EINVAL, "fv::div needs u, u0 (faces) and phi0 (cells)");
    phase_hip_mesh *m = e->mesh;
    PH_CHECK(hipSetDevice(m->device));
    byComponents(e->ncomp, [&](auto nc) {
      hipLaunchKernelGGL((kEqDiv<decltype(nc)::value>), dim3(g256(m->nCells)), dim3(kRowBlock), rowLds(e->stride),
                         m->stream, meshDev(m), uFace, u0Face, theta, bcType, phiFace, phi0Cell, phi0Face, e->stride,
                         e->cols.p, e->vals.p, e->cnt.p, e->rhs.p, e->dErr.p);
    });
    PH_CHECK(hipGetLastError());
    fresh(e);
    checkEq(e, "fv::div");
  });
}

int phase_hip_eq_divc(phase_hip_equation *e, const double *uFace, const double *u0Face, double theta,
                      const int *bcType, const double *phiFace, const double *phi0Cell, const double *phi0Face) {
  return guardedEq(e, [&] {
    if (!uFace || !u0Face || !phi0Cell) fail(PHASE_HIP_EINVAL, "fv::divc needs u, u0 (faces) and phi0 (cells)");
    phase_hip_mesh *m = e->mesh;
    PH_CHECK(hipSetDevice(m->device));
    byComponents(e->ncomp, [&](auto nc) {
      hipLaunchKernelGGL((kEqDivc<decltype(nc)::value>), dim3(g256(m->nCells)), dim3(kRowBlock), rowLds(e->stride),
                         m->stream, meshDev(m), uFace, u0Face, theta, bcType, phiFace, phi0Cell, phi0Face, e->stride,
                         e->cols.p, e->vals.p, e->cnt.p, e->rhs.p, e->dErr.p);
    });
    PH_CHECK(hipGetLastError());
    fresh(e);
    checkEq(e, "fv::divc");
  });
}

int phase_hip_eq_dive(phase_hip_equation *e, const double *u0Face, const double *u1Face, double theta,
                      const int *bcType, const double *phi0Cell, const double *phi1Cell, const double *phi0Face,
                      const double *phi1Face) {
  return guardedEq(e, [&] {
    if (!u0Face || !u1Face || !phi0Cell || !phi1Cell || !phi0Face || !phi1Face)
      fail(PHASE_HIP_EINVAL, "fv::dive needs u0, u1, phi0, phi1 (cells and faces)");
    phase_hip_mesh *m = e->mesh;
    PH_CHECK(hipSetDevice(m->device));
    byComponents(e->ncomp, [&](auto nc) {
      hipLaunchKernelGGL((kEqDive<decltype(nc)::value>), dim3(g256(m->nCells)), dim3(kRowBlock), rowLds(e->stride),
                         m->stream, meshDev(m), u0Face, u1Face, theta, bcType, phi0Cell, phi1Cell, phi0Face,
                         phi1Face, e->stride, e->cols.p, e->vals.p, e->cnt.p, e->rhs.p, e->dErr.p);
    });
    PH_CHECK(hipGetLastError());
    fresh(e);
    checkEq(e, "fv::dive");
  });
}

int phase_hip_eq_div_grad(phase_hip_equation *e, const double *phiUFace, const double *gradUCell, const int *bcType,
                          const double *uFace) {
  return guardedEq(e, [&] {
    if (e->ncomp != 2) fail(PHASE_HIP_EINVAL, "fv::div(phiU, gradU, u) builds a Vector2D equation");
    if (!phiUFace || !gradUCell) fail(PHASE_HIP_EINVAL, "fv::div needs phiU (faces) and gradU (cells)");
    phase_hip_mesh *m = e->mesh;
    PH_CHECK(hipSetDevice(m->device));
    hipLaunchKernelGGL(kEqDivGrad, dim3(g256(m->nCells)), dim3(kRowBlock), rowLds(e->stride), m->stream, meshDev(m),
                       phiUFace, gradUCell, bcType, uFace, e->stride, e->cols.p, e->vals.p, e->cnt.p, e->rhs.p,
                       e->dErr.p);
    PH_CHECK(hipGetLastError());
    fresh(e);
    checkEq(e, "fv::div");
  });
}

int phase_hip_eq_cicsam_div(phase_hip_equation *e, const double *uFace, const double *beta, double theta,
                            const int *bcType, const double *gammaFace, const double *gamma0Cell,
                            const double *gamma0Face) {
  return guardedEq(e, [&] {
    if (e->ncomp != 1) fail(PHASE_HIP_EINVAL, "cicsam::div builds a scalar equation");
    if (!uFace || !beta || !gamma0Cell) fail(PHASE_HIP_EINVAL, "cicsam::div needs u, beta (faces) and gamma0 (cells)");
    phase_hip_mesh *m = e->mesh;
    PH_CHECK(hipSetDevice(m->device));
    hipLaunchKernelGGL(kEqCicsamDiv, dim3(g256(m->nCells)), dim3(kRowBlock), rowLds(e->stride), m->stream, meshDev(m),
                       uFace, beta, theta, bcType, gammaFace, gamma0Cell, gamma0Face, e->stride, e->cols.p,
                       e->vals.p, e->cnt.p, e->rhs.p, e->dErr.p);
    PH_CHECK(hipGetLastError());
    fresh(e);
    checkEq(e, "cicsam::div");
  });
}

int phase_hip_eq_add(phase_hip_equation *e, const phase_hip_equation *o, int sign) {
  return guardedEq(e, [&] {
    if (!o || o->rank != e->rank || o->stride != e->stride || o->mesh != e->mesh)
      fail(PHASE_HIP_EINVAL, "operands of += / -= must be equations of the same mesh and rank");
    phase_hip_mesh *m = e->mesh;
    PH_CHECK(hipSetDevice(m->device));
    hipLaunchKernelGGL(kEqMerge, dim3((unsigned)std::min(16384, (e->rank + kMergeBlock - 1) / kMergeBlock)),
                       dim3(kMergeBlock), mergeLds(e->stride), m->stream, e->rank, e->stride, sign >= 0 ? 1 : -1,
                       e->cols.p, e->vals.p, e->cnt.p, e->rhs.p, o->cols.p, o->vals.p, o->cnt.p, o->rhs.p, e->dErr.p);
    PH_CHECK(hipGetLastError());
    e->compact = true;
    checkEq(e, "CrsEquation::operator+=");
  });
}

int phase_hip_eq_copy(phase_hip_equation *dst, const phase_hip_equation *src) {
  return guardedEq(dst, [&] {
    if (!src || src->rank != dst->rank || src->stride != dst->stride)
      fail(PHASE_HIP_EINVAL, "copy needs equations of the same rank");
    hipStream_t st = dst->mesh->stream;
    const size_t slots = (size_t)dst->rank * dst->stride;
    PH_CHECK(hipMemcpyAsync(dst->cols.p, src->cols.p, slots * sizeof(int), hipMemcpyDeviceToDevice, st));
    PH_CHECK(hipMemcpyAsync(dst->vals.p, src->vals.p, slots * sizeof(double), hipMemcpyDeviceToDevice, st));
    PH_CHECK(hipMemcpyAsync(dst->cnt.p, src->cnt.p, dst->rank * sizeof(int), hipMemcpyDeviceToDevice, st));
    PH_CHECK(hipMemcpyAsync(dst->rhs.p, src->rhs.p, dst->rank * sizeof(double), hipMemcpyDeviceToDevice, st));
    dst->compact = src->compact;
  });
}

int phase_hip_eq_scale(phase_hip_equation *e, double s) {
  return guardedEq(e, [&] {
    hipLaunchKernelGGL(kEqScale, dim3(g256((long)e->rank * e->stride)), dim3(256), 0, e->mesh->stream, e->rank,
                       e->stride, s, e->vals.p, e->rhs.p);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_eq_scale_cells(phase_hip_equation *e, const double *field) {
  return guardedEq(e, [&] {
    if (!field) fail(PHASE_HIP_EINVAL, "null field");
    hipLaunchKernelGGL(kEqScaleCells, dim3(g256((long)e->rank * e->stride)), dim3(256), 0, e->mesh->stream, e->rank,
                       e->mesh->nCells, e->stride, field, e->vals.p, e->rhs.p);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_eq_remove_cells(phase_hip_equation *e, const int *cellMask) {
  return guardedEq(e, [&] {
    if (!cellMask) fail(PHASE_HIP_EINVAL, "null mask");
    hipLaunchKernelGGL(kEqRemoveCells, dim3(g256(e->rank)), dim3(256), 0, e->mesh->stream, e->rank,
                       e->mesh->nCells, e->stride, cellMask, e->cols.p, e->rhs.p);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_eq_sub_vector(phase_hip_equation *e, const double *v) {
  return guardedEq(e, [&] {
    if (!v) fail(PHASE_HIP_EINVAL, "null vector");
    hipLaunchKernelGGL(kEqSubRhs, dim3(g256(e->rank)), dim3(256), 0, e->mesh->stream, e->rank, v, 0., e->rhs.p);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_eq_eq_scalar(phase_hip_equation *e, double s) {
  return guardedEq(e, [&] {
    if (s == 0.) return;  // CrsEquation.cpp:299-303
    hipLaunchKernelGGL(kEqSubRhs, dim3(g256(e->rank)), dim3(256), 0, e->mesh->stream, e->rank, (const double *)nullptr,
                       s, e->rhs.p);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_eq_relax(phase_hip_equation *e, double alpha, const double *phi) {
  return guardedEq(e, [&] {
    if (!phi || !(alpha > 0.)) fail(PHASE_HIP_EINVAL, "relax needs alpha > 0 and the current field");
    hipLaunchKernelGGL(kEqRelax, dim3(g256(e->rank)), dim3(256), 0, e->mesh->stream, e->rank, e->stride, alpha, phi,
                       e->cols.p, e->vals.p, e->cnt.p, e->rhs.p);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_eq_export(phase_hip_equation *e, int *nslots, int *rowPtr, int *colInd, double *vals, double *rhs) {
  return guardedEq(e, [&] {
    if (!nslots) fail(PHASE_HIP_EINVAL, "nslots is required");
    hipStream_t st = e->mesh->stream;
    const size_t slots = (size_t)e->rank * e->stride;
    std::vector<int> c(slots), n(e->rank);
    std::vector<double> v(slots), r(e->rank);
    PH_CHECK(hipMemcpyAsync(c.data(), e->cols.p, slots * sizeof(int), hipMemcpyDeviceToHost, st));
    PH_CHECK(hipMemcpyAsync(v.data(), e->vals.p, slots * sizeof(double), hipMemcpyDeviceToHost, st));
    PH_CHECK(hipMemcpyAsync(n.data(), e->cnt.p, e->rank * sizeof(int), hipMemcpyDeviceToHost, st));
    PH_CHECK(hipMemcpyAsync(r.data(), e->rhs.p, e->rank * sizeof(double), hipMemcpyDeviceToHost, st));
    PH_CHECK(hipStreamSynchronize(st));
    // fresh rows: the reference's 5 slots (-1 = empty) or more when a row
    // grew; rebuilt rows: exactly their entries
    int total = 0;
    for (int i = 0; i < e->rank; ++i) total += e->compact ? n[i] : std::max(5, n[i]);
    if (!rowPtr) {
      *nslots = total;
      return;
    }
    if (*nslots < total) fail(PHASE_HIP_EINVAL, "output arrays too small");
    int w = 0;
    rowPtr[0] = 0;
    for (int i = 0; i < e->rank; ++i) {
      const int width = e->compact ? n[i] : std::max(5, n[i]);
      for (int j = 0; j < width; ++j, ++w) {
        const bool used = j < n[i];
        colInd[w] = used ? c[(size_t)i * e->stride + j] : -1;
        vals[w] = used ? v[(size_t)i * e->stride + j] : 0.;
      }
      rowPtr[i + 1] = w;
      if (rhs) rhs[i] = r[i];
    }
    *nslots = total;
  });
}

int phase_hip_solver_set_equation(phase_hip_solver *s, const phase_hip_equation *e) {
  if (!s || !e) return PHASE_HIP_EINVAL;
  try {
    // scalar equations carry one row per cell: their centroids order the rows
    const bool scalar = e->ncomp == 1;
    solverSetFromRows(s, e->rank, e->stride, e->cols.p, e->vals.p, e->rhs.p, e->mesh->stream,
                      scalar ? e->mesh->dCC.p : nullptr, scalar ? e->mesh->iptr.data() : nullptr,
                      scalar ? e->mesh->inb.data() : nullptr);
    return PHASE_HIP_OK;
  } catch (const HipError &x) {
    s->err = x.msg;
    return x.code;
  } catch (const std::exception &x) {
    s->err = x.what();
    return PHASE_HIP_EINVAL;
  }
}

int phase_hip_field_src_div(phase_hip_mesh *m, const double *uFace, double *out) {
  return guardedM(m, [&] {
    if (!uFace || !out) fail(PHASE_HIP_EINVAL, "null field");
    PH_CHECK(hipSetDevice(m->device));
    hipLaunchKernelGGL(kSrcDiv, dim3(g256(m->nCells)), dim3(256), 0, m->stream, meshDev(m), uFace, out);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_field_src_src(phase_hip_mesh *m, int ncomp, const double *phiCell, double *out) {
  return guardedM(m, [&] {
    if (!phiCell || !out || (ncomp != 1 && ncomp != 2)) fail(PHASE_HIP_EINVAL, "bad field");
    PH_CHECK(hipSetDevice(m->device));
    hipLaunchKernelGGL(kSrcSrc, dim3(g256(m->nCells)), dim3(256), 0, m->stream, meshDev(m), ncomp, phiCell, out);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_field_grad(phase_hip_mesh *m, const double *phiCell, const double *phiFace, double *gradFace,
                         double *gradCell) {
  return guardedM(m, [&] {
    if (!phiCell || !phiFace || !gradFace || !gradCell) fail(PHASE_HIP_EINVAL, "null field");
    PH_CHECK(hipSetDevice(m->device));
    hipLaunchKernelGGL(kGradFaces, dim3(g256(m->nFaces)), dim3(256), 0, m->stream, m->nFaces, m->dFL.p, m->dFR.p,
                       m->dFaceD.p, phiCell, phiFace, gradFace);
    hipLaunchKernelGGL(kGradCells, dim3(g256(m->nCells)), dim3(256), 0, m->stream, meshDev(m), gradFace, gradCell);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_field_interpolate_faces(phase_hip_mesh *m, int ncomp, const double *phiCell, const int *bcType,
                                      double *phiFace) {
  return guardedM(m, [&] {
    if (!phiCell || !phiFace || (ncomp != 1 && ncomp != 2)) fail(PHASE_HIP_EINVAL, "bad field");
    PH_CHECK(hipSetDevice(m->device));
    byComponents(ncomp, [&](auto nc) {
      hipLaunchKernelGGL((kInterpFaces<decltype(nc)::value>), dim3(g256(m->nFaces)), dim3(256), 0, m->stream,
                         m->nFaces, m->dFL.p, m->dFR.p, m->dFaceW.p, m->dSf.p, bcType, phiCell, phiFace);
    });
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_field_face_to_cell(phase_hip_mesh *m, const double *faceVec, const double *cellWeight,
                                 const double *faceWeight, double *cellVec) {
  return guardedM(m, [&] {
    if (!faceVec || !cellVec) fail(PHASE_HIP_EINVAL, "null field");
    if (!cellWeight != !faceWeight) fail(PHASE_HIP_EINVAL, "faceToCell takes both weights or neither");
    PH_CHECK(hipSetDevice(m->device));
    hipLaunchKernelGGL(kFaceToCell, dim3(g256(m->nCells)), dim3(256), 0, m->stream, meshDev(m), faceVec, cellWeight,
                       faceWeight, cellVec);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_cicsam_weights(phase_hip_mesh *m, const double *uFace, const double *gammaCell,
                             const double *gradGammaCell, double timeStep, double *beta) {
  return guardedM(m, [&] {
    if (!uFace || !gammaCell || !gradGammaCell || !beta) fail(PHASE_HIP_EINVAL, "null field");
    PH_CHECK(hipSetDevice(m->device));
    const bool cells = courantPerCell(m->nCells, m->maxDeg);
    if (cells)
      hipLaunchKernelGGL(kCellCourant, dim3(g256(m->nCells)), dim3(256), 0, m->stream, meshDev(m), uFace, timeStep,
                         m->dCourant.p);
    hipLaunchKernelGGL(cells ? kCicsamWeights<true> : kCicsamWeights<false>, dim3(g256(m->nFaces)), dim3(256), 0,
                       m->stream, meshDev(m), m->nFaces, m->dFL.p, m->dFR.p, uFace, gammaCell, gradGammaCell, timeStep,
                       m->dCourant.p, beta);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_cicsam_momentum_flux(phase_hip_mesh *m, double rho1, double rho2, const double *uFace,
                                   const double *gammaCell, const double *gammaFace, const double *beta,
                                   double *rhoU) {
  return guardedM(m, [&] {
    if (!uFace || !gammaCell || !gammaFace || !beta || !rhoU) fail(PHASE_HIP_EINVAL, "null field");
    PH_CHECK(hipSetDevice(m->device));
    hipLaunchKernelGGL(kCicsamMomentumFlux, dim3(g256(m->nFaces)), dim3(256), 0, m->stream, meshDev(m), m->nFaces,
                       m->dFL.p, m->dFR.p, rho1, rho2, uFace, gammaCell, gammaFace, beta, rhoU);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_vof_properties(phase_hip_mesh *m, double rho1, double rho2, double mu1, double mu2,
                             const double *gammaCell, const double *gammaFace, double *rhoCell, double *rhoFace,
                             double *muCell, double *muFace) {
  return guardedM(m, [&] {
    if (!gammaCell || !gammaFace || !rhoCell || !rhoFace || !muCell || !muFace) fail(PHASE_HIP_EINVAL, "null field");
    if (!(mu1 > 0.) || !(mu2 > 0.)) fail(PHASE_HIP_EINVAL, "viscosities must be positive");
    PH_CHECK(hipSetDevice(m->device));
    hipLaunchKernelGGL(kVofProperties, dim3(g256(m->nCells)), dim3(256), 0, m->stream, m->nCells, rho1, rho2, mu1,
                       mu2, gammaCell, rhoCell, muCell);
    hipLaunchKernelGGL(kVofProperties, dim3(g256(m->nFaces)), dim3(256), 0, m->stream, m->nFaces, rho1, rho2, mu1,
                       mu2, gammaFace, rhoFace, muFace);
    PH_CHECK(hipGetLastError());
  });
}

int phase_hip_mesh_synchronize(phase_hip_mesh *m) {
  return guardedM(m, [&] { PH_CHECK(hipStreamSynchronize(m->stream)); });
}

}  // extern "C"
