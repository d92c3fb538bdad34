// Launchers shared by the solver and the multigrid hierarchy (included by the
// files that run solver kernels): grid sizes, the ILU(0) sweeps and
// factorisation of one ordering, and the lazily built FP64 / FP32 factors.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "solver.h"
#include "solver_kernels.h"

namespace phase {

inline int gridFor(long n, int block, int cap) {
  long g = (n + block - 1) / block;
  if (g < 1) g = 1;
  return (int)std::min<long>(g, cap);
}

constexpr int kElemCap = 4096;
constexpr int kRedCap = 1024;


// entries of phase_hip_solver_time_kernels / phase_hip_solver_kernel_bytes
constexpr int kTimedKernels = 22;

template <class T>
IluDev<T> iluDev(phase_hip_solver *s, T *fac) {
  IluDev<T> L;
  L.blocks = s->dBlocks.p;
  L.rows = s->dRows.p;
  L.lanes = s->dLanes.p;
  L.lCol = s->dLCol.p;
  L.uCol = s->dUCol.p;
  L.fac = fac;
  L.nb = s->ord.nBlocks;
  L.nLSlots = s->ord.nLSlots;
  L.nUSlots = s->ord.nUSlots;
  L.n = s->rank;
  return L;
}

// Scalars slot that is never set done: sweeps run outside a Krylov iteration
inline const Scalars *idleScalars(phase_hip_solver *s) { return s->dSc.p + 3; }

// Calls f with the ordering's sweep register width as a compile-time constant.
template <class F>
void byWidth(const phase_hip_solver *s, F &&f) {
  if (s->ord.regWidth == 4) f(std::integral_constant<int, 4>());
  else f(std::integral_constant<int, 8>());
}

// Calls f with the backward levels' form for a launch of `blocks` blocks (fused:
// kLUSolve) as a compile-time constant: out of registers, or through the LDS
// array.  An FP64 value is two crossbar words, which the register form moves for
// every lane at every level, the array only for the level's rows.  Once the
// launch fills the chip the crossbar counts, not the trip: of kLUSolve from some
// 4,000 blocks (15 wavefronts a CU) on -- 3,000 blocks of quads 5.80 us in
// registers, 6.48 through the array; 3,900 of triangles 8.18 and 7.90; 6,500
// 11.47 and 10.49; 19,500 24.59 and 22.77 --, of kUSolve, whose blocks are
// shorter, only while one generation of wavefronts (32 on each of 256 CUs) holds
// the whole launch: 4,500 blocks 6.74 and 6.68, 5,500 7.84 and 7.40, 6,500 8.58
// and 8.03, but 8,600 10.16 and 10.21, 15,000 of quads 12.05 and 12.99.  FP32
// moves one word: in registers always.  (The forward levels too: 6.35 us against
// 6.65 at 6,500 blocks in FP64.)
constexpr int kLdsFusedBlocks = 4096, kLdsBlocks = 5120, kOneGeneration = 32 * 256;
inline bool backwardInRegisters(bool fp64, bool fused, int blocks) {
  if (!fp64) return true;
  return fused ? blocks <= kLdsFusedBlocks : blocks <= kLdsBlocks || blocks > kOneGeneration;
}
template <class T, class F>
void byLevels(bool fused, int blocks, F &&f) {
  if constexpr (std::is_same<T, double>::value) {
    if (!backwardInRegisters(true, fused, blocks)) return f(std::false_type());
  }
  f(std::true_type());
}

// One colour's sweep launch each.
template <class T, int PRO, int W>
void launchLColour(phase_hip_solver *s, const IluDev<T> &L, int c, const Scalars *sc, const T *in, T *y, T *pv,
                   const T *r, const T *v, double *xs) {
  const int first = s->ord.colourPtr[c], blocks = s->ord.colourPtr[c + 1] - first;
  if (blocks < 1) return;
  hipLaunchKernelGGL((kLSolve<T, PRO, W>), dim3(blocks), dim3(64), 0, s->stream, L, first, sc, in, y, pv, r, v, xs);
}

template <class T, int W>
void launchUColour(phase_hip_solver *s, const IluDev<T> &L, int c, const Scalars *sc, const T *y, T *x,
                   const T *addFrom, T *addTo) {
  const int first = s->ord.colourPtr[c], blocks = s->ord.colourPtr[c + 1] - first;
  if (blocks < 1) return;
  byLevels<T>(false, blocks, [&](auto reg) {
    hipLaunchKernelGGL((kUSolve<T, W, decltype(reg)::value>), dim3(blocks), dim3(64), 0, s->stream, L, first, sc, y, x,
                       addFrom, addTo);
  });
}

template <class T, int PRO, int W>
void launchLUColour(phase_hip_solver *s, const IluDev<T> &L, int c, const Scalars *sc, const T *in, const T *y, T *pv,
                    const T *r, const T *v, T *out, double *xs, const T *addFrom, T *addTo) {
  const int first = s->ord.colourPtr[c], blocks = s->ord.colourPtr[c + 1] - first;
  if (blocks < 1) return;
  byLevels<T>(true, blocks, [&](auto reg) {
    hipLaunchKernelGGL((kLUSolve<T, PRO, W, decltype(reg)::value>), dim3(blocks), dim3(64), 0, s->stream, L, first, sc,
                       in, y, pv, r, v, out, xs, addFrom, addTo);
  });
}

// Sweep launchers: one launch per block colour (forward colours ascending,
// backward descending).
template <class T, int PRO>
void launchL(phase_hip_solver *s, const IluDev<T> &L, const Scalars *sc, const T *in, T *y, T *pv, const T *r,
             const T *v, double *xs = nullptr) {
  byWidth(s, [&](auto Wc) {
    constexpr int W = decltype(Wc)::value;
    for (int c = 0; c < s->ord.nColours; ++c) launchLColour<T, PRO, W>(s, L, c, sc, in, y, pv, r, v, xs);
  });
}

template <class T>
void launchU(phase_hip_solver *s, const IluDev<T> &L, const Scalars *sc, const T *y, T *x) {
  byWidth(s, [&](auto Wc) {
    constexpr int W = decltype(Wc)::value;
    for (int c = s->ord.nColours - 1; c >= 0; --c)
      launchUColour<T, W>(s, L, c, sc, y, x, (const T *)nullptr, (T *)nullptr);
  });
}

// out = U^{-1} L^{-1} (right-hand side formed by PRO); the last forward colour
// and the first backward colour run fused in one launch.  With addTo set,
// addTo = addFrom + out as well (row by row, in the launch that finishes it).
template <class T, int PRO>
void launchLU(phase_hip_solver *s, const IluDev<T> &L, const Scalars *sc, const T *in, T *y, T *pv, const T *r,
              const T *v, T *out, double *xs = nullptr, const T *addFrom = nullptr, T *addTo = nullptr) {
  const int C = s->ord.nColours;
  if (C < 1) return;
  byWidth(s, [&](auto Wc) {
    constexpr int W = decltype(Wc)::value;
    for (int c = 0; c + 1 < C; ++c) launchLColour<T, PRO, W>(s, L, c, sc, in, y, pv, r, v, xs);
    launchLUColour<T, PRO, W>(s, L, C - 1, sc, in, y, pv, r, v, out, xs, addFrom, addTo);
    for (int c = C - 2; c >= 0; --c) launchUColour<T, W>(s, L, c, sc, y, out, addFrom, addTo);
  });
}

template <class T>
void factorize(phase_hip_solver *s, DBuf<T> &fac) {
  const IluDev<T> L = iluDev<T>(s, fac.p);
  const std::vector<int> &cp = s->ord.colourPtr;
  const size_t lds = (size_t)s->facSlots * 64 * sizeof(T);
  for (int c = 0; c + 1 < (int)cp.size(); ++c)
    if (cp[c + 1] > cp[c])
      hipLaunchKernelGGL((kIluFactor<T>), dim3(cp[c + 1] - cp[c]), dim3(64), lds, s->stream, L, s->rank, s->dVals.p,
                         s->dFacSrc.p, s->dUpdPtr.p, s->dUpdSrc.p, s->dUpdDst.p, s->dErr.p, cp[c]);
  PH_CHECK(hipGetLastError());
}

inline int spmvGrid(phase_hip_solver *s) { return std::max(1, (s->ord.nSlices + 3) / 4); }


// The three scalar records (Krylov run, outer refinement, misc) to the host.
inline void pullScalars(phase_hip_solver *s) {
  PH_CHECK(hipMemcpyAsync(s->hSc, s->dSc.p, 3 * sizeof(Scalars), hipMemcpyDeviceToHost, s->stream));
  PH_CHECK(hipStreamSynchronize(s->stream));
}

// One value of the device to the host.  By way of the handle's pinned memory: a
// copy to a variable on the stack is staged by the runtime and takes the host
// about twice as long.
template <class T>
T pullValue(phase_hip_solver *s, const T *d) {
  static_assert(sizeof(T) <= sizeof(Scalars), "the slot behind the three records");
  PH_CHECK(hipMemcpyAsync(s->hSc + 3, d, sizeof(T), hipMemcpyDeviceToHost, s->stream));
  PH_CHECK(hipStreamSynchronize(s->stream));
  return *reinterpret_cast<const T *>(s->hSc + 3);
}

inline void checkDeviceErr(phase_hip_solver *s) {
  const int e = pullValue(s, s->dErr.p);
  if (e & 2) {
    PH_CHECK(hipMemsetAsync(s->dErr.p, 0, sizeof(int), s->stream));
    fail(PHASE_HIP_EBREAKDOWN, "zero pivot in ILU(0) factorisation");
  }
}

// fac = [L slots | U slots | diagonal (n) | inverse diagonal (n)]
inline size_t facSize(const phase_hip_solver *s) { return (size_t)s->ord.nLSlots + s->ord.nUSlots + 2 * (size_t)s->rank; }

inline void ensureFactor64(phase_hip_solver *s) {
  if (s->fac64Valid) return;
  s->dFac64.alloc(facSize(s));
  factorize<double>(s, s->dFac64);
  checkDeviceErr(s);
  s->fac64Valid = true;
}

inline void ensureSingle(phase_hip_solver *s) {
  if (!s->sell32Valid) {
    s->dSell32.alloc(s->dSell64.n);
    const int m = (int)s->dSell64.n;
    hipLaunchKernelGGL((kConvert<double, float>), dim3(gridFor(m, 256, kElemCap)), dim3(256), 0, s->stream,
                       m, s->dSell64.p, s->dSell32.p);
    s->sell32Valid = true;
  }
  if (!s->fac32Valid) {
    // factor in FP64, store and apply in FP32: rounding the finished factor
    // keeps the FP64 pivots, where an FP32 factorisation of an ill-conditioned
    // matrix loses them to cancellation
    ensureFactor64(s);
    const int m = (int)s->dFac64.n;
    s->dFac32.alloc(m);
    hipLaunchKernelGGL((kConvert<double, float>), dim3(gridFor(m, 256, kElemCap)), dim3(256), 0, s->stream, m,
                       s->dFac64.p, s->dFac32.p);
    PH_CHECK(hipGetLastError());
    s->fac32Valid = true;
  }
}


}  // namespace phase
