// Device-resident unstructured 2D mesh shared by the assembly, operator and
// field kernels: topology in the reference's first-encounter face order
// (FiniteVolumeGrid2D.cpp:20-35, 84-114, 396-418) and geometry computed on the
// device (Cell.cpp:8-29, Face.cpp:9-18, CellLink.cpp:8, InteriorLink.cpp:9,
// BoundaryLink.cpp:8).
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "phase_internal.h"

struct phase_hip_mesh {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  int nNodes = 0, nCells = 0, nFaces = 0, nInterior = 0, nBoundary = 0;
  int maxDeg = 0;  // most interior links of one cell
  bool repeated = false;  // a cell meets a neighbour (or itself) over more than one face
  std::vector<int> fNode1, fNode2, fL, fR;
  std::vector<int> iptr, iface, inb, bptr, bface;
  phase::DBuf<double> dXY, dVol, dCC, dFC, dSf;  // vectors interleaved (x, y)
  phase::DBuf<int> dCptr, dCind, dFNode1, dFNode2, dFL, dFR;
  phase::DBuf<int> dIptr, dIface, dInb, dBptr, dBface;
  phase::DBuf<double> dIDot, dIMs, dBDot, dBMs;  // per link: dot(r, Sf_out), |r|^2
  phase::DBuf<int> dIfaceS, dBfaceS;  // per link: the face, kFlip set where Sf points into the cell
  phase::DBuf<double> dFaceD, dFaceW;  // per face: r (interleaved), and the left cell's distance weight
  phase::DBuf<double> dCourant;  // per cell: work space of the CICSAM weights (courantPerCell)
};

namespace phase {

struct Dv2 {
  double x, y;
};

// A vector of the interleaved fields as one 16-byte access (fields of callers
// are only known to be 8-byte aligned, which the hardware takes).
typedef double dv2_t __attribute__((ext_vector_type(2), aligned(8)));

// The CICSAM weights form a donor's Courant number per face, its faces read again
// for each, or first once per cell, a launch of its own: worth it on large meshes
// of triangles only (per face / per cell: 2,000 triangles 4.3 / 6.1 us, 130,000
// 11.3 / 13.2, 200,000 17.4 / 17.3, 400,000 31.8 / 28.0, one million 76.2 / 63.3;
// 16,384 quads 4.3 / 8.6, 500,000 30.5 / 33.2, one million 43.2 / 56.0, two million
// 103.8 / 104.9).
constexpr int kCourantCells = 1 << 18;
inline bool courantPerCell(int nCells, int maxDeg) { return maxDeg <= 3 && nCells > kCourantCells; }

// Link entries of dIfaceS / dBfaceS: the outward test of Face::outwardNorm is a
// property of the mesh, so the operators read its result with the face instead
// of the face centroid (16 bytes a link less).
constexpr int kFlip = (int)0x80000000;
__device__ __forceinline__ int faceOf(int link) { return link & ~kFlip; }
__device__ __forceinline__ Dv2 outwardOf(int link, const double *__restrict__ sf) {
  const dv2_t n = *(const dv2_t *)(sf + 2 * (size_t)faceOf(link));
  return link < 0 ? Dv2{-n.x, -n.y} : Dv2{n.x, n.y};
}

// Face::outwardNorm(point), Face.cpp:48-50: dot(centroid - point, normal) > 0
// ? normal : -normal
__device__ __forceinline__ Dv2 outward(Dv2 fc, Dv2 sf, Dv2 p) {
  const double dx = fc.x - p.x, dy = fc.y - p.y;
  return (dx * sf.x + dy * sf.y) > 0. ? sf : Dv2{-sf.x, -sf.y};
}

}  // namespace phase
