// CPU emulation of the device solver's layout and kernels (test-only).
//
// Builds the product's ordering (phase_amd/csrc/ordering.cpp) and replays the
// SELL-64 SpMV, the ILU(0) factorisation (a block's entries in its LDS array) and
// both triangular sweeps (in-block levels out of registers and through the LDS
// array) as the gfx950 kernels in solver_kernels.h do -- block by block in launch
// order, level by level inside a block -- while checking every array index,
// those into LDS included, against its bounds and every dependency against the
// schedule (a predecessor block must already be finished, an in-block dependency
// must sit at a lower level).
// The results are compared with the oracle by tests/test_ordering_emul.py.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../phase_amd/csrc/phase_internal.h"

using namespace phase;

namespace {
struct Bad {
  std::string msg;
};
#define REQ(c, m) \
  do {            \
    if (!(c)) throw Bad{m}; \
  } while (0)
}  // namespace

namespace {
bool gBlockJacobi = false;
}
// The next emul_run builds block-Jacobi orderings (one colour, factor of the
// block-diagonal part).
extern "C" void emul_set_block_jacobi(int on) { gBlockJacobi = on != 0; }

extern "C" int emul_run(int n, const int *rowPtr, const int *colInd, const double *vals, int blockRows,
                        int *perm, int *facRowPtr, int *facCol, double *facVal, int cap, const double *rhsIn,
                        double *y, double *x, const double *xin, double *spmvOut, int *info, char *err,
                        int errLen, const double *cellXY) {
  try {
    Ordering o;
    try {
      buildOrdering(o, n, rowPtr, colInd, blockRows, cellXY, gBlockJacobi);
    } catch (const HipError &e) {
      throw Bad{e.msg};
    }
    const int nslots = rowPtr[n];
    const int nb = o.nBlocks;
    info[0] = nb;
    info[1] = o.nColours;
    info[2] = o.nLSlots;
    info[3] = o.nUSlots;
    int maxLev = 0, maxULev = 0;
    for (auto &B : o.blocks) {
      maxLev = std::max(maxLev, B.nLev);
      maxULev = std::max(maxULev, B.nULev);
    }
    info[4] = maxLev;
    info[5] = maxULev;
    int maxIn = 0;  // widest in-block L / in-block U / off-block U count of a row
    for (const RowInfo &r : o.rows) maxIn = std::max({maxIn, r.nL - r.nLoff, (int)r.nUin, r.nU - r.nUin});
    info[6] = maxIn;
    for (int k = 0; k < n; ++k) perm[k] = o.perm[k];
    // --- value gathers (kGather)
    const size_t nSell = o.sellCol.size();
    REQ(o.sellSrc.size() == nSell, "sellSrc size");
    std::vector<double> sell(nSell);
    for (size_t i = 0; i < nSell; ++i) {
      REQ(o.sellSrc[i] < nslots, "sellSrc out of range");
      sell[i] = o.sellSrc[i] >= 0 ? vals[o.sellSrc[i]] : 0.;
    }
    const size_t nFac = (size_t)o.nLSlots + o.nUSlots + n;
    REQ(o.facSrc.size() == nFac, "facSrc size");
    for (size_t i = 0; i < nFac; ++i) REQ(o.facSrc[i] < nslots, "facSrc out of range");
    std::vector<double> fac(nFac, NAN);  // written by the factorisation only
    // --- SpMV (kSpmv)
    REQ((int)o.sliceOff.size() == o.nSlices + 1, "sliceOff size");
    for (int k = 0; k < n; ++k) {
      int s = k / 64, lane = k % 64;
      int off = o.sliceOff[s], K = (o.sliceOff[s + 1] - off) / 64;
      REQ((o.sliceOff[s + 1] - off) % 64 == 0, "slice not a multiple of 64");
      double acc = 0.;
      for (int e = 0; e < K; ++e) {
        size_t idx = off + e * 64 + lane;
        REQ(idx < nSell, "sell index out of range");
        int c = o.sellCol[idx];
        REQ(c < n, "sell column out of range");
        if (c >= 0) acc = std::fma(sell[idx], xin[c], acc);
      }
      spmvOut[k] = acc;
    }
    const int dbase = o.nLSlots + o.nUSlots;
    auto lslot = [&](const BlockInfo &B, int e, int lane) {
      int s = B.lOff + e * 64 + lane;
      REQ(s >= 0 && s < o.nLSlots, "L slot out of range");
      return s;
    };
    auto uslot = [&](const BlockInfo &B, int e, int lane) {
      int s = B.uOff + e * 64 + lane;
      REQ(s >= 0 && s < o.nUSlots, "U slot out of range");
      return s;
    };
    // per-colour launches: every predecessor block of a block lies in an
    // earlier colour, every successor in a later one
    REQ((int)o.colourPtr.size() == o.nColours + 1 && o.colourPtr[0] == 0 && o.colourPtr[o.nColours] == nb,
        "colourPtr");
    std::vector<int> colourOf(nb, -1);
    for (int c = 0; c < o.nColours; ++c)
      for (int b = o.colourPtr[c]; b < o.colourPtr[c + 1]; ++b) colourOf[b] = c;
    for (int b = 0; b < nb; ++b) {
      const BlockInfo &B = o.blocks[b];
      for (int q = B.predBeg; q < B.predEnd; ++q) REQ(colourOf[o.pred[q]] < colourOf[b], "pred not in an earlier colour");
      for (int q = B.succBeg; q < B.succEnd; ++q) REQ(colourOf[o.succ[q]] > colourOf[b], "succ not in a later colour");
    }
    // per-lane sweep records agree with the row records
    REQ(o.lanes.size() == (size_t)nb * 64, "lane record count");
    for (int b = 0; b < nb; ++b) {
      const BlockInfo &B = o.blocks[b];
      for (int lane = 0; lane < 64; ++lane) {
        const LaneRec &L = o.lanes[(size_t)b * 64 + lane];
        if (lane >= B.nRows) {
          REQ(L.row == -1, "idle lane with a row");
          continue;
        }
        const int k = B.rowStart + lane;
        const RowInfo &ri = o.rows[k];
        REQ(L.row == k, "lane row");
        REQ((int)(L.info & 15u) == ri.nL - ri.nLoff && (int)((L.info >> 4) & 63u) == ri.nLoff &&
                (int)((L.info >> 10) & 15u) == ri.nUin && (int)((L.info >> 14) & 15u) == ri.nU - ri.nUin &&
                (int)((L.info >> 18) & 63u) == ri.lev && (int)((L.info >> 24) & 63u) == ri.ulev,
            "lane info packing");
      }
    }
    std::vector<char> doneBlk(nb, 0), rowDone(n, 0);
    // --- factorisation (kIluFactor), blocks in launch order: a block's entries in
    // its LDS array, the pivots and first update sources of earlier blocks loaded
    // before the levels, the results and the inverse diagonal stored at the end
    int facSlots = 1;
    for (const BlockInfo &B : o.blocks) facSlots = std::max(facSlots, B.kL + B.kU + 1);
    REQ((size_t)facSlots * 64 * sizeof(double) <= 65536, "factor block beyond the LDS of a launch");
    for (int b = 0; b < nb; ++b) {
      const BlockInfo &B = o.blocks[b];
      REQ(B.nRows >= 1 && B.nRows <= 64, "block size");
      REQ(B.predEnd - B.predBeg <= 64, "too many preds");
      for (int q = B.predBeg; q < B.predEnd; ++q) {
        REQ(o.pred[q] < b, "pred block not earlier");
        REQ(doneBlk[o.pred[q]], "pred block not finished");
      }
      std::vector<double> lds((size_t)facSlots * 64, NAN);
      auto f = [&](int at) -> double & {
        REQ(at >= 0 && (size_t)at < lds.size(), "LDS index");
        return lds[at];
      };
      const int uFirst = o.nLSlots + B.uOff, nSlot = B.kL + B.kU;
      auto place = [&](int s) {
        if (s < o.nLSlots) return s - B.lOff;
        if (s < dbase) return s >= uFirst && s < uFirst + (B.kU << 6) ? (B.kL << 6) + s - uFirst : -1;
        return s - dbase >= B.rowStart && s - dbase < B.rowStart + B.nRows
                   ? ((B.kL + B.kU) << 6) + s - dbase - B.rowStart
                   : -1;
      };
      // a value of an earlier block, read from memory
      auto earlier = [&](int s) {
        REQ(s >= o.nLSlots && (size_t)s < nFac, "off-block factor index");
        if (s >= dbase) REQ(s - dbase < B.rowStart && rowDone[s - dbase], "off-block pivot not final");
        else REQ(s < uFirst, "off-block update source not in an earlier block");
        return fac[s];
      };
      // a value of this block: its row must sit at a lower level
      auto inBlock = [&](int at, int lev) {
        REQ((at & 63) < B.nRows && o.rows[B.rowStart + (at & 63)].lev < lev, "in-block value not at a lower level");
        return f(at);
      };
      for (int lane = 0; lane < 64; ++lane) {
        const bool act = lane < B.nRows;
        for (int e = 0; e <= nSlot; ++e) {
          int src = -1;
          if (e < B.kL) src = o.facSrc[lslot(B, e, lane)];
          else if (e < nSlot) src = o.facSrc[o.nLSlots + uslot(B, e - B.kL, lane)];
          else if (act) src = o.facSrc[dbase + B.rowStart + lane];
          f((e << 6) + lane) = src >= 0 ? vals[src] : 0.;
        }
      }
      constexpr int kFacW = 4;
      struct Ahead {
        double pv[kFacW], sv[kFacW][2];
      };
      std::vector<Ahead> ahead(64);
      for (int lane = 0; lane < B.nRows; ++lane) {
        const int nL = o.rows[B.rowStart + lane].nL;
        for (int e = 0; e < kFacW && e < nL; ++e) {
          const int s = lslot(B, e, lane), p = dbase + o.lCol[s];
          ahead[lane].pv[e] = place(p) < 0 ? earlier(p) : NAN;
          for (int u = 0; u < 2; ++u) {
            ahead[lane].sv[e][u] = NAN;
            if (o.updPtr[s] + u < o.updPtr[s + 1] && place(o.updSrc[o.updPtr[s] + u]) < 0)
              ahead[lane].sv[e][u] = earlier(o.updSrc[o.updPtr[s] + u]);
          }
        }
      }
      for (int lev = 0; lev < B.nLev; ++lev) {
        for (int lane = 0; lane < B.nRows; ++lane) {
          const int row = B.rowStart + lane;
          const RowInfo &ri = o.rows[row];
          if (ri.lev != lev) continue;
          for (int e = 0; e < ri.nL; ++e) {
            const int s = lslot(B, e, lane);
            const int k = o.lCol[s];
            REQ(k >= 0 && k < row, "L column not below diagonal");
            if (e < ri.nLoff) REQ(k < B.rowStart, "off-block L entry inside block");
            else REQ(k >= B.rowStart, "in-block L entry outside block");
            const int pAt = place(dbase + k);
            const double piv = pAt >= 0 ? inBlock(pAt, lev) : e < kFacW ? ahead[lane].pv[e] : earlier(dbase + k);
            const double lik = f((e << 6) + lane) / piv;
            f((e << 6) + lane) = lik;
            REQ(o.updPtr[s] <= o.updPtr[s + 1], "updPtr");
            for (int u = o.updPtr[s]; u < o.updPtr[s + 1]; ++u) {
              const int n0 = u - o.updPtr[s], from = place(o.updSrc[u]), to = place(o.updDst[u]);
              REQ(o.updSrc[u] >= o.nLSlots && o.updSrc[u] < dbase, "update source not a U entry");
              REQ((to & 63) == lane, "update of another row");
              const double src = from >= 0               ? inBlock(from, lev)
                                 : e < kFacW && n0 < 2 ? ahead[lane].sv[e][n0]
                                                         : earlier(o.updSrc[u]);
              f(to) = std::fma(-lik, src, f(to));
            }
          }
          rowDone[row] = 1;
        }
      }
      for (int lane = 0; lane < 64; ++lane) {
        for (int e = 0; e < B.kL; ++e) fac[lslot(B, e, lane)] = f((e << 6) + lane);
        for (int e = 0; e < B.kU; ++e) fac[o.nLSlots + uslot(B, e, lane)] = f(((B.kL + e) << 6) + lane);
        if (lane < B.nRows) fac[dbase + B.rowStart + lane] = f((nSlot << 6) + lane);
      }
      for (int lane = 0; lane < B.nRows; ++lane) REQ(rowDone[B.rowStart + lane], "row left unprocessed");
      doneBlk[b] = 1;
    }
    // export factor (solver order, sorted columns)
    int w = 0;
    facRowPtr[0] = 0;
    for (int b = 0; b < nb; ++b) {
      const BlockInfo &B = o.blocks[b];
      for (int lane = 0; lane < B.nRows; ++lane) {
        const int k = B.rowStart + lane;
        const RowInfo &ri = o.rows[k];
        REQ(w + ri.nL + ri.nU + 1 <= cap, "factor capacity");
        for (int e = 0; e < ri.nL; ++e) { int s = lslot(B, e, lane); facCol[w] = o.lCol[s]; facVal[w++] = fac[s]; }
        facCol[w] = k;
        facVal[w++] = fac[dbase + k];
        for (int e = 0; e < ri.nU; ++e) {
          int s = uslot(B, e, lane);
          facCol[w] = o.uCol[s];
          facVal[w++] = fac[o.nLSlots + s];
        }
        facRowPtr[k + 1] = w;
      }
    }
    // --- forward sweep (kLSolve)
    std::fill(doneBlk.begin(), doneBlk.end(), 0);
    std::fill(rowDone.begin(), rowDone.end(), 0);
    for (int b = 0; b < nb; ++b) {
      const BlockInfo &B = o.blocks[b];
      for (int q = B.predBeg; q < B.predEnd; ++q) REQ(doneBlk[o.pred[q]], "fwd pred not finished");
      std::vector<double> acc(64, 0.), lds(64, 0.);
      for (int lane = 0; lane < B.nRows; ++lane) {
        const int row = B.rowStart + lane;
        const RowInfo &ri = o.rows[row];
        acc[lane] = rhsIn[row];
        for (int e = 0; e < ri.nLoff; ++e) {
          const int s = lslot(B, e, lane);
          REQ(rowDone[o.lCol[s]], "fwd off-block value not ready");
          acc[lane] = std::fma(-fac[s], y[o.lCol[s]], acc[lane]);
        }
      }
      // in-block levels: out of registers, every lane forming its row again at each
      // level from the others' values of the level before (__shfl), or through the
      // LDS array where a row is wider than the registers
      int most = 0;
      for (int lane = 0; lane < B.nRows; ++lane)
        most = std::max(most, o.rows[B.rowStart + lane].nL - o.rows[B.rowStart + lane].nLoff);
      auto entry = [&](int lane, int e, double v, auto &&value) {
        const int s = lslot(B, e, lane), li = o.lCol[s] - B.rowStart;
        REQ(li >= 0 && li < lane, "fwd in-block column");
        return std::fma(-fac[s], value(li), v);
      };
      if (most > o.regWidth) {
        for (int lev = 0; lev < B.nLev; ++lev)
          for (int lane = 0; lane < B.nRows; ++lane) {
            const RowInfo &ri = o.rows[B.rowStart + lane];
            if (ri.lev != lev) continue;
            for (int e = ri.nLoff; e < ri.nL; ++e)
              acc[lane] = entry(lane, e, acc[lane], [&](int li) {
                REQ(o.rows[B.rowStart + li].lev < lev, "fwd in-block value not ready");
                return lds[li];
              });
            lds[lane] = acc[lane];
          }
      } else {
        lds = acc;  // rows of level 0 are final
        for (int lev = 1; lev < B.nLev; ++lev) {
          const std::vector<double> before = lds;
          for (int lane = 0; lane < B.nRows; ++lane) {
            const RowInfo &ri = o.rows[B.rowStart + lane];
            double v = acc[lane];
            for (int e = ri.nLoff; e < ri.nL; ++e) v = entry(lane, e, v, [&](int li) { return before[li]; });
            REQ(ri.lev >= lev || v == lds[lane], "fwd row changed after its level");
            lds[lane] = v;
          }
        }
      }
      for (int lane = 0; lane < B.nRows; ++lane) {
        y[B.rowStart + lane] = lds[lane];
        rowDone[B.rowStart + lane] = 1;
      }
      doneBlk[b] = 1;
    }
    // --- backward sweep (kUSolve), blocks in reverse
    std::fill(doneBlk.begin(), doneBlk.end(), 0);
    std::fill(rowDone.begin(), rowDone.end(), 0);
    for (int t = 0; t < nb; ++t) {
      const int b = nb - 1 - t;
      const BlockInfo &B = o.blocks[b];
      for (int q = B.succBeg; q < B.succEnd; ++q) {
        REQ(o.succ[q] > b, "succ block not later");
        REQ(doneBlk[o.succ[q]], "bwd succ not finished");
      }
      std::vector<double> acc(64, 0.), lds(64, 0.), soff(64, 0.);
      for (int lane = 0; lane < B.nRows; ++lane) {
        const int row = B.rowStart + lane;
        const RowInfo &ri = o.rows[row];
        acc[lane] = y[row];
        // later-block terms: one sum, formed before the levels (kUSolve)
        REQ(ri.nU - ri.nUin <= 15, "too many off-block U entries");
        for (int e = ri.nUin; e < ri.nU; ++e) {
          const int s = uslot(B, e, lane);
          REQ(o.uCol[s] >= B.rowStart + B.nRows && rowDone[o.uCol[s]], "bwd off-block value not ready");
          soff[lane] = std::fma(fac[o.nLSlots + s], x[o.uCol[s]], soff[lane]);
        }
      }
      int most = 0;
      for (int lane = 0; lane < B.nRows; ++lane) most = std::max(most, (int)o.rows[B.rowStart + lane].nUin);
      auto solve = [&](int lane, double v, auto &&value) {
        const int row = B.rowStart + lane;
        for (int e = 0; e < o.rows[row].nUin; ++e) {
          const int s = uslot(B, e, lane), li = o.uCol[s] - B.rowStart;
          REQ(li > lane && li < B.nRows, "bwd in-block column");
          v = std::fma(-fac[o.nLSlots + s], value(li), v);
        }
        return (v - soff[lane]) * (1.0 / fac[dbase + row]);
      };
      // through the LDS array: wide rows, and FP64 launches that fill the chip
      for (int lev = 0; lev < B.nULev; ++lev)
        for (int lane = 0; lane < B.nRows; ++lane) {
          if (o.rows[B.rowStart + lane].ulev != lev) continue;
          lds[lane] = solve(lane, acc[lane], [&](int li) {
            REQ(o.rows[B.rowStart + li].ulev < lev, "bwd in-block value not ready");
            return lds[li];
          });
        }
      if (most <= o.regWidth) {  // out of registers: the same bits
        std::vector<double> reg(64, 0.);
        for (int lane = 0; lane < B.nRows; ++lane)
          reg[lane] = (acc[lane] - soff[lane]) * (1.0 / fac[dbase + B.rowStart + lane]);
        for (int lev = 1; lev < B.nULev; ++lev) {
          const std::vector<double> before = reg;
          for (int lane = 0; lane < B.nRows; ++lane)
            reg[lane] = solve(lane, acc[lane], [&](int li) { return before[li]; });
        }
        for (int lane = 0; lane < B.nRows; ++lane) REQ(reg[lane] == lds[lane], "bwd forms differ");
      }
      for (int lane = 0; lane < B.nRows; ++lane) {
        x[B.rowStart + lane] = lds[lane];
        rowDone[B.rowStart + lane] = 1;
      }
      doneBlk[b] = 1;
    }
    return 0;
  } catch (const Bad &e) {
    std::snprintf(err, errLen, "%s", e.msg.c_str());
    return 1;
  }
}

// Aggregation hierarchy of the multigrid preconditioner, built with the
// product's host code (buildOrdering per level, buildCoarse between levels)
// until a level has at most denseMax rows.  Writes, per level l < last: n,
// perm[n], the aggregate count na, aggPtr[na + 1], then the coarse pattern
// rowPtr[na + 1], nnz, colInd[nnz], galPtr[nnz + 1], galSrc[galPtr[nnz]];
// the file ends with the last level's n and a 0.  All int32.
extern "C" int emul_hierarchy(int n, const int *rowPtr, const int *colInd, const double *cellXY, int fineRows,
                              int coarseRows, int denseMax, const char *outPath, char *err, int errLen) {
  try {
    FILE *f = std::fopen(outPath, "wb");
    REQ(f != nullptr, "cannot open output");
    auto put = [&](const int *p, size_t k) { std::fwrite(p, sizeof(int), k, f); };
    std::vector<int> rp(rowPtr, rowPtr + n + 1), ci(colInd, colInd + rowPtr[n]);
    std::vector<double> xy;
    if (cellXY) xy.assign(cellXY, cellXY + 2 * (size_t)n);
    int level = 0;
    while (n > denseMax) {
      Ordering o;
      CoarseLevel c;
      try {
        buildOrdering(o, n, rp.data(), ci.data(), level == 0 ? fineRows : coarseRows, xy.empty() ? nullptr : xy.data());
        buildCoarse(o, xy.empty() ? nullptr : xy.data(), c);
      } catch (const HipError &e) {
        std::fclose(f);
        throw Bad{"level " + std::to_string(level) + ": " + e.msg};
      }
      REQ(c.n < n, "aggregation did not coarsen");
      // every finer compact entry lands in exactly one coarse slot
      std::vector<int> seen(rp[n], 0);
      for (int s : c.galSrc) {
        REQ(s >= 0 && s < rp[n] && ci[s] >= 0, "Galerkin source out of range");
        ++seen[s];
      }
      for (int s = 0; s < rp[n]; ++s) REQ(seen[s] == (ci[s] >= 0 ? 1 : 0), "Galerkin map does not cover the entries once");
      put(&n, 1);
      put(o.perm.data(), n);
      const int na = c.n;
      put(&na, 1);
      put(o.aggPtr.data(), na + 1);
      put(c.rowPtr.data(), na + 1);
      const int nnz = (int)c.colInd.size();
      put(&nnz, 1);
      put(c.colInd.data(), nnz);
      put(c.galPtr.data(), nnz + 1);
      put(c.galSrc.data(), c.galSrc.size());
      n = na;
      rp = c.rowPtr;
      ci = c.colInd;
      xy = c.xy;
      ++level;
    }
    put(&n, 1);
    const int zero = 0;
    put(&zero, 1);
    std::fclose(f);
    return level;
  } catch (const Bad &b) {
    std::snprintf(err, errLen, "%s", b.msg.c_str());
    return -1;
  }
}

// The product's rule for the Krylov iterations queued between host checks.
extern "C" int emul_next_chunk(double rrLast, double rr, double tol2, int itLast, int it, int cg, int chunk) {
  return nextChunk(rrLast, rr, tol2, itLast, it, cg != 0, chunk);
}
