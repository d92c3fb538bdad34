// Learned correction for the pressure-correction solve: a message-passing
// network on the matrix graph, trained on (residual, correction) pairs the
// solver emits, applied between FP64 refinement passes.  No counterpart in the
// reference; the network is defined here and restated in FP64 by the oracle
// (oracle/gnn_oracle.py) that the gradient tests compare against.
//
// With d_i = |a_ii|, sd_i = sqrt(d_i), A_hat_ij = a_ij / (sd_i sd_j) (i != j):
//   X_i  = [r_i/(sd_i s), z_i sd_i / s, (sum_j a_ij)/a_ii, 1],  s = rms(r/sd),
//          z = ILU(0)^{-1} r
//   h0   = relu(X W_in + b_in)
//   h_l  = h_{l-1} + relu([h_{l-1}, A_hat h_{l-1}] Wsm + mean(h_{l-1}) Wg + b)
//   out  = h_L w_out + b_out,   correction e_i = out_i s / sd_i
// Loss on a captured pair (r, e*), with t_i = e*_i sd_i / s:
//   error objective (default):  1 - (out . t)^2 / (|out|^2 |t|^2)
//   residual objective:         1 - (q . r)^2 / (|q|^2 |r|^2),  q = A (out / sd),
//     the part of ||r||^2 the minimal-residual step leaves (A symmetric:
//     dloss/dout = (A dloss/dq) / sd).
//
// Dense layers run on BF16 MFMA (v_mfma_f32_16x16x32_bf16, FP32 accumulate):
// activations are stored as BF16 rows of 64 features, weights as BF16 copies
// of FP32 master parameters (Adam).  All reductions over rows go through
// per-block partials summed in a fixed order, so training is deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <string>

#include "gnn.h"
#include "solver.h"
#include "solver_kernels.h"

using namespace phase;

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int H = kGnnH;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

// Rows of a layer kernel's tile (16 per wavefront): one SELL-64 slice, so a
// tile's row offsets are a single pair of scalars.
constexpr int kTileRows = 64;
// Workgroups of the layer kernels.  Each takes a contiguous run of tiles (its
// weights stay in LDS and its sums in registers over the run), and every
// workgroup leaves one partial record: more of them cost the finishing sums,
// fewer leave the gathers with too few wavefronts in flight (a forward
// workgroup holds 18 KB of LDS, a backward one 46 KB: three per CU).  Twice as
// many of either: mean 10.0 us instead of 7.2, backward layer 91 us instead of
// 79 (200,000 rows).
constexpr int kFwdGroups = 1280;
constexpr int kBwdGroups = 768;
constexpr int kFinThreads = 1024;  // 64 columns x 16 slices of the partial records

struct Tiles {
  int n, per, groups;  // tiles, tiles per workgroup, workgroups
};
Tiles tilesFor(int n, int groups) {
  Tiles t;
  t.n = std::max(1, (n + kTileRows - 1) / kTileRows);
  t.per = (t.n + groups - 1) / groups;
  t.groups = (t.n + t.per - 1) / t.per;
  return t;
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

int gridFor1(long n) { return (int)std::max<long>(1, std::min<long>((n + kRedBlock - 1) / kRedBlock, 1024)); }

// ---------------------------------------------------------------- features
// sd_i = sqrt|a_ii| and the row-sum ratio from the SELL FP32 copy of A
__global__ void kGnnDiag(int n, const int *__restrict__ sliceOff, const int *__restrict__ col,
                         const float *__restrict__ val, float *__restrict__ sd, float *__restrict__ rs) {
  for (int row = blockIdx.x * blockDim.x + threadIdx.x; row < n; row += gridDim.x * blockDim.x) {
    const int s = row >> 6, lane = row & 63;
    const int o = sliceOff[s], K = (sliceOff[s + 1] - o) >> 6;
    float d = 0.f, sum = 0.f;
    for (int e = 0; e < K; ++e) {
      const int idx = o + (e << 6) + lane;
      const int c = col[idx];
      if (c < 0) continue;
      sum += val[idx];
      if (c == row) d = val[idx];
    }
    sd[row] = sqrtf(fabsf(d));
    rs[row] = d != 0.f ? sum / d : 0.f;
  }
}

// Graph weights in the SELL layout: a_ij / (sd_i sd_j), 0 for the diagonal
// and padding.  Formed once per matrix: the layers read them twelve times (each
// direction of each layer), and forming them in the layers cost a gather of
// sd and a division per entry, repeated by the lanes that share a row.
__global__ void kGnnWeights(int n, const int *__restrict__ sliceOff, const int *__restrict__ col,
                            const float *__restrict__ val, const float *__restrict__ sd, float *__restrict__ ah) {
  for (int row = blockIdx.x * blockDim.x + threadIdx.x; row < n; row += gridDim.x * blockDim.x) {
    const int s = row >> 6, lane = row & 63;
    const int o = sliceOff[s], K = (sliceOff[s + 1] - o) >> 6;
    for (int e = 0; e < K; ++e) {
      const int idx = o + (e << 6) + lane;
      const int c = col[idx];
      ah[idx] = (c < 0 || c == row) ? 0.f : val[idx] / (sd[row] * sd[c]);
    }
  }
}

// partials of sum_i (r_i / sd_i)^2; kGnnRmsFinish: scal[0] = rms
__global__ __launch_bounds__(kRedBlock) void kGnnRms(int n, const float *__restrict__ r, const float *__restrict__ sd,
                                                     double *partials) {
  double d[1] = {0.};
  for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
    const double v = (double)r[i] / (double)sd[i];
    d[0] += v * v;
  }
  blockPartials<1>(d, partials, blockIdx.x);
}

__global__ __launch_bounds__(kFinBlock) void kGnnRmsFinish(int n, const double *partials, int nb, double *scal) {
  double d[1];
  finishPartials<1, kFinBlock>(partials, nb, d);
  if (threadIdx.x == 0) {
    const double rms = sqrt(d[0] / (double)n);
    scal[0] = rms > 0. ? rms : 1.;
  }
}

__global__ void kGnnFeatures(int n, const float *__restrict__ r, const float *__restrict__ z,
                             const float *__restrict__ sd, const float *__restrict__ rowsum,
                             const double *__restrict__ scal, float *__restrict__ X) {
  const float inv = (float)(1.0 / scal[0]);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    X[4 * i + 0] = r[i] / sd[i] * inv;
    X[4 * i + 1] = z[i] * sd[i] * inv;
    X[4 * i + 2] = rowsum[i];
    X[4 * i + 3] = 1.f;
  }
}

// target t_i = e_i sd_i / s
__global__ void kGnnTarget(int n, const float *__restrict__ e, const float *__restrict__ sd,
                           const double *__restrict__ scal, float *__restrict__ t) {
  const float inv = (float)(1.0 / scal[0]);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) t[i] = e[i] * sd[i] * inv;
}

// ---------------------------------------------------------------- input layer
// h0 = relu(X W_in + b_in), eight features of a row per thread (its columns of
// W_in in registers), and the workgroup's column sums of h0 for the first
// layer's mean.
__global__ __launch_bounds__(256) void kGnnIn(int n, const float *__restrict__ X, const float *__restrict__ P,
                                              __bf16 *__restrict__ pre0, __bf16 *__restrict__ h0,
                                              float *__restrict__ colPart) {
  __shared__ float red[32][H + 1];
  const int f0 = 8 * (threadIdx.x & 7), q = threadIdx.x >> 3;
  float W[kGnnDin][8], b[8], sum[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
#pragma unroll
    for (int k = 0; k < kGnnDin; ++k) W[k][j] = P[k * H + f0 + j];
    b[j] = P[kGnnDin * H + f0 + j];
    sum[j] = 0.f;
  }
  for (int i = blockIdx.x * 32 + q; i < n; i += gridDim.x * 32) {
    const f32x4 x = *(const f32x4 *)&X[4 * (size_t)i];
    bf16x8 pv, hv;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float v = b[j];
#pragma unroll
      for (int k = 0; k < kGnnDin; ++k) v = fmaf(x[k], W[k][j], v);
      pv[j] = (__bf16)v;
      hv[j] = (__bf16)fmaxf(v, 0.f);
      sum[j] += (float)hv[j];
    }
    *(bf16x8 *)&pre0[(size_t)i * H + f0] = pv;
    *(bf16x8 *)&h0[(size_t)i * H + f0] = hv;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) red[q][f0 + j] = sum[j];
  __syncthreads();
  if (threadIdx.x < H) {
    float v = 0.f;
    for (int k = 0; k < 32; ++k) v += red[k][threadIdx.x];
    colPart[(size_t)blockIdx.x * H + threadIdx.x] = v;
  }
}

// Sum over the partial records of column `col` (thread f of 64 columns, slice
// q of 16): the calling block's 1024 threads leave the total in every thread
// with q == 0.  Records are `stride` floats apart; the order is fixed.
__device__ __forceinline__ float sumRecords(const float *__restrict__ partials, int records, size_t stride, int col,
                                            bool act, float (*red)[H]) {
  const int f = threadIdx.x & 63, q = threadIdx.x >> 6;
  float s = 0.f;
  for (int b0 = q; b0 < records; b0 += 16 * 8) {
    float t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = act && b0 + 16 * u < records ? partials[(size_t)(b0 + 16 * u) * stride + col] : 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) s += t[u];
  }
  red[q][f] = s;
  __syncthreads();
  float v = 0.f;
  if (q == 0)
    for (int k = 0; k < 16; ++k) v += red[k][f];
  __syncthreads();
  return v;
}

// g = column mean (from the partial column sums), c = b + g Wg
__global__ __launch_bounds__(kFinThreads) void kGnnMeanFold(int n, int records, const float *__restrict__ colPart,
                                                            const float *__restrict__ Wg, const float *__restrict__ b,
                                                            float *__restrict__ g, float *__restrict__ c) {
  __shared__ float red[16][H], gs[H];
  const int f = threadIdx.x & 63, q = threadIdx.x >> 6;
  const float s = sumRecords(colPart, records, H, f, true, red);
  if (q == 0) {
    gs[f] = s * (1.f / n);
    g[f] = gs[f];
  }
  __syncthreads();
  float v = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) v = fmaf(gs[4 * q + k], Wg[(4 * q + k) * H + f], v);
  red[q][f] = v;
  __syncthreads();
  if (q == 0) {
    float t = b[f];
    for (int k = 0; k < 16; ++k) t += red[k][f];
    c[f] = t;
  }
}

// ---------------------------------------------------------------- message-passing layer
// One wavefront per 16 rows of a 64-row tile: activations [h | A_hat h]
// (K = 128) against Wsm (LDS, stored [out col][k]).  The weights are the first
// MFMA operand and the activations the second, with the output features dealt
// to the weight rows so that a lane's accumulators are the features it holds as
// an operand (8 gq + 0..7 of each half of its row): h is not read again for the
// sum, and every access is 16 bytes of 64 contiguous ones.
// Writes agg, pre and h_new = h + relu(pre + c); LAST also forms
// out = h_new w_out + b_out, the other layers leave the workgroup's column
// sums of h_new for the next layer's mean.
// Bound by HBM: 4 x 128 B per row and the neighbours' rows out of L2.  At
// 200,000 triangles 36.9 us (57.4 us with the graph weights formed per lane and
// 2-byte accesses, and a separate 249 us column-sum kernel); with 8-byte
// accesses 47.4 us.  Six wavefronts per SIMD: with the weights held in registers
// over the tiles (196 of them, two wavefronts) 85 us.
template <bool LAST>
__global__ __launch_bounds__(256, 6) void kGnnLayerFwd(int n, int nTiles, int per, const __bf16 *__restrict__ h,
                                                    const int *__restrict__ sliceOff, const int *__restrict__ col,
                                                    const float *__restrict__ ah, const __bf16 *__restrict__ wT,
                                                    const float *__restrict__ c, __bf16 *__restrict__ agg,
                                                    __bf16 *__restrict__ pre, __bf16 *__restrict__ hNew,
                                                    float *__restrict__ colPart, const float *__restrict__ wo,
                                                    float *__restrict__ outp) {
  __shared__ __attribute__((aligned(16))) __bf16 W[H][128 + 8];
  __shared__ __attribute__((aligned(16))) float cs[H], wos[H];
  __shared__ float red[4][H];
  for (int t = threadIdx.x; t < H * 16; t += 256) {  // 64 cols x 16 chunks of 8
    const int o = t / 16, k8 = (t % 16) * 8;
    // row 16 t + m of W: feature 32 (t / 2) + 8 (m / 4) + 4 (t % 2) + m % 4
    const int at = 16 * (2 * (o >> 5) + ((o >> 2) & 1)) + 4 * ((o >> 3) & 3) + (o & 3);
    *(bf16x8 *)&W[at][k8] = *(const bf16x8 *)&wT[o * 128 + k8];
  }
  if (threadIdx.x < H) {
    cs[threadIdx.x] = c[threadIdx.x];
    if (LAST) wos[threadIdx.x] = wo[threadIdx.x];
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, gq = lane >> 4;
  const int group = xcdTile(blockIdx.x, gridDim.x);
  const int t1 = min(nTiles, (group + 1) * per);
  f32x4 sum[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) sum[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int tile = group * per; tile < t1; ++tile) {
    const int l = 16 * wave + (lane & 15), r = tile * kTileRows + l;
    const bool act = r < n;
    const int o = sliceOff[tile], K = act ? (sliceOff[tile + 1] - o) >> 6 : 0;
    const size_t at = (size_t)(act ? r : 0) * H;
    const bf16x8 zero = {};
    bf16x8 a[4];
    // one half of the features at a time (both halves' sums and neighbours'
    // rows together hold 40 more registers); the columns and weights come from
    // L1 the second time
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      asm volatile("" ::: "memory");
      const int f0 = 32 * kc + 8 * gq;
      a[kc] = act ? *(const bf16x8 *)&h[at + f0] : zero;
      float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      for (int e0 = 0; e0 < K; e0 += 4) {
        int cc[4];
        float w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bool in = e0 + q < K;
          const int idx = o + ((e0 + (in ? q : 0)) << 6) + l;
          cc[q] = col[idx];
          w[q] = in ? ah[idx] : 0.f;
        }
        bf16x8 x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = w[q] != 0.f ? *(const bf16x8 *)&h[(size_t)cc[q] * H + f0] : zero;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[j] = fmaf(w[q], (float)x[q][j], acc[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) a[2 + kc][j] = (__bf16)acc[j];
      if (act) *(bf16x8 *)&agg[at + f0] = a[2 + kc];
    }
    // lane: row r, half kc, features 32 kc + 8 gq + 4 u + v
    float dot = 0.f;
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      asm volatile("" ::: "memory");  // this half's weights are read here, not held
      const int f0 = 32 * kc + 8 * gq;
      bf16x8 pv, hv;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        f32x4 out = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c4 = 0; c4 < 4; ++c4)
          out = mfma(*(const bf16x8 *)&W[16 * (2 * kc + u) + (lane & 15)][32 * c4 + 8 * gq], a[c4], out);
        const f32x4 cv = *(const f32x4 *)&cs[f0 + 4 * u];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float p = out[v] + cv[v];
          const __bf16 hn = (__bf16)((float)a[kc][4 * u + v] + fmaxf(p, 0.f));
          pv[4 * u + v] = (__bf16)p;
          hv[4 * u + v] = hn;
          if (!LAST) sum[2 * kc + u][v] += act ? (float)hn : 0.f;
          if (LAST) dot = fmaf((float)hn, wos[f0 + 4 * u + v], dot);
        }
      }
      if (act) {
        *(bf16x8 *)&pre[at + f0] = pv;
        *(bf16x8 *)&hNew[at + f0] = hv;
      }
    }
    if (LAST) {
      dot += __shfl_xor(dot, 16, 64);
      dot += __shfl_xor(dot, 32, 64);
      if (act && gq == 0) outp[r] = dot + wo[H];
    }
  }
  if (!LAST) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float x = sum[t][v];
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) x += __shfl_xor(x, m, 64);
        if ((lane & 15) == 0) red[wave][32 * (t >> 1) + 8 * gq + 4 * (t & 1) + v] = x;
      }
    __syncthreads();
    if (threadIdx.x < H)
      colPart[(size_t)blockIdx.x * H + threadIdx.x] =
          red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
  }
}

// a = out.t, p = |out|^2, q = |t|^2 (partials); kGnnLossFinish: loss =
// 1 - a^2/(p q) -> scal[1..4]; scal[5] accumulates losses over training steps
__global__ __launch_bounds__(kRedBlock) void kGnnLossCos(int n, const float *__restrict__ out,
                                                         const float *__restrict__ t, double *partials) {
  double d[3] = {0., 0., 0.};
  for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
    const double o = out[i], ti = t[i];
    d[0] += o * ti;
    d[1] += o * o;
    d[2] += ti * ti;
  }
  blockPartials<3>(d, partials, blockIdx.x);
}

__global__ __launch_bounds__(kFinBlock) void kGnnLossFinish(const double *partials, int nb, double *scal) {
  double d[3];
  finishPartials<3, kFinBlock>(partials, nb, d);
  if (threadIdx.x == 0) {
    const double pq = d[1] * d[2];
    const double loss = pq > 0. ? 1.0 - d[0] * d[0] / pq : 1.0;
    scal[1] = loss;
    scal[2] = d[0];
    scal[3] = d[1];
    scal[4] = d[2];
    scal[5] += loss;
  }
}

// dout_i = 2a/(p q) (a out_i / p - t_i)
__global__ void kGnnDout(int n, const float *__restrict__ out, const float *__restrict__ t,
                         const double *__restrict__ scal, float *__restrict__ dout) {
  const double a = scal[2], p = scal[3], q = scal[4];
  const bool ok = p > 0. && q > 0.;
  const float c1 = ok ? (float)(2.0 * a / (p * q)) : 0.f, c2 = ok ? (float)(a / p) : 0.f;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    dout[i] = c1 * (c2 * out[i] - t[i]);
}

// residual objective: c = out / sd
__global__ void kGnnResC(int n, const float *__restrict__ out, const float *__restrict__ sd, float *__restrict__ c) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) c[i] = out[i] / sd[i];
}

// residual objective: dq_i = 2a/(p rr) (a q_i / p - r_i), a = q.r, p = |q|^2, rr = |r|^2
__global__ void kGnnResDq(int n, const float *__restrict__ q, const float *__restrict__ r,
                          const double *__restrict__ scal, float *__restrict__ dq) {
  const double a = scal[2], p = scal[3], rr = scal[4];
  const bool ok = p > 0. && rr > 0.;
  const float c1 = ok ? (float)(2.0 * a / (p * rr)) : 0.f, c2 = ok ? (float)(a / p) : 0.f;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) dq[i] = c1 * (c2 * q[i] - r[i]);
}

// residual objective: dout_i = g_i / sd_i (g = A dq)
__global__ void kGnnResDout(int n, const float *__restrict__ g, const float *__restrict__ sd,
                            float *__restrict__ dout) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) dout[i] = g[i] / sd[i];
}

// grad of w_out / b_out: per-workgroup partials of h^T dout and sum(dout),
// eight features of a row per thread
__global__ __launch_bounds__(256) void kGnnOutGrad(int n, const __bf16 *__restrict__ h, const float *__restrict__ dout,
                                                   float *__restrict__ partials) {
  __shared__ float red[32][H + 1];
  const int f0 = 8 * (threadIdx.x & 7), q = threadIdx.x >> 3;
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0}, accb = 0.f;
  for (int i = blockIdx.x * 32 + q; i < n; i += gridDim.x * 32) {
    const float d = dout[i];
    const bf16x8 hv = *(const bf16x8 *)&h[(size_t)i * H + f0];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = fmaf((float)hv[j], d, acc[j]);
    accb += d;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) red[q][f0 + j] = acc[j];
  if (f0 == 0) red[q][H] = accb;
  __syncthreads();
  if (threadIdx.x < H + 1) {
    float v = 0.f;
    for (int k = 0; k < 32; ++k) v += red[k][threadIdx.x];
    partials[(size_t)blockIdx.x * (H + 1) + threadIdx.x] = v;
  }
}

// ---------------------------------------------------------------- backward layer
// Rows of a feature, eight to a 16-byte chunk: chunk `chunk` (of 8) of feature
// f in a transposed tile of 64 rows.  Pitch 72 elements and the chunk index
// xored with f / 8 keep both the packed 4-byte writes (eight features of one
// row pair per instruction step) and the 16-byte reads (16 neighbouring
// features) free of bank conflicts.
constexpr int kTPitch = 72;
__device__ __forceinline__ int tileAt(int f, int chunk) { return f * kTPitch + ((chunk ^ ((f >> 3) & 7)) << 3); }

// Backward pass of one layer over the workgroup's tiles:
//   dh    = FIRST ? dout w_out^T : dhIn + gterm + A_hat^T daggIn   (A_hat symmetric)
//   dpre  = dh * (pre > 0)
//   dhOut = dh + dpre Ws^T, daggOut = dpre Wm^T                    (FP32)
//   partials of dWsm = [h | agg]^T dpre and db = column sums of dpre
// The combination with the layer above (dhIn, daggIn, gterm) is formed as it is
// read, and dpre stays in registers and LDS, so per row the kernel moves
// 11 x 128 B to and from HBM: pre, h and agg in BF16, dh in and out and dagg in and
// out in FP32 (two each); the neighbours' dagg rows beyond the first reading come
// out of L2.  MFMA operands: the data product takes the
// weights first and dpre second, the output features dealt to the weight rows
// as in the forward layer: a lane holds the same 16 features of its row in dh,
// dpre and the products.  The
// weight product contracts over rows: both operands go through LDS transposed,
// two rows packed per 4-byte write.
// At 200,000 triangles 79 us per layer, 3.6 TB/s; as three kernels 66.7 us
// (data product), 637 us (weight product: 98 workgroups, 2-byte transposed
// writes) and 116 us (combination).
template <bool FIRST>
__global__ __launch_bounds__(256) void kGnnLayerBwd(
    int n, int nTiles, int per, const float *__restrict__ dout, const float *__restrict__ wo, const float *dhIn,
    const float *__restrict__ daggIn, const float *__restrict__ gterm, const int *__restrict__ sliceOff,
    const int *__restrict__ col, const float *__restrict__ ah, const __bf16 *__restrict__ pre,
    const __bf16 *__restrict__ h, const __bf16 *__restrict__ agg, const __bf16 *__restrict__ wN, float *dhOut,
    float *__restrict__ daggOut, float *__restrict__ partials) {
  __shared__ __attribute__((aligned(16))) __bf16 W[128][H + 8];  // [k][c]
  __shared__ __attribute__((aligned(16))) __bf16 HA[128 * kTPitch], DP[H * kTPitch];
  __shared__ __attribute__((aligned(16))) float fs[H];           // FIRST: w_out, else gterm
  for (int t = threadIdx.x; t < 128 * 8; t += 256) {
    const int k = t >> 3, c8 = 8 * (t & 7);
    // row 16 t + m of W: feature 32 (t / 2) + 8 (m / 4) + 4 (t % 2) + m % 4
    const int at = 16 * (2 * (k >> 5) + ((k >> 2) & 1)) + 4 * ((k >> 3) & 3) + (k & 3);
    *(bf16x8 *)&W[at][c8] = *(const bf16x8 *)&wN[k * H + c8];
  }
  if (threadIdx.x < H) fs[threadIdx.x] = FIRST ? wo[threadIdx.x] : gterm[threadIdx.x];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, gq = lane >> 4, l16 = lane & 15;
  auto feat = [&](int t) { return 32 * (t >> 1) + 8 * gq + 4 * (t & 1); };  // first feature of dh[t]
  const int group = xcdTile(blockIdx.x, gridDim.x);
  const int t1 = min(nTiles, (group + 1) * per);
  f32x4 acc[2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[a][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float db = 0.f;
  for (int tile = group * per; tile < t1; ++tile) {
    __syncthreads();  // the previous tile's LDS reads are done (first tile: W and fs are written)
    const int base = tile * kTileRows;
    // stage [h | agg]^T: row pair rp, octet of features o8 (0..15)
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int item = threadIdx.x + 256 * it;
      const int o8 = item & 15, rp = item >> 4;
      const int row = base + 2 * rp;
      const __bf16 *src = o8 < 8 ? h : agg;
      const int f0 = 8 * (o8 & 7);
      bf16x8 u = {}, v = {};
      if (row < n) u = *(const bf16x8 *)&src[(size_t)row * H + f0];
      if (row + 1 < n) v = *(const bf16x8 *)&src[(size_t)(row + 1) * H + f0];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
        *(bf16x2 *)&HA[tileAt(8 * o8 + j, rp >> 2) + 2 * (rp & 3)] = bf16x2{u[j], v[j]};
      }
    }
    const int l = 16 * wave + l16, r = base + l;
    const bool act = r < n;
    const size_t at = (size_t)(act ? r : 0) * H;
    f32x4 dh[4];
    if (FIRST) {
      const float d = act ? dout[r] : 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t) dh[t] = d * *(const f32x4 *)&fs[feat(t)];
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) dh[t] = *(const f32x4 *)&dhIn[at + feat(t)] + *(const f32x4 *)&fs[feat(t)];
      const int o = sliceOff[tile], K = act ? (sliceOff[tile + 1] - o) >> 6 : 0;
      for (int e0 = 0; e0 < K; e0 += 2) {
        int cc[2];
        float w[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const bool in = e0 + q < K;
          const int idx = o + ((e0 + (in ? q : 0)) << 6) + l;
          cc[q] = col[idx];
          w[q] = in ? ah[idx] : 0.f;
        }
        f32x4 x[2][4];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            x[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (w[q] != 0.f) x[q][t] = *(const f32x4 *)&daggIn[(size_t)cc[q] * H + feat(t)];
          }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) dh[t][v] = fmaf(w[q], x[q][t][v], dh[t][v]);
      }
    }
    bf16x8 a[2];
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      const bf16x8 pv = *(const bf16x8 *)&pre[at + 32 * kc + 8 * gq];
#pragma unroll
      for (int j = 0; j < 8; ++j) a[kc][j] = (__bf16)(act && (float)pv[j] > 0.f ? dh[2 * kc + (j >> 2)][j & 3] : 0.f);
    }
    // dpre^T: lanes of rows r, r ^ 1 exchange halves and write row pairs; the
    // even row writes the features of kc = 0, the odd row those of kc = 1
    {
      typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
      const u32x4 w0 = __builtin_bit_cast(u32x4, a[0]), w1 = __builtin_bit_cast(u32x4, a[1]);
      const bool odd = lane & 1;
      const int rp = l >> 1;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const unsigned got = __shfl_xor(odd ? w0[m] : w1[m], 1, 64);
        const unsigned lo = odd ? got : w0[m], hi = odd ? w1[m] : got;  // row pair's even / odd row
        // word m: features j = 2 m, 2 m + 1 of the half
        const int f = (odd ? 32 : 0) + 8 * gq + 2 * m;
        *(unsigned *)&DP[tileAt(f, rp >> 2) + 2 * (rp & 3)] = (lo & 0xffffu) | (hi << 16);
        *(unsigned *)&DP[tileAt(f + 1, rp >> 2) + 2 * (rp & 3)] = (lo >> 16) | (hi & 0xffff0000u);
      }
    }
    // data product
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      f32x4 p = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) p = mfma(*(const bf16x8 *)&W[16 * t + l16][32 * kc + 8 * gq], a[kc], p);
      if (act) {
        if (t < 4) *(f32x4 *)&dhOut[at + feat(t)] = dh[t & 3] + p;
        else *(f32x4 *)&daggOut[at + feat(t - 4)] = p;
      }
    }
    __syncthreads();
    // weight product: wave w owns k in [32 w, 32 w + 32)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 av[2], bv[4];
#pragma unroll
      for (int q = 0; q < 2; ++q) av[q] = *(const bf16x8 *)&HA[tileAt(32 * wave + 16 * q + l16, 4 * kk + gq)];
#pragma unroll
      for (int t = 0; t < 4; ++t) bv[t] = *(const bf16x8 *)&DP[tileAt(16 * t + l16, 4 * kk + gq)];
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[q][t] = mfma(av[q], bv[t], acc[q][t]);
      const bf16x8 mine = *(const bf16x8 *)&DP[tileAt(16 * wave + l16, 4 * kk + gq)];
#pragma unroll
      for (int j = 0; j < 8; ++j) db += (float)mine[j];
    }
  }
  // partial record: [128][64] dW then [64] db
  float *P = partials + (size_t)blockIdx.x * (128 * H + H);
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) P[(32 * wave + 16 * q + 4 * gq + v) * H + 16 * t + l16] = acc[q][t][v];
  db += __shfl_xor(db, 16, 64);
  db += __shfl_xor(db, 32, 64);
  if (gq == 0) P[128 * H + 16 * wave + l16] = db;
}

// grad[k] = sum of the partial records' entry k (fixed order), 64 entries per block
__global__ __launch_bounds__(kFinThreads) void kSumPartials(int records, int m, const float *__restrict__ partials,
                                                            float *__restrict__ grad) {
  __shared__ float red[16][H];
  const int k = blockIdx.x * H + (threadIdx.x & 63);
  const float v = sumRecords(partials, records, m, k, k < m, red);
  if (threadIdx.x < H && k < m) grad[k] = v;
}

// The sums of a backward layer's records: dWsm (blocks 0 to 127) and db (block
// 128), which then also gives dWg[k][c] = g[k] db[c] and
// gterm[k] = sum_c Wg[k][c] db[c] / n.
__global__ __launch_bounds__(kFinThreads) void kGnnSumLayer(int n, int records, const float *__restrict__ partials,
                                                            const float *__restrict__ g, const float *__restrict__ Wg,
                                                            float *__restrict__ dWsm, float *__restrict__ db,
                                                            float *__restrict__ dWg, float *__restrict__ gterm) {
  __shared__ float red[16][H], dbs[H];
  const int f = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int k = blockIdx.x * H + f;
  const float v = sumRecords(partials, records, 128 * H + H, k, true, red);
  if (blockIdx.x < 128) {
    if (q == 0) dWsm[k] = v;
    return;
  }
  if (q == 0) {
    db[f] = v;
    dbs[f] = v;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = 4 * q + j;
    dWg[row * H + f] = g[row] * dbs[f];
    float s = Wg[row * H + f] * dbs[f];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (f == 0) gterm[row] = s / (float)n;
  }
}

// input layer gradient partials: dW_in[k][c] = sum_r X[r][k] dpre0[r][c],
// db_in[c], with dh0 = dhIn + gterm + A_hat^T dagg of the first layer formed
// as it is read: four features of a row per thread, 16 rows per step
__global__ __launch_bounds__(256) void kGnnInGrad(int n, const float *__restrict__ X, const __bf16 *__restrict__ pre0,
                                                  const float *__restrict__ dhIn, const float *__restrict__ dagg,
                                                  const float *__restrict__ gterm, const int *__restrict__ sliceOff,
                                                  const int *__restrict__ col, const float *__restrict__ ah,
                                                  float *__restrict__ partials) {
  __shared__ float red[16][H];
  const int f0 = 4 * (threadIdx.x & 15), q = threadIdx.x >> 4;
  const f32x4 g = *(const f32x4 *)&gterm[f0];
  f32x4 acc[kGnnDin + 1];
#pragma unroll
  for (int k = 0; k <= kGnnDin; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int b = xcdTile(blockIdx.x, gridDim.x); b * 16 < n; b += gridDim.x) {
    const int i = b * 16 + q;
    if (i >= n) continue;
    const size_t at = (size_t)i * H + f0;
    f32x4 dh = *(const f32x4 *)&dhIn[at] + g;
    const int s = i >> 6, l = i & 63;
    const int o = sliceOff[s], K = (sliceOff[s + 1] - o) >> 6;
    for (int e = 0; e < K; ++e) {
      const int idx = o + (e << 6) + l;
      const float w = ah[idx];
      if (w == 0.f) continue;
      const f32x4 x = *(const f32x4 *)&dagg[(size_t)col[idx] * H + f0];
#pragma unroll
      for (int v = 0; v < 4; ++v) dh[v] = fmaf(w, x[v], dh[v]);
    }
    const bf16x4 pv = *(const bf16x4 *)&pre0[at];
    const f32x4 x = *(const f32x4 *)&X[4 * (size_t)i];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float dp = (float)pv[v] > 0.f ? dh[v] : 0.f;
#pragma unroll
      for (int k = 0; k < kGnnDin; ++k) acc[k][v] = fmaf(x[k], dp, acc[k][v]);
      acc[kGnnDin][v] += dp;
    }
  }
#pragma unroll
  for (int k = 0; k <= kGnnDin; ++k) {
    *(f32x4 *)&red[q][f0] = acc[k];
    __syncthreads();
    if (threadIdx.x < H) {
      float v = 0.f;
      for (int j = 0; j < 16; ++j) v += red[j][threadIdx.x];
      partials[(size_t)blockIdx.x * (kGnnDin + 1) * H + k * H + threadIdx.x] = v;
    }
    __syncthreads();
  }
}

// Adam (Kingma & Ba 2015), then refresh the BF16 weight copies
__global__ void kAdam(int m, float *__restrict__ p, const float *__restrict__ g, float *__restrict__ mo,
                      float *__restrict__ ve, float lr, float b1, float b2, float eps, float c1, float c2,
                      float clip) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) {
    float gi = g[i];
    gi = fminf(fmaxf(gi, -clip), clip);
    const float mi = b1 * mo[i] + (1.f - b1) * gi;
    const float vi = b2 * ve[i] + (1.f - b2) * gi * gi;
    mo[i] = mi;
    ve[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

// wT[l][o][k] = Wsm[l][k][o] ; wN[l][k][o] = Wsm[l][k][o]  (BF16)
__global__ void kGnnCast(int L, const float *__restrict__ P, size_t layer0, size_t layerSize, __bf16 *__restrict__ wT,
                         __bf16 *__restrict__ wN) {
  const int per = 128 * H;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < L * per; t += gridDim.x * blockDim.x) {
    const int l = t / per, kk = (t % per) / H, o = t % H;
    const float v = P[layer0 + (size_t)l * layerSize + (size_t)kk * H + o];
    wT[(size_t)l * per + (size_t)o * 128 + kk] = (__bf16)v;
    wN[(size_t)l * per + (size_t)kk * H + o] = (__bf16)v;
  }
}

__global__ void kGnnScaleOut(int n, const float *__restrict__ out, const float *__restrict__ sd,
                             const double *__restrict__ scal, double *__restrict__ e) {
  const double s = scal[0];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    e[i] = (double)out[i] * s / (double)sd[i];
}

// ---------------------------------------------------------------- host side
inline int g1(long n, int cap = 8192) { return (int)std::max<long>(1, std::min<long>((n + 255) / 256, cap)); }

void ensureNet(phase_hip_solver *s) {
  if (!s->gnn) s->gnn = new GnnState();
  GnnState &G = *s->gnn;
  if (!G.initialised) {
    const size_t P = G.lay.total();
    G.params.alloc(P);
    G.grad.alloc(P);
    G.adamM.alloc(P);
    G.adamV.alloc(P);
    // He-style initialisation from a fixed seed (deterministic)
    std::mt19937 rng(1234);
    std::normal_distribution<float> nd(0.f, 1.f);
    std::vector<float> h(P, 0.f);
    for (size_t i = 0; i < (size_t)kGnnDin * H; ++i) h[G.lay.inW() + i] = nd(rng) * std::sqrt(2.f / kGnnDin);
    for (int l = 0; l < G.lay.L; ++l) {
      for (size_t i = 0; i < (size_t)128 * H; ++i) h[G.lay.wsm(l) + i] = nd(rng) * (0.5f / std::sqrt((float)H));
      for (size_t i = 0; i < (size_t)H * H; ++i) h[G.lay.wg(l) + i] = nd(rng) * (0.1f / std::sqrt((float)H));
    }
    for (int i = 0; i < H; ++i) h[G.lay.outW() + i] = nd(rng) * (1.f / std::sqrt((float)H));
    G.params.upload(h, s->stream);
    G.adamM.zero(s->stream);
    G.adamV.zero(s->stream);
    G.step = 0;
    G.initialised = true;
  }
  const int n = s->rank;
  if (G.n != n) {
    const int L = G.lay.L;
    G.n = n;
    G.sd.alloc(n);
    G.rowsum.alloc(n);
    G.X.alloc(4 * (size_t)n);
    G.out.alloc(n);
    G.dOut.alloc(n);
    G.h.alloc((size_t)(L + 1) * n * H);
    G.agg.alloc((size_t)L * n * H);
    G.pre.alloc((size_t)L * n * H);
    G.pre0.alloc((size_t)n * H);
    G.dh.alloc((size_t)n * H);
    G.dagg.alloc(2 * (size_t)n * H);
    G.gmean.alloc((size_t)L * H);
    G.cvec.alloc((size_t)L * H);
    G.partials.alloc(std::max<size_t>((size_t)tilesFor(n, kBwdGroups).groups * (128 * H + H),
                                      (size_t)kFwdGroups * (kGnnDin + 1) * H));
    G.scal.alloc(8);
    G.scal.zero(s->stream);
    G.wT.alloc((size_t)L * 128 * H);
    G.wN.alloc((size_t)L * 128 * H);
  }
}

// Graph quantities of the current matrix (FP32 SELL copy): sd, row-sum ratio,
// graph weights.
void prepareGraph(phase_hip_solver *s) {
  GnnState &G = *s->gnn;
  const int n = s->rank;
  G.ahat.alloc(s->dSell32.n);
  hipLaunchKernelGGL(kGnnDiag, dim3(g1(n)), dim3(256), 0, s->stream, n, s->dSliceOff.p, s->dSellCol.p, s->dSell32.p,
                     G.sd.p, G.rowsum.p);
  hipLaunchKernelGGL(kGnnWeights, dim3(g1(n)), dim3(256), 0, s->stream, n, s->dSliceOff.p, s->dSellCol.p,
                     s->dSell32.p, G.sd.p, G.ahat.p);
}

void castWeights(phase_hip_solver *s) {
  GnnState &G = *s->gnn;
  hipLaunchKernelGGL(kGnnCast, dim3(g1((long)G.lay.L * 128 * H)), dim3(256), 0, s->stream, G.lay.L, G.params.p,
                     G.lay.layer(0), GnnLayout::layerSize(), G.wT.p, G.wN.p);
}

__bf16 *hL(GnnState &G, int l) { return G.h.p + (size_t)l * G.n * H; }

// features of residual r (FP32, solver order) with z = ILU32^{-1} r supplied
void gnnFeatures(phase_hip_solver *s, const float *r, const float *z) {
  GnnState &G = *s->gnn;
  const int n = s->rank;
  const int gr = gridFor1(n);
  hipLaunchKernelGGL(kGnnRms, dim3(gr), dim3(kRedBlock), 0, s->stream, n, r, G.sd.p, s->dPartials.p);
  hipLaunchKernelGGL(kGnnRmsFinish, dim3(1), dim3(kFinBlock), 0, s->stream, n, s->dPartials.p, gr, G.scal.p);
  hipLaunchKernelGGL(kGnnFeatures, dim3(g1(n)), dim3(256), 0, s->stream, n, r, z, G.sd.p, G.rowsum.p, G.scal.p, G.X.p);
}

}  // namespace

namespace phase {

void gnnForward(phase_hip_solver *s) {
  GnnState &G = *s->gnn;
  const int n = s->rank, L = G.lay.L;
  const float *P = G.params.p;
  const Tiles T = tilesFor(n, kFwdGroups);
  int records = std::min(kFwdGroups, std::max(1, (n + 31) / 32));
  hipLaunchKernelGGL(kGnnIn, dim3(records), dim3(256), 0, s->stream, n, G.X.p, P + G.lay.inW(), G.pre0.p, hL(G, 0),
                     G.partials.p);
  for (int l = 0; l < L; ++l) {
    hipLaunchKernelGGL(kGnnMeanFold, dim3(1), dim3(kFinThreads), 0, s->stream, n, records, G.partials.p,
                       P + G.lay.wg(l), P + G.lay.b(l), G.gmean.p + l * H, G.cvec.p + l * H);
    auto layer = l + 1 < L ? kGnnLayerFwd<false> : kGnnLayerFwd<true>;
    hipLaunchKernelGGL(layer, dim3(T.groups), dim3(256), 0, s->stream, n, T.n, T.per, (const __bf16 *)hL(G, l),
                       s->dSliceOff.p, s->dSellCol.p, G.ahat.p, G.wT.p + (size_t)l * 128 * H, G.cvec.p + l * H,
                       G.agg.p + (size_t)l * n * H, G.pre.p + (size_t)l * n * H, hL(G, l + 1), G.partials.p,
                       P + G.lay.outW(), G.out.p);
    records = T.groups;
  }
  PH_CHECK(hipGetLastError());
}

// Loss of the last forward: against target t (error objective) or on the
// residual r of the pair (residual objective, with the FP32 copy of A);
// dout for backward.
void gnnLoss(phase_hip_solver *s, const float *target, const float *r) {
  GnnState &G = *s->gnn;
  const int n = s->rank, gr = gridFor1(n);
  if (s->learnedObjective == 1) {
    for (DBuf<float> *b : {&G.resC, &G.resQ, &G.resDq, &G.resG}) b->alloc(n);
    const int gs = std::max(1, (s->ord.nSlices + 3) / 4);
    hipLaunchKernelGGL(kGnnResC, dim3(g1(n)), dim3(256), 0, s->stream, n, G.out.p, G.sd.p, G.resC.p);
    hipLaunchKernelGGL((kSpmv<float>), dim3(gs), dim3(kRedBlock), 0, s->stream, n, s->ord.nSlices, s->dSliceOff.p,
                       s->dSellCol.p, s->dSell32.p, (const float *)G.resC.p, G.resQ.p);
    hipLaunchKernelGGL(kGnnLossCos, dim3(gr), dim3(kRedBlock), 0, s->stream, n, G.resQ.p, r, s->dPartials.p);
    hipLaunchKernelGGL(kGnnLossFinish, dim3(1), dim3(kFinBlock), 0, s->stream, s->dPartials.p, gr, G.scal.p);
    hipLaunchKernelGGL(kGnnResDq, dim3(g1(n)), dim3(256), 0, s->stream, n, G.resQ.p, r, G.scal.p, G.resDq.p);
    hipLaunchKernelGGL((kSpmv<float>), dim3(gs), dim3(kRedBlock), 0, s->stream, n, s->ord.nSlices, s->dSliceOff.p,
                       s->dSellCol.p, s->dSell32.p, (const float *)G.resDq.p, G.resG.p);
    hipLaunchKernelGGL(kGnnResDout, dim3(g1(n)), dim3(256), 0, s->stream, n, G.resG.p, G.sd.p, G.dOut.p);
  } else {
    hipLaunchKernelGGL(kGnnLossCos, dim3(gr), dim3(kRedBlock), 0, s->stream, n, G.out.p, target, s->dPartials.p);
    hipLaunchKernelGGL(kGnnLossFinish, dim3(1), dim3(kFinBlock), 0, s->stream, s->dPartials.p, gr, G.scal.p);
    hipLaunchKernelGGL(kGnnDout, dim3(g1(n)), dim3(256), 0, s->stream, n, G.out.p, target, G.scal.p, G.dOut.p);
  }
  PH_CHECK(hipGetLastError());
}

// Gradient of the loss of the last forward (with target) into G.grad.
void gnnBackward(phase_hip_solver *s) {
  GnnState &G = *s->gnn;
  const int n = s->rank, L = G.lay.L;
  const float *P = G.params.p;
  const int nbO = std::min(kFwdGroups, std::max(1, (n + 31) / 32));
  hipLaunchKernelGGL(kGnnOutGrad, dim3(nbO), dim3(256), 0, s->stream, n, (const __bf16 *)hL(G, L), G.dOut.p,
                     G.partials.p);
  hipLaunchKernelGGL(kSumPartials, dim3((H + 1 + H - 1) / H), dim3(kFinThreads), 0, s->stream, nbO, H + 1,
                     G.partials.p, G.grad.p + G.lay.outW());
  const Tiles T = tilesFor(n, kBwdGroups);
  float *dagg[2] = {G.dagg.p, G.dagg.p + (size_t)n * H};
  float *gterm = G.cvec.p;  // the forward's c vectors are no longer needed
  for (int l = L - 1; l >= 0; --l) {
    auto layer = l == L - 1 ? kGnnLayerBwd<true> : kGnnLayerBwd<false>;
    hipLaunchKernelGGL(layer, dim3(T.groups), dim3(256), 0, s->stream, n, T.n, T.per, G.dOut.p, P + G.lay.outW(),
                       (const float *)G.dh.p, (const float *)dagg[(l + 1) & 1], (const float *)gterm, s->dSliceOff.p,
                       s->dSellCol.p, G.ahat.p, G.pre.p + (size_t)l * n * H, (const __bf16 *)hL(G, l),
                       (const __bf16 *)(G.agg.p + (size_t)l * n * H), G.wN.p + (size_t)l * 128 * H, G.dh.p,
                       dagg[l & 1], G.partials.p);
    hipLaunchKernelGGL(kGnnSumLayer, dim3(129), dim3(kFinThreads), 0, s->stream, n, T.groups, G.partials.p,
                       G.gmean.p + l * H, P + G.lay.wg(l), G.grad.p + G.lay.wsm(l), G.grad.p + G.lay.b(l),
                       G.grad.p + G.lay.wg(l), gterm);
  }
  const int nbI = std::min(kFwdGroups, std::max(1, (n + 15) / 16));
  hipLaunchKernelGGL(kGnnInGrad, dim3(nbI), dim3(256), 0, s->stream, n, G.X.p, G.pre0.p, G.dh.p, dagg[0], gterm,
                     s->dSliceOff.p, s->dSellCol.p, G.ahat.p, G.partials.p);
  hipLaunchKernelGGL(kSumPartials, dim3(kGnnDin + 1), dim3(kFinThreads), 0, s->stream, nbI, (kGnnDin + 1) * H,
                     G.partials.p, G.grad.p + G.lay.inW());
  PH_CHECK(hipGetLastError());
}

}  // namespace phase

namespace {

void gnnTrainStep(phase_hip_solver *s, int pair, float lr) {
  GnnState &G = *s->gnn;
  const int n = s->rank;
  KrylovVecs<float> &K = s->k32;
  if (pair < 0 || pair >= G.nPairs || K.y.n < (size_t)n || K.sh.n < (size_t)n || !s->dFac32.p)
    fail(PHASE_HIP_ESTATE, "training state not prepared");
  const float *r = G.pairR.p + (size_t)pair * n;
  const float *e = G.pairE.p + (size_t)pair * n;
  // z = ILU(0)^{-1} r (FP32 factor)
  iluApplyDev<float>(s, s->dFac32.p, r, K.y.p, K.sh.p);
  gnnFeatures(s, r, K.sh.p);
  hipLaunchKernelGGL(kGnnTarget, dim3(g1(n)), dim3(256), 0, s->stream, n, e, G.sd.p, G.scal.p, K.s.p);
  gnnForward(s);
  gnnLoss(s, K.s.p, r);
  gnnBackward(s);
  ++G.step;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)G.step), c2 = 1.f - std::pow(b2, (float)G.step);
  const int P = (int)G.lay.total();
  hipLaunchKernelGGL(kAdam, dim3(g1(P)), dim3(256), 0, s->stream, P, G.params.p, G.grad.p, G.adamM.p, G.adamV.p, lr,
                     b1, b2, 1e-8f, c1, c2, 10.f);
  castWeights(s);
}

// r64 (solver order, device) -> e64 network correction (solver order, device)
void applyNet(phase_hip_solver *s, const double *r64, double *e64) {
  GnnState &G = *s->gnn;
  const int n = s->rank;
  KrylovVecs<float> &K = s->k32;
  if (K.t.n < (size_t)n || K.y.n < (size_t)n || K.sh.n < (size_t)n || !s->dFac32.p || G.n != n)
    fail(PHASE_HIP_ESTATE, "network not prepared for this system");
  hipLaunchKernelGGL((kConvert<double, float>), dim3(g1(n)), dim3(256), 0, s->stream, n, r64, K.t.p);
  iluApplyDev<float>(s, s->dFac32.p, K.t.p, K.y.p, K.sh.p);
  gnnFeatures(s, K.t.p, K.sh.p);
  gnnForward(s);
  hipLaunchKernelGGL(kGnnScaleOut, dim3(g1(n)), dim3(256), 0, s->stream, n, G.out.p, G.sd.p, G.scal.p, e64);
  PH_CHECK(hipGetLastError());
}

template <class F>
int guardedG(phase_hip_solver *s, F &&f) {
  if (!s) return PHASE_HIP_EINVAL;
  try {
    f();
    return PHASE_HIP_OK;
  } catch (const HipError &e) {
    s->err = e.msg;
    return e.code;
  } catch (const std::exception &e) {
    s->err = e.what();
    return PHASE_HIP_EINVAL;
  }
}

void requireSystem(phase_hip_solver *s) {
  if (!s->havePattern || !s->haveValues) fail(PHASE_HIP_ESTATE, "no system: call set() or assemble first");
}

}  // namespace

namespace phase {

void gnnFree(phase_hip_solver *s) {
  delete s->gnn;
  s->gnn = nullptr;
}

void gnnPrepare(phase_hip_solver *s) {
  solverEnsureSingle(s);
  // the FP32 work vectors (ILU apply of the features, inference staging) exist
  // even when only FP64 solves have run
  s->k32.alloc(s->rank);
  ensureNet(s);
  prepareGraph(s);
  castWeights(s);
}

void gnnApply(phase_hip_solver *s, const double *r64, double *e64) { applyNet(s, r64, e64); }

// Capture hooks (FP64 solves): snapshot (r, x) every `captureEvery`
// iterations; the correction e = x_final - x is known when the solve ends.
void gnnCaptureIter(phase_hip_solver *s, const double *r, const double *x, int iter) {
  GnnState *G = s->gnn;
  if (!G || G->captureEvery <= 0) return;
  if (G->nPairs + (int)G->pendingSnap.size() >= G->maxPairs) return;
  const int n = s->rank;
  const int slot = G->nPairs + (int)G->pendingSnap.size();
  const int k = (int)G->pendingSnap.size();
  if ((size_t)(k + 1) * n > G->snapX.n) {
    // grow the snapshot store (device-to-device copy of what it holds)
    DBuf<double> nb;
    nb.alloc((size_t)(k + 8) * n);
    if (k) PH_CHECK(hipMemcpyAsync(nb.p, G->snapX.p, (size_t)k * n * sizeof(double), hipMemcpyDeviceToDevice, s->stream));
    G->snapX = std::move(nb);
  }
  hipLaunchKernelGGL((kConvert<double, float>), dim3(g1(n)), dim3(256), 0, s->stream, n, r, G->pairR.p + (size_t)slot * n);
  PH_CHECK(hipMemcpyAsync(G->snapX.p + (size_t)k * n, x, n * sizeof(double), hipMemcpyDeviceToDevice, s->stream));
  G->pendingSnap.push_back(slot);
  (void)iter;
}

__global__ void kPairE(int n, const double *__restrict__ xf, const double *__restrict__ xk, float *__restrict__ e) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) e[i] = (float)(xf[i] - xk[i]);
}

void gnnCaptureFinish(phase_hip_solver *s, const double *xFinal, bool converged) {
  GnnState *G = s->gnn;
  if (!G || G->captureEvery <= 0) return;
  const int n = s->rank;
  if (converged) {
    for (size_t k = 0; k < G->pendingSnap.size(); ++k)
      hipLaunchKernelGGL(kPairE, dim3(g1(n)), dim3(256), 0, s->stream, n, xFinal, G->snapX.p + k * n,
                         G->pairE.p + (size_t)G->pendingSnap[k] * n);
    G->nPairs += (int)G->pendingSnap.size();
  }
  G->pendingSnap.clear();
}

}  // namespace phase

extern "C" {

int phase_hip_learned_capture(phase_hip_solver *s, int everyIters, int maxPairs) {
  return guardedG(s, [&] {
    requireSystem(s);
    if (everyIters < 0 || maxPairs < 0) fail(PHASE_HIP_EINVAL, "negative capture settings");
    PH_CHECK(hipSetDevice(s->device));
    ensureNet(s);
    GnnState &G = *s->gnn;
    G.captureEvery = everyIters;
    if (maxPairs != G.maxPairs) {
      G.maxPairs = maxPairs;
      G.pairR.alloc((size_t)std::max(1, maxPairs) * s->rank);
      G.pairE.alloc((size_t)std::max(1, maxPairs) * s->rank);
      G.nPairs = 0;
    }
    G.pendingSnap.clear();
  });
}

int phase_hip_learned_n_pairs(const phase_hip_solver *s, int *count) {
  if (!s || !count) return PHASE_HIP_EINVAL;
  *count = s->gnn ? s->gnn->nPairs : 0;
  return PHASE_HIP_OK;
}

// Captured pairs [first, first + count) to the host, original numbering,
// pair-major (count * rank floats each for r and e).
int phase_hip_learned_pairs(phase_hip_solver *s, int first, int count, float *r, float *e) {
  return guardedG(s, [&] {
    requireSystem(s);
    PH_CHECK(hipSetDevice(s->device));
    const int have = s->gnn ? s->gnn->nPairs : 0;
    if (first < 0 || count < 0 || first + count > have) fail(PHASE_HIP_EINVAL, "pair range outside the captured pairs");
    if (count > 0 && (!r || !e)) fail(PHASE_HIP_EINVAL, "null pair buffer");
    GnnState &G = *s->gnn;
    const int n = s->rank;
    DBuf<float> tmp;
    tmp.alloc(2 * (size_t)n);
    for (int k = 0; k < count; ++k) {
      const size_t slot = (size_t)(first + k) * n;
      hipLaunchKernelGGL((kPermuteOut<float, float>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p,
                         G.pairR.p + slot, tmp.p);
      hipLaunchKernelGGL((kPermuteOut<float, float>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p,
                         G.pairE.p + slot, tmp.p + n);
      PH_CHECK(hipMemcpyAsync(r + (size_t)k * n, tmp.p, n * sizeof(float), hipMemcpyDeviceToHost, s->stream));
      PH_CHECK(hipMemcpyAsync(e + (size_t)k * n, tmp.p + n, n * sizeof(float), hipMemcpyDeviceToHost, s->stream));
      PH_CHECK(hipStreamSynchronize(s->stream));
    }
  });
}

// Append count pairs (original numbering, the layout phase_hip_learned_pairs
// writes) to the capture store set up by phase_hip_learned_capture.
int phase_hip_learned_add_pairs(phase_hip_solver *s, int count, const float *r, const float *e) {
  return guardedG(s, [&] {
    requireSystem(s);
    PH_CHECK(hipSetDevice(s->device));
    if (count < 0 || (count > 0 && (!r || !e))) fail(PHASE_HIP_EINVAL, "bad pair count or null pair buffer");
    if (!s->gnn || s->gnn->maxPairs == 0) fail(PHASE_HIP_ESTATE, "no pair store: call phase_hip_learned_capture first");
    GnnState &G = *s->gnn;
    if (!G.pendingSnap.empty()) fail(PHASE_HIP_ESTATE, "a capture is in progress");
    if (G.nPairs + count > G.maxPairs) fail(PHASE_HIP_EINVAL, "more pairs than the store holds (maxPairs)");
    const int n = s->rank;
    DBuf<float> tmp;
    tmp.alloc(2 * (size_t)n);
    for (int k = 0; k < count; ++k) {
      const size_t slot = (size_t)(G.nPairs + k) * n;
      PH_CHECK(hipMemcpyAsync(tmp.p, r + (size_t)k * n, n * sizeof(float), hipMemcpyHostToDevice, s->stream));
      PH_CHECK(hipMemcpyAsync(tmp.p + n, e + (size_t)k * n, n * sizeof(float), hipMemcpyHostToDevice, s->stream));
      hipLaunchKernelGGL((kPermuteIn<float, float>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p, tmp.p,
                         G.pairR.p + slot, 1.0);
      hipLaunchKernelGGL((kPermuteIn<float, float>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p, tmp.p + n,
                         G.pairE.p + slot, 1.0);
      PH_CHECK(hipStreamSynchronize(s->stream));
    }
    G.nPairs += count;
  });
}

int phase_hip_learned_train(phase_hip_solver *s, int steps, double lr, int seed, double *lastLoss) {
  return guardedG(s, [&] {
    requireSystem(s);
    PH_CHECK(hipSetDevice(s->device));
    if (!s->gnn || s->gnn->nPairs == 0) fail(PHASE_HIP_ESTATE, "no captured (residual, correction) pairs");
    gnnPrepare(s);
    GnnState &G = *s->gnn;
    std::mt19937 rng((unsigned)seed);
    double loss = 0.;
    PH_CHECK(hipMemsetAsync(G.scal.p + 5, 0, sizeof(double), s->stream));
    for (int t = 0; t < steps; ++t) gnnTrainStep(s, (int)(rng() % (unsigned)G.nPairs), (float)lr);
    PH_CHECK(hipMemcpyAsync(&loss, G.scal.p + 5, sizeof(double), hipMemcpyDeviceToHost, s->stream));
    PH_CHECK(hipStreamSynchronize(s->stream));
    if (steps > 0) loss /= steps;
    G.trained = true;
    if (lastLoss) *lastLoss = loss;
  });
}

int phase_hip_learned_params(phase_hip_solver *s, float *params, int *count) {
  return guardedG(s, [&] {
    PH_CHECK(hipSetDevice(s->device));
    if (!s->gnn) s->gnn = new GnnState();
    GnnState &G = *s->gnn;
    if (count) *count = (int)G.lay.total();
    if (!params) return;
    if (!G.initialised) {
      if (!s->havePattern) fail(PHASE_HIP_ESTATE, "network not initialised");
      ensureNet(s);
    }
    PH_CHECK(hipMemcpyAsync(params, G.params.p, G.lay.total() * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    PH_CHECK(hipStreamSynchronize(s->stream));
  });
}

int phase_hip_learned_set_params(phase_hip_solver *s, const float *params, int count) {
  return guardedG(s, [&] {
    requireSystem(s);
    PH_CHECK(hipSetDevice(s->device));
    ensureNet(s);
    GnnState &G = *s->gnn;
    if (count != (int)G.lay.total()) fail(PHASE_HIP_EINVAL, "parameter count mismatch");
    PH_CHECK(hipMemcpyAsync(G.params.p, params, count * sizeof(float), hipMemcpyHostToDevice, s->stream));
    G.adamM.zero(s->stream);
    G.adamV.zero(s->stream);
    G.step = 0;
    G.trained = true;
    PH_CHECK(hipStreamSynchronize(s->stream));
  });
}

// Forward + backward on a given residual r, ILU-preconditioned residual z and
// correction target e (original numbering): network output (original
// numbering), loss and flat parameter gradient.  For gradient checks.
int phase_hip_learned_eval(phase_hip_solver *s, const double *r, const double *z, const double *target, double *out,
                           double *loss, float *grad) {
  return guardedG(s, [&] {
    requireSystem(s);
    PH_CHECK(hipSetDevice(s->device));
    gnnPrepare(s);
    GnnState &G = *s->gnn;
    const int n = s->rank;
    KrylovVecs<float> &K = s->k32;
    K.alloc(n);
    DBuf<double> &tmp = G.stage;
    tmp.alloc(3 * (size_t)n);
    PH_CHECK(hipMemcpyAsync(tmp.p, r, n * sizeof(double), hipMemcpyHostToDevice, s->stream));
    PH_CHECK(hipMemcpyAsync(tmp.p + n, z, n * sizeof(double), hipMemcpyHostToDevice, s->stream));
    PH_CHECK(hipMemcpyAsync(tmp.p + 2 * n, target, n * sizeof(double), hipMemcpyHostToDevice, s->stream));
    hipLaunchKernelGGL((kPermuteIn<double, float>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p, tmp.p, K.t.p, 1.0);
    hipLaunchKernelGGL((kPermuteIn<double, float>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p, tmp.p + n,
                       K.sh.p, 1.0);
    hipLaunchKernelGGL((kPermuteIn<double, float>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p, tmp.p + 2 * n,
                       K.s.p, 1.0);
    gnnFeatures(s, K.t.p, K.sh.p);
    gnnForward(s);
    gnnLoss(s, K.s.p, K.t.p);
    gnnBackward(s);
    hipLaunchKernelGGL((kConvert<float, double>), dim3(g1(n)), dim3(256), 0, s->stream, n, G.out.p, tmp.p);
    hipLaunchKernelGGL((kPermuteOut<double>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p, tmp.p, tmp.p + n);
    PH_CHECK(hipMemcpyAsync(out, tmp.p + n, n * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    PH_CHECK(hipMemcpyAsync(loss, G.scal.p + 1, sizeof(double), hipMemcpyDeviceToHost, s->stream));
    PH_CHECK(hipMemcpyAsync(grad, G.grad.p, G.lay.total() * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    PH_CHECK(hipStreamSynchronize(s->stream));
  });
}

// e = network correction of residual r (original numbering, FP64 in and out)
int phase_hip_learned_apply(phase_hip_solver *s, const double *r, double *e) {
  return guardedG(s, [&] {
    requireSystem(s);
    PH_CHECK(hipSetDevice(s->device));
    gnnPrepare(s);
    const int n = s->rank;
    DBuf<double> &tmp = s->gnn->stage;
    tmp.alloc(3 * (size_t)n);
    PH_CHECK(hipMemcpyAsync(tmp.p, r, n * sizeof(double), hipMemcpyHostToDevice, s->stream));
    hipLaunchKernelGGL((kPermuteIn<double, double>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p, tmp.p,
                       tmp.p + n, 1.0);
    applyNet(s, tmp.p + n, tmp.p + 2 * n);
    hipLaunchKernelGGL((kPermuteOut<double>), dim3(g1(n)), dim3(256), 0, s->stream, n, s->dPerm.p, tmp.p + 2 * n, tmp.p);
    PH_CHECK(hipMemcpyAsync(e, tmp.p, n * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    PH_CHECK(hipStreamSynchronize(s->stream));
  });
}

}  // extern "C"
