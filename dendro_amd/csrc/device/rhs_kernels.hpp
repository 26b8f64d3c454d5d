// Kernels that evaluate functions at element points: quadrature right-hand sides, nodal values
// and L2 errors (the reference's ComputeRHS2 / ComputeSol / ComputeError5 loops,
// examples/src/backend/omgRhs.C).  One thread per element; elements are located by their DA
// anchor and level; the unit cube is DA coordinates / 2^(maxD-1).
//
// The quadrature kernels work in child 0's frame: the axes of a mirrored child run backwards, so
// the Gauss nodes keep their tensor order and the shape functions of a hanging element are the
// trilinear ones through P_H (kernels.hpp).  Sums over the 27 nodes are factored by axis (114
// products against 216 with a table of hanging shape functions, and no table reads).
#pragma once

#include <hip/hip_runtime.h>

#include "dendro_hip.h"
#include "kernels.hpp"
#include "vector_kernels.hpp"

namespace dgh {

constexpr int NQ = 27;   // 3x3x3 Gauss nodes, index 9 m + 3 n + p (m along x)

struct FnDev {
  int kind, nfreq;
  double a0, a1;
  double c[8];
};

// the Gaussians (the three boxes are disjoint) or the polynomial
__device__ __forceinline__ double eval_other(const FnDev& f, double x, double y, double z) {
  if (f.kind == DGH_FN_GAUSSIANS) {
    double mid = 0.0;
    if (x >= 0.0 && y >= 0.0 && z >= 0.0 && x < 0.2 && y < 0.2 && z < 0.2) mid = 0.1;
    if (x >= 0.2 && y >= 0.2 && z >= 0.2 && x <= 0.4 && y <= 0.4 && z <= 0.4) mid = 0.3;
    if (x >= 0.5 && y >= 0.5 && z >= 0.5 && x <= 0.7 && y <= 0.7 && z <= 0.7) mid = 0.6;
    if (mid == 0.0) return 0.0;
    const double dx = x - mid, dy = y - mid, dz = z - mid;
    return exp(-((dx * dx + dy * dy + dz * dz) / 0.005));
  }
  return f.c[0] + f.c[1] * x + f.c[2] * y + f.c[3] * z + f.c[4] * x * y + f.c[5] * y * z + f.c[6] * z * x +
         f.c[7] * x * y * z;
}

__device__ __forceinline__ double eval_fn(const FnDev& f, double x, double y, double z) {
  if (f.kind != DGH_FN_COS_SUM) return eval_other(f, x, y, z);
  const double pi = 3.14159265358979323846;
  double r = 0.0;
  for (int k = 1; k <= f.nfreq; ++k) {
    const double kk = double(k);
    r += (f.a0 + 3.0 * f.a1 * kk * kk * pi * pi) * cos(kk * pi * x) * cos(kk * pi * y) * cos(kk * pi * z);
  }
  return r;
}

// Gauss node t (0..2) of the 3-point rule on [-1, 1]: {0, +sqrt(3/5), -sqrt(3/5)}, weights
// {8/9, 5/9, 5/9}
__device__ __forceinline__ double gauss_pt(int t) {
  return t == 0 ? 0.0 : (t == 1 ? 0.77459666924148337704 : -0.77459666924148337704);
}
__device__ __forceinline__ double gauss_wt(int t) { return t == 0 ? 8.0 / 9.0 : 5.0 / 9.0; }

struct ElemGeo {
  double x, y, z, h;
};
// geo: anchor x, y, z and level | child << 8 | hang_bits << 16 (fem_api.hip)
__device__ __forceinline__ ElemGeo elem_geo(int4 a, uint32_t maxD) {
  const double unit = 1.0 / double(1u << (maxD - 1));
  return ElemGeo{double(a.x) * unit, double(a.y) * unit, double(a.z) * unit,
                 double(1u << (maxD - (uint32_t(a.w) & 0xffu))) * unit};
}
__device__ __forceinline__ double gauss_at(double x, double h, int t) { return h * (1.0 + gauss_pt(t)) * 0.5 + x; }

// The cosine sum's factors cos(k pi x) at an element's Gauss nodes depend on one coordinate
// interval (coordinate, level) only, and the consecutive elements of a workgroup share few of them
// (256 elements of a cluster about 40 to 100, against 768): the workgroup lists its distinct
// intervals in LDS and evaluates each factor once, for as many frequencies at a time as FQ_VALS
// holds (8 up to 128 intervals, 1 at the most, 768).
constexpr int FQ_SLOTS = 1024;          // hash slots of the interval list
constexpr int FQ_LIST = 3 * VBLOCK;     // three intervals per element
constexpr int FQ_VALS = 1024, FQ_K = 8;
static_assert(FQ_LIST < FQ_SLOTS && FQ_LIST <= FQ_VALS, "every interval finds a slot and room for one frequency");
struct FnShared {
  uint32_t key[FQ_SLOTS];
  uint16_t idx[FQ_SLOTS];
  uint32_t list[FQ_LIST];
  uint32_t n;
  double v[FQ_VALS][3];                 // [interval][frequency of this pass][Gauss node]
};

// f[9 m + 3 n + p] = the function at the 27 Gauss nodes of this thread's element, in child 0's
// order; called by the whole workgroup (in: whether the thread has an element).  COS: the cosine
// sum, else the other functions.
template <bool COS>
__device__ __forceinline__ void eval_nodes(const FnDev& fn, bool in, int4 a, uint32_t maxD, FnShared& sh, double f[NQ]) {
  const uint32_t c = (uint32_t(a.w) >> 8) & 7u, lev = uint32_t(a.w) & 0xffu;
  // Gauss node of child 0's node t along axis b: mirrored axes swap the outer two
  auto node = [&](int t, int b) { return t == 0 ? 0 : ((c >> b) & 1u) ? 3 - t : t; };
#pragma unroll
  for (int q = 0; q < NQ; ++q) f[q] = 0.0;
  if constexpr (!COS) {
    const ElemGeo G = elem_geo(a, maxD);
    if (in)
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        f[q] = eval_other(fn, gauss_at(G.x, G.h, node(q / 9, 0)), gauss_at(G.y, G.h, node(q / 3 % 3, 1)),
                          gauss_at(G.z, G.h, node(q % 3, 2)));
    return;
  }
  for (int i = threadIdx.x; i < FQ_SLOTS; i += VBLOCK) sh.key[i] = 0u;
  if (threadIdx.x == 0) sh.n = 0u;
  __syncthreads();
  const int co[3] = {a.x, a.y, a.z};
  uint32_t slot[3] = {0u, 0u, 0u};
  if (in) {
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      const uint32_t key = ((uint32_t(co[b]) << 5) | lev) + 1u;
      uint32_t s = (key * 2654435761u) >> 22;
      for (;;) {   // ends: at most 768 of the 1024 slots are taken
        const uint32_t old = atomicCAS(&sh.key[s], 0u, key);
        if (old == 0u) {
          const uint32_t i = atomicAdd(&sh.n, 1u);
          sh.idx[s] = uint16_t(i);
          sh.list[i] = key - 1u;
        }
        if (old == 0u || old == key) break;
        s = (s + 1u) & (FQ_SLOTS - 1u);
      }
      slot[b] = s;
    }
  }
  __syncthreads();
  const uint32_t nint = sh.n, per = min(uint32_t(FQ_K), uint32_t(FQ_VALS) / nint);   // frequencies per pass
  uint32_t row[3];
#pragma unroll
  for (int b = 0; b < 3; ++b) row[b] = in ? sh.idx[slot[b]] * per : 0u;
  const double pi = 3.14159265358979323846;
  const double unit = 1.0 / double(1u << (maxD - 1));
  for (int k0 = 1; k0 <= fn.nfreq; k0 += int(per)) {
    const uint32_t nk = min(per, uint32_t(fn.nfreq - k0 + 1));
    for (uint32_t i = threadIdx.x; i < nint * 3u * nk; i += VBLOCK) {
      const uint32_t e = i / (3u * nk), r = i % (3u * nk), t = r % 3u, k = r / 3u, key = sh.list[e];
      const double X = gauss_at(double(key >> 5) * unit, double(1u << (maxD - (key & 31u))) * unit, int(t));
      sh.v[e * per + k][t] = cos(double(k0 + int(k)) * pi * X);
    }
    __syncthreads();
    if (in)
      for (uint32_t k = 0; k < nk; ++k) {
        const double kk = double(k0 + int(k));
        const double ck = fn.a0 + 3.0 * fn.a1 * kk * kk * pi * pi;
        double cv[3][3];
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
          for (int t = 0; t < 3; ++t) cv[b][t] = sh.v[row[b] + k][node(t, b)];
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
          for (int n = 0; n < 3; ++n) {
            const double w = ck * cv[0][m] * cv[1][n];
#pragma unroll
            for (int p = 0; p < 3; ++p) f[9 * m + 3 * n + p] += w * cv[2][p];
          }
      }
    __syncthreads();   // the next frequencies overwrite the factors
  }
}

// One-dimensional shape functions at the Gauss nodes 0, +g, -g: lower vertex 1/2, FS, FL, upper
// vertex 1/2, FL, FS.
constexpr double FS = 0.11270166537925831148, FL = 0.88729833462074168852;

// LDS list of a workgroup's nodes with their sums: at most 8 VBLOCK of RQ_SLOTS are taken
constexpr int RQ_SLOTS = 4096;
struct NodeShared {
  uint32_t key[RQ_SLOTS];
  double sum[RQ_SLOTS];
};
union RhsShared {
  FnShared fn;
  NodeShared nd;
};

// b[idx[j]] += h^3/8 sum_q w_q f(x_q) S[s][j][q]  (b zeroed by the caller).  A workgroup first adds
// its elements' terms in LDS, by node, then makes one device addition per node it touches (about a
// fifth of the 8 per element: additions to memory run at about 32 per nanosecond device-wide).
// 318k elements, nine cosines, 504 us with the factors and the shape-function table read per
// element and node and an addition to memory per vertex -> 36 us.
template <bool COS>
__global__ void __launch_bounds__(VBLOCK)
rhs_quad_kernel(uint32_t E, uint32_t maxD, const int4* __restrict__ geo, const uint32_t* __restrict__ nl, FnDev fn,
                double* __restrict__ b) {
  extern __shared__ __align__(16) unsigned char smem_fn[];
  RhsShared& sh = *reinterpret_cast<RhsShared*>(smem_fn);
  const uint32_t e = blockIdx.x * VBLOCK + threadIdx.x;
  const bool in = e < E;
  const int4 a = geo[min(e, E - 1u)];
  double f[NQ];
  eval_nodes<COS>(fn, in, a, maxD, sh.fn, f);
  __syncthreads();
  for (int i = threadIdx.x; i < RQ_SLOTS; i += VBLOCK) {
    sh.nd.key[i] = 0u;
    sh.nd.sum[i] = 0.0;
  }
  __syncthreads();
  if (in) {
    constexpr double W0 = 4.0 / 9.0, WS = 5.0 / 9.0 * FS, WL = 5.0 / 9.0 * FL;   // weight times shape function
    double g1[9][2], g2[3][2][2], v[1][8];
#pragma unroll
    for (int q = 0; q < 9; ++q) {   // over p (z)
      g1[q][0] = W0 * f[3 * q] + WS * f[3 * q + 1] + WL * f[3 * q + 2];
      g1[q][1] = W0 * f[3 * q] + WL * f[3 * q + 1] + WS * f[3 * q + 2];
    }
#pragma unroll
    for (int m = 0; m < 3; ++m)     // over n (y)
#pragma unroll
      for (int z = 0; z < 2; ++z) {
        g2[m][0][z] = W0 * g1[3 * m][z] + WS * g1[3 * m + 1][z] + WL * g1[3 * m + 2][z];
        g2[m][1][z] = W0 * g1[3 * m][z] + WL * g1[3 * m + 1][z] + WS * g1[3 * m + 2][z];
      }
#pragma unroll
    for (int y = 0; y < 2; ++y)     // over m (x)
#pragma unroll
      for (int z = 0; z < 2; ++z) {
        v[0][2 * y + 4 * z] = W0 * g2[0][y][z] + WS * g2[1][y][z] + WL * g2[2][y][z];
        v[0][1 + 2 * y + 4 * z] = W0 * g2[0][y][z] + WL * g2[1][y][z] + WS * g2[2][y][z];
      }
    double quarter = 0.25;
    asm("" : "+s"(quarter));
    hang_interp_t(v, (uint32_t(a.w) >> 16) & 63u, quarter);
    const ElemGeo G = elem_geo(a, maxD);
    const double fac = G.h * G.h * G.h / 8.0;
    const uint32_t c = (uint32_t(a.w) >> 8) & 7u;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t key = nl[size_t(e) * 8 + (uint32_t(k) ^ c)] + 1u;
      uint32_t s = (key * 2654435761u) >> 20;
      for (;;) {   // ends: at most 2048 of the 4096 slots are taken
        const uint32_t old = atomicCAS(&sh.nd.key[s], 0u, key);
        if (old == 0u || old == key) break;
        s = (s + 1u) & (RQ_SLOTS - 1u);
      }
      atomic_add(&sh.nd.sum[s], fac * v[0][k]);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < RQ_SLOTS; i += VBLOCK)
    if (sh.nd.key[i]) atomic_add(&b[sh.nd.key[i] - 1u], sh.nd.sum[i]);
}

// u[node] = f(node) over the non-hanging vertices of every element (equal values when written
// twice)
__global__ void __launch_bounds__(VBLOCK)
nodal_values_kernel(uint32_t E, uint32_t maxD, const int4* __restrict__ geo, const uint32_t* __restrict__ nl,
                    const uint8_t* __restrict__ hn, FnDev f, double* __restrict__ u) {
  const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= E) return;
  const ElemGeo G = elem_geo(geo[e], maxD);
  const uint8_t mask = hn[e];
  for (int k = 0; k < 8; ++k) {
    if (mask & (1u << k)) continue;
    u[nl[size_t(e) * 8 + k]] =
        eval_fn(f, G.x + double(k & 1) * G.h, G.y + double((k >> 1) & 1) * G.h, G.z + double((k >> 2) & 1) * G.h);
  }
}

// part[block] = sum over the block's elements of h^3/8 sum_q w_q (f(x_q) - u_h(x_q))^2, in a
// fixed order (chunks of VBLOCK elements per block, wavefront sums, then the block)
template <bool COS>
__global__ void __launch_bounds__(VBLOCK)
l2_error_kernel(uint32_t E, uint32_t maxD, const int4* __restrict__ geo, const uint32_t* __restrict__ nl, FnDev fn,
                const double* __restrict__ u, double* __restrict__ part) {
  __shared__ FnShared sh;
  double tot = 0.0;
  double quarter = 0.25;
  asm("" : "+s"(quarter));
  for (uint32_t e0 = blockIdx.x * VBLOCK; e0 < E; e0 += gridDim.x * VBLOCK) {
    const uint32_t e = e0 + threadIdx.x;
    const bool in = e < E;
    const int4 a = geo[min(e, E - 1u)];
    double v[1][8];   // nodal values in child 0's order, loaded while the function is evaluated
    const uint32_t c = (uint32_t(a.w) >> 8) & 7u;
#pragma unroll
    for (int k = 0; k < 8; ++k) v[0][k] = u[nl[size_t(min(e, E - 1u)) * 8 + (uint32_t(k) ^ c)]];
    double f[NQ];
    eval_nodes<COS>(fn, in, a, maxD, sh, f);
    if (in) {
      hang_interp(v, (uint32_t(a.w) >> 16) & 63u, quarter);
      // u_h at the nodes, axis by axis: x (vertex bit 0), y, z
      double hx[3][4], acc = 0.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double lo = v[0][2 * q], up = v[0][2 * q + 1];
        hx[0][q] = 0.5 * (lo + up);
        hx[1][q] = FS * lo + FL * up;
        hx[2][q] = FL * lo + FS * up;
      }
#pragma unroll
      for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int n = 0; n < 3; ++n) {
          const double ln = n == 0 ? 0.5 : n == 1 ? FS : FL, un = n == 0 ? 0.5 : n == 1 ? FL : FS;
          const double z0 = ln * hx[m][0] + un * hx[m][1], z1 = ln * hx[m][2] + un * hx[m][3];
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            const double lp = p == 0 ? 0.5 : p == 1 ? FS : FL, upp = p == 0 ? 0.5 : p == 1 ? FL : FS;
            const double d = f[9 * m + 3 * n + p] - (lp * z0 + upp * z1);
            acc += gauss_wt(m) * gauss_wt(n) * gauss_wt(p) * d * d;
          }
        }
      const ElemGeo G = elem_geo(a, maxD);
      tot += acc * (G.h * G.h * G.h / 8.0);
    }
    __syncthreads();   // the next chunk rebuilds the interval list
  }
  __shared__ double red[VBLOCK / 64];
  tot = wave_sum(tot);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = tot;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < VBLOCK / 64; ++w) t += red[w];
    part[blockIdx.x] = t;
  }
}

}  // namespace dgh
