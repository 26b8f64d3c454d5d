// Linear elasticity operator (3 dofs per node) of libdendrohip: the reference's
// ElasticityMatMult (examples/src/backend/elasticityJac.C:129-211),
//   y_k = sum_j fac (mu L[k][j] I + (mu + lambda) GD[3k..3k+2][3j..3j+2]) x_j,  fac = h/2,
// with optional Dirichlet flags (boundary rows y = x, boundary columns dropped).
//
// Owner-computes tiles as for the scalar operator (tiles.cpp plan; one workgroup per tile):
// the tile's touched nodes' three components are staged in LDS, every record (own and halo
// elements) is evaluated, the rows of the nodes the tile owns are accumulated with 64-bit
// fixed-point LDS additions, and each owned node is stored once (no global atomics, no
// zeroing of y, bit-reproducible).
// Element matrices: child c's element is child 0's with the vertex order k^c (the plan's
// vertex permutation) and the signs s_a s_b on the (a, b) blocks (s_a = -1 when bit a of c is
// set: the mirror flips axis a).  Child 0's element of hanging mask H is the regular one
// constrained by the interpolation P_H of its hanging vertices, K_H = P_H^T K_0 P_H (kernels.hpp).
// K_0 is applied in the Walsh-Hadamard modes of its three components (bit a of a mode: difference
// along axis a): the Laplacian and the (a, a) blocks are diagonal there, and the (a, b) block,
// d_a phi_k d_b phi_j, is one entry per pair of modes, from mode n ^ a ^ b (bit a clear, bit b
// set) of component b to mode n (bit a set, bit b clear) of component a: 24 + 12 products and
// 144 additions instead of 576 FMAs with the matrix rows read through the scalar cache.  Every
// lane uses the same seven constants (ElasModes), whatever its element's type; the mirror signs
// fall on the 12 coupling products only, and the element's size on the final conversion.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "kernels.hpp"
#include "vector_kernels.hpp"

namespace dgh {

constexpr int ELAS_NSTRIDE = 24;   // LDS bytes per node: three doubles (sums or staged x)

// Threads per tile, owned-node capacity and node budget (owned capacity + touched nodes) of an
// elasticity tile: 128 registers allow 16 wavefronts per CU, as two 512-thread workgroups with
// half a CU's LDS each (24 B per node slot); 256 threads and a quarter of the LDS take 18% more at 17k
// elements, 2 to 7% more from 90k on.  Products of 13k / 119k / 318k / 657k elements, tiles of
// elas_tile_elems, same buffers: 5.9 / 12.4 / 20.3 / 30.9 us; before (24x24 matrix rows, 256 threads, 2200
// slots) 37.1 / 38.0 / 49.7 / 84.8.  With another mesh and vectors each time, 318k: 63.3 -> 20.6.
// It is bound by its 48 LDS operations per record (about 530 cycles per 64 records and CU: 20 us
// at 1.0M elements) and, at as much again, by its vector instructions.
constexpr int ELAS_BLOCK = 512;
constexpr uint32_t ELAS_OWN_CAP = 1024u;
constexpr uint32_t ELAS_BUDGET = 3360u;
// touched and owned nodes per thread
constexpr int ELAS_XC = int((ELAS_BUDGET - ELAS_OWN_CAP + ELAS_BLOCK - 1) / ELAS_BLOCK);
constexpr int ELAS_OC = int((ELAS_OWN_CAP + ELAS_BLOCK - 1) / ELAS_BLOCK);
constexpr uint32_t ELAS_XS_OFF = ELAS_NSTRIDE * ELAS_OWN_CAP + 64u;
__host__ constexpr size_t elas_lds_bytes(uint32_t max_touch) {
  return size_t(ELAS_XS_OFF) + size_t(ELAS_NSTRIDE) * max_touch;
}

// K_0 = mu L + (mu + lambda) GD of the unit-size element over its modes (factor 1/8 of the
// inverse transform included): d0[p], d1[p] = the diagonal of component a at a mode of p
// difference axes with bit a clear / set; o[bit] = the coupling with third axis sum / difference.
// big: staged values from 2^big on are scaled by 2^-ELAS_UP first (fx_big; here the modes multiply the
// transformed values before the last scale, so the modulus of K_0 counts: sums of a row's modes reach
// 68 times the largest, and the rows themselves at least that one).
struct ElasModes {
  double d0[4], d1[4], o[2];
  int big;
};
constexpr int ELAS_UP = 8;
__host__ inline ElasModes elas_modes(double mu, double lam) {
  ElasModes m{};
  for (int p = 1; p <= 3; ++p) {
    double c = 2.0 / 8.0;   // 2 (1/6)^(p-1) (1/2)^(3-p) / 8
    for (int i = 1; i < p; ++i) c /= 6.0;
    for (int i = p; i < 3; ++i) c /= 2.0;
    m.d0[p] = mu * p * c;
    m.d1[p] = mu * p * c + (mu + lam) * c;
  }
  m.o[0] = (mu + lam) / 16.0;
  m.o[1] = (mu + lam) / 48.0;
  int e = 0;
  std::frexp(std::max(std::fabs(m.d0[1]), std::fabs(m.d1[1])), &e);   // the largest modes: p = 1
  m.big = fx_top<double>() - std::max(0, e + 4);
  return m;
}

// v with its sign flipped by bit 31 of s
__device__ __forceinline__ double flip_sign(double v, uint32_t s) {
  return __longlong_as_double(__double_as_longlong(v) ^ (static_cast<long long>(s & 0x80000000u) << 32));
}

// v <- W v
__device__ __forceinline__ void wht8(double v[8]) {
#pragma unroll
  for (int b = 1; b < 8; b <<= 1)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (!(i & b)) {
        const double s = v[i] + v[i | b];
        v[i | b] = v[i] - v[i | b];
        v[i] = s;
      }
}

// A record: 8 tile-local vertex ids in 14 bits, its hanging vertices in the top bits of ids 5..7
// (rec_hang), the mirror signs s_x s_y, s_y s_z, s_z s_x in bits 14, 15 and 30 of the first word,
// the level's low four bits in the second word's spare bits and its fifth in bit 31 of the first.
__host__ inline void elas_pack(uint16_t id[8], uint32_t mask, uint32_t child, uint32_t lev) {
  const uint32_t hb = hang_bits(mask);
  const uint32_t sg = ((child ^ (child >> 1)) & 1u) | ((((child >> 1) ^ (child >> 2)) & 1u) << 1) |
                      (((child >> 2) ^ child) & 1u) << 2;
  const uint32_t top[8] = {sg & 3u, (sg >> 2) | ((lev >> 4) << 1), lev & 3u, (lev >> 2) & 3u, 0u,
                           hb & 3u, (hb >> 2) & 3u, (hb >> 4) & 3u};
  for (int q = 0; q < 8; ++q) id[q] = uint16_t(id[q] | (top[q] << 14));
}
__device__ __forceinline__ uint32_t elas_level(uint4 lp) {
  return ((lp.y >> 14) & 3u) | ((lp.y >> 28) & 12u) | ((lp.x >> 27) & 16u);
}

// texp[t]: exponent bound of the tile's
// row sums of |h K_H| and log2 bound of the terms per node (as for the scalar operator).
__global__ void __launch_bounds__(ELAS_BLOCK)
elas_tile_kernel(const TileRec* __restrict__ tiles, int ntiles, const uint16_t* __restrict__ lid,
                 const uint32_t* __restrict__ node_tab,
                 const int2* __restrict__ texp, ElasModes md, uint32_t maxD, double hFac,
                 const uint8_t* __restrict__ bdy, const double* __restrict__ x, double* __restrict__ y) {
  constexpr int BLOCK = ELAS_BLOCK;
  constexpr int NW = BLOCK / 64;
  constexpr uint32_t XS = ELAS_XS_OFF;
  static_assert(NW <= 16, "one max |x| word per wavefront in 64 LDS bytes");
  static_assert(XS + 16u <= 65535u, "staged x must start within the ds immediate offset range");
  const lds_ptr<uint32_t> s_xhi = lds_at<uint32_t>(ELAS_NSTRIDE * ELAS_OWN_CAP);
  const int t = xcd_tile(blockIdx.x, ntiles);
  if (t >= ntiles) return;
  const TileRec rec = tiles[t];
  const uint32_t* nodes = node_tab + rec.node_off;
  const uint32_t n_own = rec.n_own;
  // the wavefront's records: w0, w0 + BLOCK, ...; lanes past the last record load it again and
  // add nothing
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t w0 = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x - lane)));
  auto load = [&](uint32_t r0) {
    return reinterpret_cast<const uint4*>(lid)[rec.elem_off + min(r0 + lane, rec.n_elem - 1u)];
  };
  uint4 lp = load(w0);
  // stage the touched nodes' x (boundary nodes as 0: their columns drop out); indexes past the
  // end are clamped, so that all loads go out together
  uint32_t nid[ELAS_XC];
  const uint32_t last = rec.n_touch - 1u;
#pragma unroll
  for (int q = 0; q < ELAS_XC; ++q) nid[q] = nodes[min(threadIdx.x + uint32_t(q * BLOCK), last)];
  uint32_t xhi = 0, own_bdy = 0;
  double v[ELAS_XC][3];
#pragma unroll
  for (int q = 0; q < ELAS_XC; ++q)
#pragma unroll
    for (int a = 0; a < 3; ++a) v[q][a] = x[3 * size_t(nid[q]) + a];
  if (bdy) {
#pragma unroll
    for (int q = 0; q < ELAS_XC; ++q)
      if (bdy[nid[q]]) {
        v[q][0] = v[q][1] = v[q][2] = 0.0;
        own_bdy |= 1u << q;
      }
  }
#pragma unroll
  for (int q = 0; q < ELAS_XC; ++q) {
    const uint32_t i = threadIdx.x + uint32_t(q * BLOCK);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (i < rec.n_touch) *lds_at<double>(XS + ELAS_NSTRIDE * i + 8u * a) = v[q][a];
      xhi = max(xhi, uint32_t(uint64_t(__double_as_longlong(v[q][a])) >> 32) & 0x7fffffffu);
    }
  }
  for (uint32_t i = threadIdx.x; i < 3 * n_own; i += BLOCK) lds_at<unsigned long long>(0)[i] = 0ull;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) xhi = max(xhi, uint32_t(__shfl_xor(int(xhi), off)));
  if ((threadIdx.x & 63) == 0) s_xhi[threadIdx.x >> 6] = xhi;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) xhi = max(xhi, s_xhi[w]);
  const bool finite = (xhi >> 20) < 0x7ffu;
  const int ex = fx_ex<double>(xhi);
  const int es = fx_scale<double>(texp[t], ex);
  const bool big = __builtin_amdgcn_readfirstlane(ex) > md.big;
  const uint32_t own_bytes = n_own * ELAS_NSTRIDE;
  double quarter = 0.25;
  asm("" : "+s"(quarter));
  for (uint32_t r0 = w0; r0 < rec.n_elem; r0 += BLOCK) {
    const uint4 lpn = load(r0 + BLOCK);   // in flight during the evaluation
    const uint32_t w[4] = {lp.x, lp.y, lp.z, lp.w};
    uint32_t l[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) l[j] = ((w[j >> 1] >> (16 * (j & 1))) & REC_ID_MASK) * ELAS_NSTRIDE;
    const uint32_t hb = rec_hang(lp);
    // one component after the other (the fences keep the three from being interleaved, which
    // takes 138 registers instead of 128)
    double xe[3][8];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
      for (int k = 0; k < 8; ++k) xe[a][k] = *lds_at<double>(XS + l[k] + 8u * a);
      if (big) {
        DGH_NO_SELECT;
#pragma unroll
        for (int k = 0; k < 8; ++k) xe[a][k] *= 1.0 / (1 << ELAS_UP);
      }
      hang_interp(reinterpret_cast<double(&)[1][8]>(xe[a]), hb, quarter);
      wht8(xe[a]);
      __builtin_amdgcn_sched_barrier(0);
    }
    const uint32_t sg[3] = {lp.x << 17, lp.x << 16, lp.x << 1};   // mirror signs of (x,y), (y,z), (z,x)
    // modes, in place
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int A = 1 << a, B = 1 << (a + 1) % 3, C = 1 << (a + 2) % 3;
      xe[a][B] *= md.d0[1];
      xe[a][C] *= md.d0[1];
      xe[a][B | C] *= md.d0[2];
      xe[a][7] *= md.d1[3];
      // (a, A|C) and (b, B|C): third axis c, difference; the mirror's sign s_a s_b
      const int b = (a + 1) % 3;
      const double o = flip_sign(md.o[1], sg[a]);
      const double u = xe[a][A | C], v2 = xe[b][B | C];
      xe[a][A | C] = md.d1[2] * u + o * v2;
      xe[b][B | C] = md.d1[2] * v2 + o * u;
    }
    {   // (x, 1), (y, 2), (z, 4): third axis sum
      const double oxy = flip_sign(md.o[0], sg[0]), oyz = flip_sign(md.o[0], sg[1]), ozx = flip_sign(md.o[0], sg[2]);
      const double u = xe[0][1], v2 = xe[1][2], z = xe[2][4];
      xe[0][1] = md.d1[1] * u + (oxy * v2 + ozx * z);
      xe[1][2] = md.d1[1] * v2 + (oxy * u + oyz * z);
      xe[2][4] = md.d1[1] * z + (ozx * u + oyz * v2);
    }
    // the element's size h and 2^es in one scale
    const double sc = ldexp(hFac, int(maxD - elas_level(lp)) + (big ? es + ELAS_UP : es));
    const uint32_t own = r0 + lane < rec.n_elem ? own_bytes : 0u;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      double* y8 = xe[a];
      y8[0] = y8[1];   // first step of the inverse transform: the mean mode is zero
      y8[1] = -y8[1];
#pragma unroll
      for (int b = 1; b < 8; b <<= 1)
#pragma unroll
        for (int i = b == 1 ? 2 : 0; i < 8; ++i)
          if (!(i & b)) {
            const double s = y8[i] + y8[i | b];
            y8[i | b] = y8[i] - y8[i | b];
            y8[i] = s;
          }
      hang_interp_t(reinterpret_cast<double(&)[1][8]>(xe[a]), hb, quarter);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (l[k] < own) lds_add(lds_at<unsigned long long>(l[k] + 8u * a), fx_round_fma(y8[k], sc));
      __builtin_amdgcn_sched_barrier(0);
    }
    lp = lpn;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < ELAS_OC; ++q) {
    const uint32_t i = threadIdx.x + uint32_t(q * BLOCK);
    if (i >= n_own) break;
    const uint32_t n = nid[q];
    const bool b = (own_bdy >> q) & 1u;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double s = fx_value<double>(lds_at<unsigned long long>(0)[3 * i + a], es);
      y[3 * size_t(n) + a] = b ? x[3 * size_t(n) + a] : (finite ? s : __builtin_nan(""));
    }
  }
}

}  // namespace dgh
