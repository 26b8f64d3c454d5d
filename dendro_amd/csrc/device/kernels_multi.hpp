// Batched (multi right-hand side) kernels of libdendrohip.
//
// k right-hand sides are stored node-major: X[n * k + j], so the k values of a node are one
// contiguous row and every node gather is a coalesced row segment.  The operator kernel
// keeps the owner-computes tiling of the single right-hand-side kernel; one workgroup
// handles one tile and one slice of right-hand sides, staging the slice of every touched
// node in LDS.  The element products Y_e = K_e X_e ([8x8] x [8 x slice]) run on the vector
// ALUs (tile_multi_kernel, FP32 and FP64) or, as an FP32 variant, on the matrix cores as
// v_mfma_f32_4x4x1_16b_f32 (tile_multi_mfma_kernel: 16 independent 4x4 blocks per
// instruction, 4 elements x 2 row blocks x 2 column blocks); the autotuner picks the FP32
// variant per mesh.  Row sums of owned nodes accumulate in LDS and are stored once per node.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "kernels.hpp"
#include "vector_kernels.hpp"

namespace dgh {

constexpr int KS = 8;            // right-hand sides per workgroup slice (FP32)
constexpr int KS64 = 4;          // right-hand sides per workgroup slice (FP64: same LDS bytes)
constexpr int MAXK = 32;         // right-hand sides per batch
constexpr int MBLOCK = 512;      // threads per batched-operator workgroup

template <class T>
struct MultiIO {
  const T* x;      // [N][k] operator input
  T* y;            // [N][k] output
  const T* b;      // [N][k] right-hand sides (RESID, SMOOTH)
  const T* invd;   // [N] inverse diagonal (SMOOTH)
  T omega;         // Richardson scale (SMOOTH)
  int k;           // right-hand sides per node row
  double* part;    // CG: per tile and column, the owned nodes' partial of x.y ([ntiles][k])
};

typedef float mfma_f4 __attribute__((ext_vector_type(4)));

// 16-byte vectors of the gathers and stores: 4 FP32 or 2 FP64 values
template <class T> struct Vec16;
template <> struct Vec16<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct Vec16<double> { typedef double type __attribute__((ext_vector_type(2))); };
template <class T> using vec16_t = typename Vec16<T>::type;

// Vector-ALU batched operator.  Lane = (element of the round, CPL adjacent right-hand sides
// c .. c + CPL - 1 of the slice): the KSL / CPL lanes of an element share its record, read
// the element's 8 node values of their columns from LDS, apply the factored element product
// (fact_product, kernels.hpp) and accumulate its 8 rows, so LDS carries only the minimum per
// element and column: 8 reads and at most 8 additions, while the record, its hanging vertices,
// the mode factors and the LDS addresses are shared by the CPL columns of a lane.  Sums
// accumulate in fixed point as in the single right-hand-side kernel (64-bit integers for
// FP64, 32-bit for FP32), with one scale per column of the slice; two adjacent FP32 columns of a
// lane are added as one 64-bit integer (PACK).  Gathers and stores move 16-byte vectors of a
// node's slice.  LDS rows are padded so the lanes of different elements spread over the banks.
// FP32, k = 32, 630k elements with a coefficient, launches on the same buffers: 318 us with stencil
// triangles in scalar registers (tiles of 1024, one column per lane) -> 145 us in tiles of 512, two
// columns per lane, FP64 397 -> 231; with another mesh and vectors each time, whose 118 MB come from
// memory, FP32 369 -> 163.  It is bound by the vector ALUs (95% of their issue slots): about 118 instructions per element
// and column, 56 of them the product, 24 the conversion and packing of the sums, the rest record
// unpacking, hanging vertices and addresses; 1.67 records per element (halo).  Eight
// columns per lane (the same), 256 or 1024 threads (15 and 11% more) do not pay.
// LDS: owned sums [ys_len][multi_row_y] (fixed point), touched x [max_touch][multi_row] (T).
template <class T>
__host__ __device__ constexpr int multi_row(int ksl) { return ksl + 1; }
template <class T>
__host__ __device__ constexpr int multi_row_y(int ksl) { return sizeof(T) == 4 ? ksl + 2 : ksl + 1; }

// Two FP32 columns' fixed-point terms as one 64-bit integer hi 2^32 + lo: sums of such integers
// hold both 32-bit sums exactly (neither overflows, see FX32_BITS): the low word is the lower
// column's, and the high word is the upper one's minus one where the lower one's is negative.
__device__ __forceinline__ unsigned long long fx_pack(unsigned int lo, unsigned int hi) {
  return (static_cast<unsigned long long>(hi + static_cast<unsigned int>(static_cast<int>(lo) >> 31)) << 32) | lo;
}

// One record for CPL columns.  n_own = 0 adds nothing; d[p]: the record's mode factors scaled by
// the tile's bound, cs[q]: the column's scale; big (uniform): see fx_big, cs holds 2^FX_UP then; node
// l's values sit at LDS byte address xb + l RSX sizeof(T) (x) and yb + l RSY sizeof(acc) (sums), one 24-bit multiply-add each
// (written out: the compiler shares l * stride between the two addresses and adds twice; the
// strides are at most 64, inline constants).
template <class T, bool MASS, int CPL, int RSX, int RSY, bool PACK>
__device__ __forceinline__ void eval_multi(uint4 lp, uint32_t n_own, const T d[4], const T cs[CPL], bool big,
                                           uint32_t xb, uint32_t yb) {
  using TA = fx_acc_t<T>;
  const uint32_t w[4] = {lp.x, lp.y, lp.z, lp.w};
  uint32_t l[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) l[j] = (w[j >> 1] >> (16 * (j & 1))) & REC_ID_MASK;
  const uint32_t hb = rec_hang(lp);
  T v[CPL][8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    uint32_t a;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(a) : "v"(l[j]), "n"(int(RSX * sizeof(T))), "v"(xb));
#pragma unroll
    for (int q = 0; q < CPL; ++q) v[q][j] = *lds_at<T>(a + q * uint32_t(sizeof(T)));
  }
  if (big) {
    DGH_NO_SELECT;
#pragma unroll
    for (int q = 0; q < CPL; ++q)
#pragma unroll
      for (int j = 0; j < 8; ++j) v[q][j] *= T(1.0 / (1 << FX_UP));
  }
  T quarter = T(0.25);
  asm("" : "+s"(quarter));
  hang_interp(v, hb, quarter);
#pragma unroll
  for (int q = 0; q < CPL; ++q) {
    T dq[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) dq[p] = d[p] * cs[q];
    fact_product<T, MASS>(v[q], dq);
  }
  hang_interp_t(v, hb, quarter);
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (l[k] < n_own) {
      uint32_t ya;
      asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(ya) : "v"(l[k]), "n"(int(RSY * sizeof(TA))), "v"(yb));
      if constexpr (PACK) {
#pragma unroll
        for (int q = 0; q < CPL; q += 2)
          lds_add(lds_at<unsigned long long>(ya + q * 4u), fx_pack(fx_round(v[q][k]), fx_round(v[q + 1][k])));
      } else {
#pragma unroll
        for (int q = 0; q < CPL; ++q) lds_add(lds_at<TA>(ya + q * uint32_t(sizeof(TA))), fx_round(v[q][k]));
      }
    }
}

template <class T, bool MASS, int MODE, int KSL, int MB, int CPL>
__global__ void __launch_bounds__(MB)
tile_multi_kernel(const TileRec* __restrict__ tiles, int ntiles, int nslices,
                  const uint16_t* __restrict__ lid,
                  const T* __restrict__ kappa, const T* __restrict__ mass, double lap_fac,
                  double mass_fac, uint32_t maxD, double hFac,
                  const uint32_t* __restrict__ node_tab, const int2* __restrict__ texp, uint32_t ys_len,
                  MultiIO<T> io) {
  static_assert(MODE != OP_DIAG, "the diagonal does not depend on the right-hand side");
  constexpr int LPE = KSL / CPL;              // lanes per element
  static_assert(KSL % CPL == 0 && 64 % LPE == 0, "a wavefront holds whole elements");
  using TA = fx_acc_t<T>;
  constexpr int RS = multi_row<T>(KSL), RSY = multi_row_y<T>(KSL);   // padded LDS rows
  constexpr bool PACK = sizeof(T) == 4 && CPL % 2 == 0;
  constexpr int NW = MB / 64;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ uint32_t s_xhi[NW][KSL];
  TA* ys = reinterpret_cast<TA*>(smem_raw);
  T* xs = reinterpret_cast<T*>(ys + size_t(ys_len) * RSY);
  const int np = ntiles * nslices;
  const int pidx = xcd_tile(blockIdx.x, np);   // the slices of a tile stay on one XCD
  if (pidx >= np) return;
  const int t = pidx / nslices, sl = pidx % nslices;
  const TileRec rec = tiles[t];
  const uint32_t* nodes = node_tab + rec.node_off;
  const uint32_t n_own = rec.n_own;
  const size_t k = size_t(io.k);
  // Gathers and stores move 16-byte vectors: LPN lanes cover the KSL columns of a node's
  // slice, VEC columns each (a thread keeps columns cv .. cv + VEC - 1 throughout, since MB
  // is a multiple of LPN).  Indexes past the end are clamped to the last node, so the MGU
  // node-id loads, then the MGU vector loads of a thread go out together with no branch.
  constexpr int VEC = 16 / int(sizeof(T));
  constexpr int LPN = KSL / VEC;
  static_assert(KSL % VEC == 0 && MB % LPN == 0, "whole vectors per node slice");
  using V = vec16_t<T>;
  const int cv = int(threadIdx.x % LPN) * VEC;
  uint32_t xhv[VEC];   // high words (FP32: bits) of max |x| of this thread's gather columns
#pragma unroll
  for (int e = 0; e < VEC; ++e) xhv[e] = 0u;
  // The owned nodes lead the tile's node list, so when they fit in the first batch of
  // gathers (keep), the thread's store nodes are the node ids of that batch: own_n.
  constexpr int MGU = 4;
  const uint32_t nv = rec.n_touch * LPN;
  const uint32_t nov = n_own * LPN;
  const bool keep = nov <= uint32_t(MGU * MB);
  uint32_t own_n[MGU];
#pragma unroll
  for (int u = 0; u < MGU; ++u) own_n[u] = 0u;
  const T* xsl = io.x + size_t(sl) * KSL + cv;
  for (uint32_t i0 = threadIdx.x; i0 < nv; i0 += MGU * MB) {
    uint32_t nid[MGU];
    V v[MGU];
#pragma unroll
    for (int u = 0; u < MGU; ++u) nid[u] = nodes[min(i0 + u * MB, nv - 1) / LPN];
    if (i0 == threadIdx.x)
#pragma unroll
      for (int u = 0; u < MGU; ++u) own_n[u] = nid[u];
#pragma unroll
    for (int u = 0; u < MGU; ++u) v[u] = *reinterpret_cast<const V*>(xsl + size_t(nid[u]) * k);
#pragma unroll
    for (int u = 0; u < MGU; ++u) {
      const uint32_t i = i0 + u * MB;
      if (i < nv) {
        T* d = xs + (i / LPN) * RS + cv;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          d[e] = v[u][e];
          if constexpr (sizeof(T) == 8)
            xhv[e] = max(xhv[e], uint32_t(uint64_t(__double_as_longlong(v[u][e])) >> 32) & 0x7fffffffu);
          else   // FP32 bits order as |x| does; the maximum is converted by col_exp
            xhv[e] = max(xhv[e], __float_as_uint(v[u][e]) & 0x7fffffffu);
        }
      }
    }
  }
  for (uint32_t i = threadIdx.x; i < n_own * RSY; i += MB) ys[i] = TA(0);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int es = lane / LPE, c = (lane % LPE) * CPL;   // element of the round, first column
#pragma unroll
  for (int off = 32; off >= LPN; off >>= 1)
#pragma unroll
    for (int e = 0; e < VEC; ++e) xhv[e] = max(xhv[e], uint32_t(__shfl_xor(int(xhv[e]), off)));
  if (lane < LPN)
#pragma unroll
    for (int e = 0; e < VEC; ++e) s_xhi[wv][cv + e] = xhv[e];
  __syncthreads();
  // Per column: max |x| < 2^ex; a non-finite column gives NaN.  A term's scale 2^(es0 - ex) is the
  // tile's part 2^es0, taken into the record's mode factors, times the column's cs = 2^-ex.
  auto col_hi = [&](int col) {   // high word of the column's max |x| in FP64
    uint32_t h = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) h = max(h, s_xhi[w][col]);
    if constexpr (sizeof(T) == 4) h = uint32_t(uint64_t(__double_as_longlong(double(__uint_as_float(h)))) >> 32);
    return h;
  };
  const int es0 = fx_scale<T>(texp[t], 0);
  // One column of fx_big scales the whole slice (a wavefront's lanes hold all its columns): for the
  // others that is exact too, but for bits below their grid.
  T cs[CPL];
  bool past = false;
#pragma unroll
  for (int q = 0; q < CPL; ++q) {
    const int ex = fx_ex<T>(col_hi(c + q));
    past = past || ex > fx_top<T>();
    cs[q] = T(ldexp(1.0, -ex));
  }
  const bool big = __ballot(past) != 0;
  if (big) {
    DGH_NO_SELECT;
#pragma unroll
    for (int q = 0; q < CPL; ++q) cs[q] *= T(1 << FX_UP);
  }
  // LDS byte addresses of the lane's first column in row 0 of the staged x and of the sums
  const uint32_t xbase = uint32_t(reinterpret_cast<uintptr_t>((lds_ptr<T>)(xs + c)));
  const uint32_t ybase = uint32_t(reinterpret_cast<uintptr_t>((lds_ptr<TA>)(ys + c)));
  constexpr uint32_t EPW = 64 / LPE;          // elements per wavefront round
  constexpr uint32_t STRIDE = (MB / 64) * EPW;
  // the records of the next round are loaded while the current round is evaluated; lanes past
  // the last record load it again and add nothing
  const double u1 = lap_fac * hFac / 2.0, u2 = mass_fac * hFac * hFac * hFac / 8.0;
  RecF<T> R;
  auto load = [&](uint32_t r0) {
    const uint32_t g = rec.elem_off + min(r0 + uint32_t(es), rec.n_elem - 1u);
    if (kappa)
      load_rec_fact<T, MASS, false>(R, g, lid, kappa, mass);
    else
      load_rec_fact<T, MASS, true>(R, g, lid, kappa, mass);
  };
  uint32_t r0 = uint32_t(__builtin_amdgcn_readfirstlane(wv)) * EPW;
  load(r0);
  for (; r0 < rec.n_elem; r0 += STRIDE) {
    const RecF<T> Rc = R;
    load(r0 + STRIDE);
    T f1, f2 = T(0);
    if (kappa) {
      f1 = T(ldexp(double(Rc.k1), es0));
      if (MASS) f2 = T(ldexp(double(Rc.k2), es0));
    } else {
      const int hs = int(maxD - (rec_class(Rc.lp) >> 5));
      f1 = T(ldexp(u1, hs + es0));
      if (MASS) f2 = T(ldexp(u2, 3 * hs + es0));
    }
    T d[4];
    fact_modes<T, MASS>(f1, f2, d);
    eval_multi<T, MASS, CPL, RS, RSY, PACK>(Rc.lp, r0 + uint32_t(es) < rec.n_elem ? n_own : 0u, d, cs, big, xbase, ybase);
  }
  // the store's right-hand sides and diagonals of the kept owned nodes: loaded before the
  // barrier, so they are in flight while the other wavefronts finish their records
  constexpr int MSU = MGU;
  const size_t so = size_t(sl) * KSL + cv;
  V bpre[MSU];
  T dpre[MSU];
  if ((MODE == OP_RESID || MODE == OP_SMOOTH) && keep) {
#pragma unroll
    for (int u = 0; u < MSU; ++u) {
      bpre[u] = *reinterpret_cast<const V*>(io.b + size_t(own_n[u]) * k + so);
      dpre[u] = MODE == OP_SMOOTH ? io.invd[own_n[u]] : T(0);
    }
  }
  __syncthreads();
  // scales of the thread's store columns cv + e
  int ess[VEC];
  bool fins[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    const uint32_t h = col_hi(cv + e);
    fins[e] = (h >> 20) < 0x7ffu;
    ess[e] = es0 - fx_ex<T>(h);
  }
  // stores: 16-byte vectors as in the gather, MSU (= MGU, the batch of own_n) per thread
  // with their loads in flight together
  double dot[VEC];   // CG: this thread's partials of x.y for its columns
#pragma unroll
  for (int e = 0; e < VEC; ++e) dot[e] = 0.0;
  for (uint32_t i0 = threadIdx.x; i0 < nov; i0 += MSU * MB) {
    uint32_t nid[MSU];
    V bv[MSU];
    T dv[MSU];
#pragma unroll
    for (int u = 0; u < MSU; ++u) nid[u] = keep ? own_n[u] : nodes[min(i0 + u * MB, nov - 1) / LPN];
#pragma unroll
    for (int u = 0; u < MSU; ++u) {
      if (keep) {
        bv[u] = bpre[u];
        dv[u] = dpre[u];
      } else {
        if (MODE == OP_RESID || MODE == OP_SMOOTH)
          bv[u] = *reinterpret_cast<const V*>(io.b + size_t(nid[u]) * k + so);
        dv[u] = MODE == OP_SMOOTH ? io.invd[nid[u]] : T(0);
      }
    }
#pragma unroll
    for (int u = 0; u < MSU; ++u) {
      const uint32_t i = i0 + u * MB;
      if (i >= nov) break;
      const uint32_t nd = i / LPN;
      V out;
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        TA sum = ys[nd * RSY + cv + e];
        if constexpr (PACK) {   // the upper column of a pair: see fx_pack
          if (e & 1) sum += TA(static_cast<int>(ys[nd * RSY + cv + e - 1]) < 0 ? 1 : 0);
        }
        const T v = fins[e] ? T(fx_value<T>(sum, ess[e])) : T(__builtin_nan(""));
        if (MODE == OP_MATVEC || MODE == OP_CG) out[e] = v;
        else if (MODE == OP_RESID) out[e] = bv[u][e] - v;
        else out[e] = xs[nd * RS + cv + e] + io.omega * ((bv[u][e] - v) * dv[u]);
        if (MODE == OP_CG) dot[e] += double(xs[nd * RS + cv + e]) * double(v);
      }
      *reinterpret_cast<V*>(io.y + size_t(nid[u]) * k + so) = out;
    }
  }
  if constexpr (MODE == OP_CG) {
    // the tile's partial of x.y per column, summed in a fixed order: over the lanes that
    // share the thread's columns, then over the wavefronts (in LDS over the dead sums)
#pragma unroll
    for (int off = 32; off >= LPN; off >>= 1)
#pragma unroll
      for (int e = 0; e < VEC; ++e) dot[e] += __shfl_xor(dot[e], off);
    __syncthreads();
    double* red = reinterpret_cast<double*>(smem_raw);   // [NW][KSL]
    if (lane < LPN)
#pragma unroll
      for (int e = 0; e < VEC; ++e) red[wv * KSL + cv + e] = dot[e];
    __syncthreads();
    if (threadIdx.x < KSL) {
      double sum = 0.0;
#pragma unroll
      for (int w = 0; w < NW; ++w) sum += red[w * KSL + threadIdx.x];
      io.part[size_t(t) * k + size_t(sl) * KSL + threadIdx.x] = sum;
    }
  }
}

// out[j] = sum over tiles of part[t][j] (the CG mode's tile partials), one workgroup per
// column, in a fixed order
static __global__ void __launch_bounds__(256)
sum_tiles_multi_kernel(int ntiles, int k, const double* __restrict__ part, double* __restrict__ out) {
  const int j = blockIdx.x;
  double v = 0.0;
  for (int t = threadIdx.x; t < ntiles; t += 256) v += part[size_t(t) * k + j];
  v = wave_sum(v);
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) out[j] = (red[0] + red[1]) + (red[2] + red[3]);
}

// Matrix-core variant (FP32): lane = 4 * block + q, block = 4 * es + 2 * ib + jb: element
// es of the round, row block ib (nodes 4ib..4ib+3), column block jb (right-hand sides
// 4jb..4jb+3).  v_mfma_f32_4x4x1_16b_f32 operands: A = K[4ib + q][kk], B = X[kk][4jb + q];
// result lane 4 * block + q, register r = Y[4ib + r][4jb + q].  The full child-0 stencils
// sit in LDS after the owned sums (FP64): [18][1 + MASS][64].
template <bool MASS>
__host__ __device__ constexpr size_t multi_stencil_len() {
  return size_t(NSTENCIL) * (MASS ? 2 : 1) * 64;
}

template <bool MASS, int MODE, int MB>
__global__ void __launch_bounds__(MB)
tile_multi_mfma_kernel(const TileRec* __restrict__ tiles, int ntiles, int nslices,
                       const uint16_t* __restrict__ lid,
                       const float* __restrict__ kappa, const float* __restrict__ mass, double lap_fac,
                       double mass_fac, uint32_t maxD, double hFac, const float* __restrict__ K0,
                       const uint32_t* __restrict__ node_tab, uint32_t ys_len, MultiIO<float> io) {
  static_assert(MODE != OP_DIAG, "the diagonal does not depend on the right-hand side");
  constexpr int NM = MASS ? 2 : 1;
  constexpr int NV = KS / 4;                  // float4 vectors per node slice
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double* ys = reinterpret_cast<double*>(smem_raw);
  float* sK = reinterpret_cast<float*>(ys + size_t(ys_len) * KS);
  float* xs = sK + multi_stencil_len<MASS>();
  const int np = ntiles * nslices;
  const int pidx = xcd_tile(blockIdx.x, np);
  if (pidx >= np) return;
  const int t = pidx / nslices, sl = pidx % nslices;
  const TileRec rec = tiles[t];
  const uint32_t* nodes = node_tab + rec.node_off;
  const uint32_t n_own = rec.n_own;
  const size_t kv = size_t(io.k / 4);
  for (int i = threadIdx.x; i < int(multi_stencil_len<MASS>()); i += MB) {
    const int tp = i / (NM * 64), mm = (i / 64) % NM, kj = i % 64;
    sK[i] = K0[tp * KSTRIDE + mm * 36 + tri(kj >> 3, kj & 7)];
  }
  {
    const float4* X = reinterpret_cast<const float4*>(io.x);
    float4* xsv = reinterpret_cast<float4*>(xs);
    constexpr int MGU = 4;   // gathers per thread in flight together
    const uint32_t nx = rec.n_touch * NV;
    for (uint32_t i0 = threadIdx.x; i0 < nx; i0 += MGU * MB) {
      uint32_t nid[MGU];
      float4 v[MGU];
#pragma unroll
      for (int u = 0; u < MGU; ++u) {
        const uint32_t i = i0 + u * MB;
        nid[u] = i < nx ? nodes[i / NV] : 0u;
      }
#pragma unroll
      for (int u = 0; u < MGU; ++u) {
        const uint32_t i = i0 + u * MB;
        if (i < nx) v[u] = X[size_t(nid[u]) * kv + size_t(sl) * NV + i % NV];
      }
#pragma unroll
      for (int u = 0; u < MGU; ++u) {
        const uint32_t i = i0 + u * MB;
        if (i < nx) xsv[i] = v[u];
      }
    }
  }
  for (uint32_t i = threadIdx.x; i < n_own * KS; i += MB) ys[i] = 0.0;
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  constexpr int NW = MB / 64;
  const int blk = lane >> 2, q = lane & 3;
  const int es = blk >> 2, ib = (blk >> 1) & 1, jb = blk & 1;
  for (uint32_t r0 = uint32_t(wv) * 4; r0 < rec.n_elem; r0 += NW * 4) {
    const uint32_t r = r0 + es;
    const bool act = r < rec.n_elem;
    uint32_t L[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    float a[8], bv[8];
    if (act) {
      Rec R;
      load_rec<float, MASS>(R, rec.elem_off + r, lid, kappa, mass, lap_fac, mass_fac, maxD, hFac);
      const float f1 = float(R.k1), f2 = float(R.k2);
      const float* Lrow = sK + (R.mt & 31u) * (NM * 64) + (4 * ib + q) * 8;
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        L[kk] = R.l[kk];
        a[kk] = MASS ? f1 * Lrow[kk] + f2 * Lrow[64 + kk] : f1 * Lrow[kk];
        bv[kk] = xs[R.l[kk] * KS + 4 * jb + q];
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) a[kk] = bv[kk] = 0.f;
    }
    mfma_f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a[kk], bv[kk], acc, 0, 0, 0);
    if (act) {
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const uint32_t nd = L[4 * ib + rr];
        if (nd < n_own) atomic_add(&ys[nd * KS + 4 * jb + q], double(acc[rr]));
      }
    }
  }
  __syncthreads();
  const size_t k = size_t(io.k);
  for (uint32_t i = threadIdx.x; i < n_own * KS; i += MB) {
    const uint32_t nd = i / KS, c = i % KS;
    const size_t gi = size_t(nodes[nd]) * k + size_t(sl) * KS + c;
    const float v = float(ys[i]);
    if (MODE == OP_MATVEC) {
      io.y[gi] = v;
    } else if (MODE == OP_RESID) {
      io.y[gi] = io.b[gi] - v;
    } else {
      const float rr = io.b[gi] - v;
      io.y[gi] = xs[i] + io.omega * (rr * io.invd[nodes[nd]]);
    }
  }
}

// x[n][j] = omega (b[n][j] invd[n])  (first sweep from a zero guess)
template <class T>
__global__ void smooth_first_multi_kernel(uint32_t n, int k, T omega, const T* __restrict__ b,
                                          const T* __restrict__ invd, T* __restrict__ x) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= size_t(n) * k) return;
  x[i] = T(0) + omega * (b[i] * invd[i / k]);
}

// c[i][j] = sum_p w_p f[col_p][j], and with x1 given the coarse level's first sweep from zero, x1 =
// omega (c invd): RM_LANES x k / VEC threads per row, each summing every RM_LANES-th entry of VEC
// columns (16-byte loads, RU entries in flight), combined in a fixed order.  One thread per column
// walking the row four entries at a time was a chain of up to 13 loads.  16 columns: 84k fine nodes 12.4
// -> 6.5 us, 26k 9.5 -> 4.9, 8.9k 8.9 -> 4.7, and the sweep's own launch (5 us) saved.
constexpr int RM_LANES = 4;
template <class T>
static __global__ void __launch_bounds__(256)
restrict_multi_kernel(uint32_t nc, int k, const uint32_t* __restrict__ rowptr, const uint32_t* __restrict__ col,
                      const float* __restrict__ w, const T* __restrict__ f, T* __restrict__ c, T omega,
                      const T* __restrict__ invd, T* __restrict__ x1) {
  using V = vec16_t<T>;
  constexpr int VEC = 16 / int(sizeof(T));
  // lane l of a row's RM_LANES are adjacent threads, so they combine by shuffles
  const uint32_t gid = blockIdx.x * 256 + threadIdx.x;
  const uint32_t l = gid % RM_LANES, item = gid / RM_LANES, kv = uint32_t(k / VEC);
  const uint32_t i = item / kv, j = (item % kv) * VEC;
  const bool in = i < nc;
  V acc = {};
  if (in) {
    const uint32_t p1 = rowptr[i + 1];
    constexpr int RU = 8;
    for (uint32_t p0 = rowptr[i] + l; p0 < p1; p0 += RU * RM_LANES) {
      uint32_t cc[RU];
      T wv[RU];
      V fv[RU];
#pragma unroll
      for (int u = 0; u < RU; ++u) {
        const uint32_t p = p0 + u * RM_LANES;
        cc[u] = p < p1 ? col[p] : 0u;
        wv[u] = p < p1 ? T(w[p]) : T(0);
      }
#pragma unroll
      for (int u = 0; u < RU; ++u)
        fv[u] = p0 + u * RM_LANES < p1 ? *reinterpret_cast<const V*>(f + size_t(cc[u]) * k + j) : V{};
#pragma unroll
      for (int u = 0; u < RU; ++u) acc += wv[u] * fv[u];
    }
  }
#pragma unroll
  for (int off = RM_LANES / 2; off > 0; off >>= 1)
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] += __shfl_down(acc[e], off, RM_LANES);
  if (!in || l != 0) return;
  *reinterpret_cast<V*>(c + size_t(i) * k + j) = acc;
  if (x1) *reinterpret_cast<V*>(x1 + size_t(i) * k + j) = omega * (acc * invd[i]);
}

// f_out[j][q] = f_in[j][q] + sum_m W[s][pos_j][m] c[cnl[m]][q], VEC columns per thread
template <class T>
static __global__ void __launch_bounds__(256)
prolong_multi_kernel(uint32_t nf, int k, const uint32_t* __restrict__ celem, const uint8_t* __restrict__ pos,
                     const uint32_t* __restrict__ cnl, const uint8_t* __restrict__ cs,
                     const T* __restrict__ W, const T* __restrict__ c, const T* __restrict__ f_in,
                     T* __restrict__ f_out) {
  using V = vec16_t<T>;
  constexpr int VEC = 16 / int(sizeof(T));
  const uint32_t kv = uint32_t(k / VEC);
  const uint32_t gid = blockIdx.x * 256 + threadIdx.x;
  const uint32_t j = gid / kv;
  if (j >= nf) return;
  const size_t q = size_t(gid % kv) * VEC, at = size_t(j) * k + q;
  const uint32_t ce = celem[j];
  const T* wv = W + (size_t(cs[ce]) * 27 + pos[j]) * 8;
  // the coarse values are loaded whatever the weights: they then wait on the vertex ids only
  const uint4 a = reinterpret_cast<const uint4*>(cnl)[2 * size_t(ce)];
  const uint4 b = reinterpret_cast<const uint4*>(cnl)[2 * size_t(ce) + 1];
  const uint32_t idx[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  V cv[8];
#pragma unroll
  for (int m = 0; m < 8; ++m) cv[m] = *reinterpret_cast<const V*>(c + size_t(idx[m]) * k + q);
  V fv = {};
  if (f_in) fv = *reinterpret_cast<const V*>(f_in + at);
  V acc = {};
#pragma unroll
  for (int m = 0; m < 8; ++m) {
    const T wk = wv[m];
    if (wk != T(0)) acc += wk * cv[m];
  }
  *reinterpret_cast<V*>(f_out + at) = fv + acc;
}

// X = Ainv B for the dense coarsest inverse (row pitch ld, FP32) and k right-hand sides ([n][k]) on the
// matrix cores: FP64 products and sums of the FP32 values (v_mfma_f64_16x16x4).  A workgroup forms 16
// rows of X, its DM_WAVES wavefronts sharing the columns of Ainv; their sums meet in LDS in a fixed
// order.  In a step a lane loads 4 adjacent values of a row of Ainv (row lane % 16, columns 4 (lane /
// 16) ...) and the same 4 rows of B, so the four products of a step take any order of the columns.
// Result register r of a lane is row lane / 16 + 4 r, column lane % 16.
// The vector ALUs' form (4 x 4 blocks per thread, 16 partial sums in memory and a kernel to add them)
// took 33 + 5 us for 2634 rows and 16 columns, this one 12 (22 without the next step's loads in flight);
// reading the matrix takes about 5, its conversions and products about 7 on the 165 CUs that have rows.
constexpr int DM_WAVES = 16, DM_UNROLL = 2;
typedef double mfma_d4 __attribute__((ext_vector_type(4)));
template <int NT>   // 16-column groups of B
__global__ void __launch_bounds__(DM_WAVES * 64)
dense_multi_kernel(int n, int ld, int k, const float* __restrict__ Ainv, const float* __restrict__ B,
                   float* __restrict__ X) {
  __shared__ double red[DM_WAVES][16 * 16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int lr = lane & 15, lk = (lane >> 4) * 4;
  const int row0 = blockIdx.x * 16;
  const float* Ar = Ainv + size_t(min(row0 + lr, n - 1)) * ld;
  mfma_d4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = mfma_d4{0.0, 0.0, 0.0, 0.0};
  float4 an[DM_UNROLL];
  float bn[DM_UNROLL][NT][4];
  auto fetch = [&](int m0) {
#pragma unroll
    for (int u = 0; u < DM_UNROLL; ++u) {
      // columns past the end: the row's padding is zero and so are B's values; ld is a multiple of 8
      const int m = m0 + u * DM_WAVES * 16 + lk;
      an[u] = m < n ? *reinterpret_cast<const float4*>(Ar + m) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          bn[u][t][e] = (m + e < n && t * 16 + lr < k) ? B[size_t(m + e) * k + t * 16 + lr] : 0.f;
    }
  };
  fetch(wv * 16);
  for (int m0 = wv * 16; m0 < n; m0 += DM_UNROLL * DM_WAVES * 16) {
    float av[DM_UNROLL][4], bv[DM_UNROLL][NT][4];
#pragma unroll
    for (int u = 0; u < DM_UNROLL; ++u) {
      av[u][0] = an[u].x;
      av[u][1] = an[u].y;
      av[u][2] = an[u].z;
      av[u][3] = an[u].w;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[u][t][e] = bn[u][t][e];
    }
    fetch(m0 + DM_UNROLL * DM_WAVES * 16);   // in flight during the products
#pragma unroll
    for (int u = 0; u < DM_UNROLL; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(double(av[u][e]), double(bv[u][t][e]), acc[t], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (t) __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv][((lane >> 4) + 4 * r) * 16 + lr] = acc[t][r];
    __syncthreads();
    if (threadIdx.x < 256) {
      const int i = row0 + int(threadIdx.x >> 4), j = t * 16 + int(threadIdx.x & 15);
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < DM_WAVES; ++w) s += red[w][threadIdx.x];
      if (i < n && j < k) X[size_t(i) * k + j] = float(s);
    }
  }
}

// ---------------------------------------------------------------- column reductions
// out[q][j] = sum_n a_q[n][j] * b_q[n][j] (b_q == nullptr: sum of a_q), deterministic:
// stage 1 writes part[(q * RED_BLOCKS_M + block) * k + j], stage 2 sums over blocks in order.
constexpr int RED_BLOCKS_M = 1024;
template <class T>
__global__ void __launch_bounds__(256)
reduce1_multi_kernel(uint32_t n, int k, DotArgs<T> d, double* __restrict__ part) {
  const int j = threadIdx.x % k, rs = threadIdx.x / k, nrs = 256 / k;
  double s[MAXQ] = {0.0, 0.0, 0.0, 0.0};
  const uint32_t per = (n + RED_BLOCKS_M - 1) / RED_BLOCKS_M;
  const uint32_t lo = blockIdx.x * per, hi = min(n, lo + per);
  if (rs < nrs) {
    uint32_t i = lo + rs;
    for (; i + uint32_t(nrs) < hi; i += 2 * nrs) {       // two rows in flight per thread
      const size_t g0 = size_t(i) * k + j, g1 = size_t(i + nrs) * k + j;
#pragma unroll
      for (int q = 0; q < MAXQ; ++q)
        if (d.a[q]) {
          const double v0 = double(d.a[q][g0]) * (d.b[q] ? double(d.b[q][g0]) : 1.0);
          const double v1 = double(d.a[q][g1]) * (d.b[q] ? double(d.b[q][g1]) : 1.0);
          s[q] += v0;
          s[q] += v1;
        }
    }
    for (; i < hi; i += nrs) {
      const size_t g = size_t(i) * k + j;
#pragma unroll
      for (int q = 0; q < MAXQ; ++q)
        if (d.a[q]) s[q] += double(d.a[q][g]) * (d.b[q] ? double(d.b[q][g]) : 1.0);
    }
  }
  __shared__ double red[MAXQ][256];
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) red[q][threadIdx.x] = s[q];
  __syncthreads();
  if (threadIdx.x < k) {
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      double t = 0.0;
      for (int r = 0; r < nrs; ++r) t += red[q][r * k + threadIdx.x];
      part[(size_t(q) * RED_BLOCKS_M + blockIdx.x) * k + threadIdx.x] = t;
    }
  }
}

// out[q * ostride + j]: one workgroup per (q, j), partials summed in a fixed tree order
static __global__ void __launch_bounds__(256)
reduce2_multi_kernel(int nq, int k, const double* __restrict__ part, double* __restrict__ out, int ostride) {
  const int q = blockIdx.x / k, j = blockIdx.x % k;
  if (q >= nq) return;
  double t = 0.0;
  for (int b = threadIdx.x; b < RED_BLOCKS_M; b += 256) t += part[(size_t(q) * RED_BLOCKS_M + b) * k + j];
  t = wave_sum(t);
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) out[q * ostride + j] = (red[0] + red[1]) + (red[2] + red[3]);
}

// v[n][j] -= sum[j] / n
template <class T>
__global__ void subtract_mean_multi_kernel(uint32_t n, int k, const double* __restrict__ sum, T* __restrict__ v) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < size_t(n) * k) v[i] = v[i] - T(sum[i % k] / double(n));
}

// ---------------------------------------------------------------- batched CG
// Scalars per right-hand side j: SM[q * MAXK + j] with q a CgScalar, plus SM_DP0 (initial
// norm) and SM_ACT (1 while the column iterates).  A converged column is frozen: its
// step length is zero, so its iterate stays the one that met the test (also in an iteration that the
// host queued before it knew).
enum { SM_DP0 = S_NSCAL, SM_ACT, SM_NSCAL };

static __global__ void cg_p_multi_kernel(uint32_t n, int k, const double* __restrict__ S, const double* __restrict__ z,
                                  double* __restrict__ p) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int j = int(i % k);
  if (i < size_t(n) * k && S[SM_ACT * MAXK + j] != 0.0) p[i] = z[i] + S[S_RATIO * MAXK + j] * p[i];
}

// x += alpha_j p, r -= alpha_j w for the active columns (alpha_j = RZ / PW, stored as ALPHA),
// fused with the start of the batched V-cycle on the finest level: the FP32 right-hand side
// b32 = float(r) and the first sweep from zero x1 = omega (b32 invd), with the arithmetic of
// the conversion and first-sweep kernels.
static __global__ void cg_xr_multi_fused_kernel(uint32_t n, int k, double* __restrict__ S,
                                                const double* __restrict__ p, const double* __restrict__ w,
                                                double* __restrict__ x, double* __restrict__ r,
                                                float* __restrict__ b32, const float* __restrict__ invd,
                                                float omega, float* __restrict__ x1) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int j = int(i % k);
  const bool act = S[SM_ACT * MAXK + j] != 0.0;
  const double a = act ? S[S_RZ * MAXK + j] / S[S_PW * MAXK + j] : 0.0;
  if (i < size_t(k)) S[S_ALPHA * MAXK + j] = a;
  if (i >= size_t(n) * k) return;
  double ri = r[i];
  if (act) {
    x[i] = x[i] + a * p[i];
    ri = ri + (-a) * w[i];
    r[i] = ri;
  }
  const float bf = float(ri);
  b32[i] = bf;
  x1[i] = 0.f + omega * (bf * invd[i / k]);
}

// z = double(v) - mean_j (the column means of v, summed in FP64, in sum[j] * n): the
// conversion of the V-cycle's result and the constant-null-space projection in one pass;
// sum == nullptr: the conversion alone.
static __global__ void convert_sub_mean_multi_kernel(uint32_t n, int k, const float* __restrict__ v,
                                                     const double* __restrict__ sum, double* __restrict__ z) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= size_t(n) * k) return;
  const double zi = double(v[i]);
  z[i] = sum ? zi - double(sum[i % k] / double(n)) : zi;
}

// Tells the host about the columns after iteration its (one wavefront, lane j: column j; see CgSignal).
struct CgSignalMulti {
  double dp[4][MAXK];
  unsigned int act[4];   // bit j: column j still iterates
  unsigned long long seq;
};
__device__ __forceinline__ void cg_tell(int k, int its, double dp, bool act, CgSignalMulti* sig) {
  const int j = threadIdx.x, slot = its & 3;
  const unsigned int mask = static_cast<unsigned int>(__ballot(act));
  if (j < k) __hip_atomic_store(&sig->dp[slot][j], dp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __threadfence_system();
  if (j == 0) {
    __hip_atomic_store(&sig->act[slot], mask, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&sig->seq, static_cast<unsigned long long>(its) + 1ull, __ATOMIC_RELEASE,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

static __global__ void __launch_bounds__(64)
cg_scalar_multi_kernel(int k, double* __restrict__ S, int precond_norm, int flexible, double rtol, CgSignalMulti* sig) {
  const int j = threadIdx.x;
  const int its = int(S[S_ITS * MAXK]) + 1;
  bool act = j < k && S[SM_ACT * MAXK + j] != 0.0;
  double dp = 0.0;
  if (act) {
    dp = sqrt(precond_norm ? S[S_ZZ * MAXK + j] : S[S_RR * MAXK + j]);
    const double ratio = flexible ? (-S[S_ALPHA * MAXK + j] * S[S_ZW * MAXK + j]) / S[S_RZ * MAXK + j]
                                  : S[S_ZR * MAXK + j] / S[S_RZ * MAXK + j];
    S[S_DP * MAXK + j] = dp;
    S[S_RATIO * MAXK + j] = ratio;
    S[S_RZ * MAXK + j] = S[S_ZR * MAXK + j];
    act = dp > rtol * S[SM_DP0 * MAXK + j];
    if (!act) S[SM_ACT * MAXK + j] = 0.0;
  }
  cg_tell(k, its, dp, act, sig);
  if (j == 0) S[S_ITS * MAXK] = double(its);
}

static __global__ void __launch_bounds__(64)
cg_init_multi_kernel(int k, double* __restrict__ S, int precond_norm, CgSignalMulti* sig) {
  const int j = threadIdx.x;
  double dp = 0.0;
  if (j < k) {
    S[S_RZ * MAXK + j] = S[S_ZR * MAXK + j];
    dp = sqrt(precond_norm ? S[S_ZZ * MAXK + j] : S[S_BB * MAXK + j]);
    S[S_DP * MAXK + j] = dp;
    S[SM_DP0 * MAXK + j] = dp;
    S[S_RATIO * MAXK + j] = 0.0;
    S[SM_ACT * MAXK + j] = dp > 0.0 ? 1.0 : 0.0;
  }
  cg_tell(k, 0, dp, dp > 0.0, sig);
  if (j == 0) S[S_ITS * MAXK] = 0.0;
}

}  // namespace dgh
