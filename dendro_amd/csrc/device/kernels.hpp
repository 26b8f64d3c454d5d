// CDNA4 (gfx950) operator and transfer kernels of libdendrohip.
//
// The operator kernel is owner-computes over tiles of Morton-ordered elements (the host
// plan of tiles.cpp): one workgroup per tile stages the tile's x values in LDS, evaluates
// every record (own and halo elements) with the factored element product (or, on request, with
// the 18 child-0 stencils' rows), accumulates the rows of the nodes the tile owns with 64-bit fixed-point LDS
// atomics, and stores each owned node exactly once.  There are no global atomics, y needs no
// zeroing, and the integer sums make the result independent of the order of the additions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "host/octree.hpp"

namespace dgh {

constexpr int NXCD = 8;          // XCDs of an MI355X; workgroups are dealt round-robin
constexpr int NSTENCIL = 18;     // child-0 stencil types
constexpr int NCLASS = 1024;     // record classes: child-0 type | level << 5 (levels <= 31)

// Maps the hardware workgroup id to a tile so that each XCD works on one contiguous
// range of tiles: neighbouring tiles share halo nodes, whose x values then meet in one L2.
__device__ __forceinline__ int xcd_tile(int bid, int ntiles) {
  const int per = (ntiles + NXCD - 1) / NXCD;
  return (bid % NXCD) * per + bid / NXCD;
}

template <class T>
__device__ __forceinline__ void atomic_add(T* p, T v) {
  unsafeAtomicAdd(p, v);
}

// Element factors exactly as the reference forms them (odaJac.C:271-276,
// omgJac.C:1665-1672): h = hFac 2^(maxD - lev), fac1 = kappa h / 2, fac2 = mass h^3 / 8.
// Per-element coefficients arrive with the factors already formed per record by the host
// (h is a power of two, so the products are exact either way); uniform ones are scaled here.
__device__ __forceinline__ void elem_factors(uint32_t lev, uint32_t maxD, double hFac, double k1,
                                             double k2, double& fac1, double& fac2) {
  const double h = hFac * double(1u << (maxD - lev));
  fac1 = k1 * h / 2.0;
  fac2 = k2 * h * h * h / 8.0;
}

// MATVEC: y = A x;  DIAG: y = diag(A);  RESID: y = b - A x;
// SMOOTH: y = x + omega (invd (b - A x))  (one Richardson + Jacobi sweep, y must not alias x);
// CG: y = A x and the tile's partial sum of x.y (the CG product p.Ap).
// OP_DIRMV: the Dirichlet-masked MatVec (examples/src/backend/omgJac.C:859-1056): x of
// boundary nodes is staged as 0 (their columns drop out) and their rows return x itself.
// OP_SMOOTH0: OP_SMOOTH of x = omega (b * invd), the first sweep from a zero guess, formed as it is
// gathered (x unused).
enum OpMode { OP_MATVEC = 0, OP_DIAG = 1, OP_RESID = 2, OP_SMOOTH = 3, OP_CG = 4, OP_DIRMV = 5, OP_SMOOTH0 = 6 };

template <class T>
struct OpIO {
  T* y;            // output
  const T* b;      // right-hand side (RESID, SMOOTH)
  const T* invd;   // inverse diagonal (SMOOTH)
  T omega;         // Richardson scale (SMOOTH)
  double* part;    // CG: per-tile partial sums of x.y
  const uint8_t* bdy;   // DIRMV, and DIAG if set: boundary flags per node (nonzero = boundary)
};

// Symmetric 8x8 stencils are kept as their upper triangles (36 entries, row-major):
// entry (k, j) with k <= j sits at tri(k, j) = k*8 - k*(k-1)/2 + (j - k).
__host__ __device__ constexpr int tri(int k, int j) {
  return (k <= j) ? (k * 8 - k * (k - 1) / 2 + (j - k)) : (j * 8 - j * (j - 1) / 2 + (k - j));
}
constexpr int KSTRIDE = 72;   // per stencil type: Laplacian triangle then mass triangle

// One record: tile-local ids of its 8 vertices, child-0 type | level << 5, and its element
// factors (k1 = kappa h / 2, k2 = mass h^3 / 8).
struct Rec {
  uint32_t l[8];
  uint32_t mt;
  double k1, k2;
};

// A record on the device is 16 bytes: the 8 tile-local vertex ids in 14 bits each, the
// record's class (child-0 type | level << 5, 10 bits) in the top 2 bits of ids 0..4 and its
// hanging vertices (rec_hang) in the top 2 bits of ids 5..7 (pack_records).
constexpr uint32_t REC_ID_MASK = 0x3fffu;
constexpr uint32_t REC_MAX_TOUCH = REC_ID_MASK + 1u;
__device__ __forceinline__ uint32_t rec_class(uint4 lp) {
  return ((lp.x >> 14) & 3u) | ((lp.x >> 30) << 2) | (((lp.y >> 14) & 3u) << 4) | ((lp.y >> 30) << 6) |
         (((lp.z >> 14) & 3u) << 8);
}

// Hanging vertices of a record in child 0's order, one bit each: vertices 1, 2, 4 (edge
// midpoints) in bits 0..2, 3, 5, 6 (face centres) in bits 3..5.
__host__ __device__ constexpr uint32_t hang_bits(uint32_t mask) {
  return ((mask >> 1) & 3u) | (((mask >> 4) & 1u) << 2) | (((mask >> 3) & 1u) << 3) | (((mask >> 5) & 3u) << 4);
}
__device__ __forceinline__ uint32_t rec_hang(uint4 lp) {
  return (lp.z >> 30) | ((lp.w >> 12) & 12u) | ((lp.w >> 26) & 48u);
}

// kappa/mass: per-record factors formed by the host, or nullptr for uniform coefficients
// (lap_fac, mass_fac scaled by the element size here).  LSC scales the vertex ids (the
// single right-hand-side kernel takes them as LDS byte offsets).  UNI: 1 uniform, 0 per
// record, -1 decided by kappa at run time.
// FAC false: the factors are not formed (class matrices carry them).
template <class TC, bool MASS, uint32_t LSC = 1, int UNI = -1, bool FAC = true>
__device__ __forceinline__ void load_rec(Rec& R, uint32_t g, const uint16_t* __restrict__ lid,
                                         const TC* __restrict__ kappa, const TC* __restrict__ mass,
                                         double lap_fac, double mass_fac, uint32_t maxD, double hFac) {
  const uint4 lp = reinterpret_cast<const uint4*>(lid)[g];
  R.l[0] = (lp.x & REC_ID_MASK) * LSC; R.l[1] = ((lp.x >> 16) & REC_ID_MASK) * LSC;
  R.l[2] = (lp.y & REC_ID_MASK) * LSC; R.l[3] = ((lp.y >> 16) & REC_ID_MASK) * LSC;
  R.l[4] = (lp.z & REC_ID_MASK) * LSC; R.l[5] = ((lp.z >> 16) & REC_ID_MASK) * LSC;
  R.l[6] = (lp.w & REC_ID_MASK) * LSC; R.l[7] = ((lp.w >> 16) & REC_ID_MASK) * LSC;
  R.mt = rec_class(lp);
  if (UNI < 0 ? kappa != nullptr : UNI == 0) {
    R.k1 = double(kappa[g]);
    R.k2 = MASS ? double(mass[g]) : 0.0;
  } else if (FAC) {
    elem_factors(R.mt >> 5, maxD, hFac, lap_fac, mass_fac, R.k1, R.k2);
  }
}

// Full stencil rows for the single right-hand-side kernel: per child-0 type, the Laplacian
// rows [8][8] then the mass rows [8][8].
constexpr int KFSTRIDE = 128;

// Owned-node rows accumulate in fixed point: 64-bit integers for FP64 operators, 32-bit for
// FP32.  FP64: a contribution c enters as the integer round(c 2^es), formed by one FMA with
// 1.5 2^52: for |c 2^es| < 2^51 the bit pattern of fma(c, 2^es, 1.5 2^52) is that of
// 1.5 2^52 plus round(c 2^es), so subtracting the former leaves the integer in two's
// complement; es keeps every term below 2^FX_BITS (the host's bounds leave a margin of 2^-20 for
// the rounding of the term itself).  FP32: round-to-nearest conversion of
// c 2^es (float), es keeping every term below 2^(FX32_BITS - v) where 2^v bounds the number of
// terms a node of the tile receives, so the 32-bit sums cannot overflow.  es is chosen per
// tile: the host bounds the element factors times the stencil row sums (texp[t].x: bound
// < 2^texp) and the terms per node (texp[t].y = v), the kernel bounds max |x| over the tile's
// staged values.  Each FP64 term is rounded to 2^-FX_BITS of the tile's bound (output ~1e-14
// relative), each FP32 term to about 2^-24 of it.  Integer LDS additions run faster than
// floating-point ones on scattered addresses (ds_add_u64 about twice ds_add_f64, ds_add_u32
// faster again) and do not depend on the order of the additions, so the operator is
// bit-reproducible.
constexpr int FX_BITS = 51;
constexpr int FX32_BITS = 30;
constexpr double FX_MARGIN = 1.0 + 0x1p-20;
constexpr double FX_MAGIC = 6755399441055744.0;   // 1.5 * 2^52
constexpr unsigned long long FX_MAGIC_BITS = 0x4338000000000000ull;
constexpr int FX_XMIN = -900;                      // |x| below 2^-900 counts as 2^-900,
constexpr int FX32_XMIN = -96;                     // FP32: below 2^-96 (the scaled factors stay finite)
// max |x| < 2^ex of a tile (or column) from the high word of its max |x| in FP64
template <class T>
__device__ __forceinline__ int fx_ex(uint32_t hi) {
  return max(int(hi >> 20) - 1022, sizeof(T) == 8 ? FX_XMIN : FX32_XMIN);
}

template <class T>
using fx_acc_t = typename std::conditional<sizeof(T) == 8, unsigned long long, unsigned int>::type;

// The factored products add up to eight staged values before they scale them: values of at least
// 2^fx_top are first multiplied by 2^-FX_UP (exact but for bits far below the fixed-point grid of
// such values) and the scale of the terms by 2^FX_UP, so that no intermediate overflows where the
// product itself does not.  ex is the same in a workgroup's threads; the branch not taken costs 0.08 us
// of 9.0 (FP64, 318k elements), 0.8 of 163 in the batched product of 631k, nothing measurable elsewhere.
constexpr int FX_UP = 4;
template <class T>
__host__ __device__ constexpr int fx_top() { return sizeof(T) == 8 ? 1020 : 124; }
template <class T>
__device__ __forceinline__ bool fx_big(int ex) {
  return __builtin_amdgcn_readfirstlane(ex) > fx_top<T>();
}

// Scale exponent of a tile: every contribution times 2^es stays below the fixed-point bound.
template <class T>
__device__ __forceinline__ int fx_scale(int2 te, int ex) {
  return sizeof(T) == 8 ? FX_BITS - te.x - ex : FX32_BITS - te.y - te.x - ex;
}

// fixed-point term of a + b (a = row sum times the scaled Laplacian factor, b likewise mass)
__device__ __forceinline__ unsigned long long fx_term(double a, double f1s, double b, double f2s, bool mass) {
  const double v = mass ? __builtin_fma(a, f1s, __builtin_fma(b, f2s, FX_MAGIC)) : __builtin_fma(a, f1s, FX_MAGIC);
  return static_cast<unsigned long long>(__double_as_longlong(v)) - FX_MAGIC_BITS;
}
__device__ __forceinline__ unsigned int fx_term(float a, float f1s, float b, float f2s, bool mass) {
  const float v = mass ? __builtin_fmaf(b, f2s, a * f1s) : a * f1s;
  return static_cast<unsigned int>(__float2int_rn(v));
}

template <class T>
__device__ __forceinline__ double fx_value(fx_acc_t<T> s, int es) {
  return sizeof(T) == 8 ? ldexp(double(static_cast<long long>(s)), -es)
                        : ldexp(double(static_cast<int>(static_cast<unsigned int>(s))), -es);
}

// Fixed LDS layout of one operator tile.  tile_op_kernel declares no static LDS, so its
// dynamic LDS starts at address 0 and each region sits at a compile-time byte offset.  The
// sums start at address 0 and the staged x's offset rides in the immediate field of the ds
// instructions: a record corner costs one address computation (its id times the element
// size) for both its x read and its sum.
//   [0, tile_xhi_off)             fixed-point sums of the owned nodes, op_own_cap(BLOCK) entries
//   [tile_xhi_off, + 64)          high word of max |x|, one per wavefront (at most 16)
//   [tile_xs_off, ...)            staged x of the touched nodes, owned first
// The host plan keeps n_own <= op_own_cap(BLOCK) and op_own_cap(BLOCK) + n_touch within the
// block size's node budget.
__host__ __device__ constexpr uint32_t op_own_cap(int block) {
  return block >= 1024 ? 4096u : block >= 512 ? 2048u : 1024u;
}
template <class T, int BLOCK>
__host__ __device__ constexpr uint32_t tile_xhi_off() {
  return uint32_t(sizeof(fx_acc_t<T>)) * op_own_cap(BLOCK);
}
template <class T, int BLOCK>
__host__ __device__ constexpr uint32_t tile_xs_off() {
  return tile_xhi_off<T, BLOCK>() + 64u;
}
// Lane stencils (small levels): a copy of the stencil table follows the staged x of the
// tile, 16-byte aligned.
constexpr uint32_t KF_ELEMS = NSTENCIL * KFSTRIDE;
template <class T>
__host__ __device__ constexpr uint32_t tile_kf_off(uint32_t xs_off, uint32_t n_touch) {
  return (xs_off + uint32_t(sizeof(T)) * n_touch + 15u) & ~15u;
}
template <class T>
__host__ constexpr size_t tile_lds_bytes(int block, uint32_t max_touch, bool lane_rows = false) {
  const uint32_t xs = uint32_t(sizeof(fx_acc_t<T>)) * op_own_cap(block) + 64u;
  return lane_rows ? size_t(tile_kf_off<T>(xs, max_touch)) + sizeof(T) * KF_ELEMS
                   : size_t(xs) + sizeof(T) * size_t(max_touch);
}
template <class U>
using lds_ptr = __attribute__((address_space(3))) U*;
template <class U>
__device__ __forceinline__ lds_ptr<U> lds_at(uint32_t byte) {
  return (lds_ptr<U>)byte;
}
template <class U>
__device__ __forceinline__ void lds_add(lds_ptr<U> p, U v) {
  __atomic_fetch_add(p, v, __ATOMIC_RELAXED);
}

// Evaluates the rows of the owned vertices of one record and adds them, scaled by 2^es, to
// the fixed-point sums.  Stencil rows are read through the scalar cache, one row at a time
// (16 or 32 SGPRs live): the wavefront walks over the distinct stencil types among its
// lanes (one in class-pure wavefronts, two at the class boundaries of a tile) with a
// wave-uniform row pointer.  The compiler computes a row only when some lane owns it.
// R.l holds LDS byte offsets (ids times sizeof(T)); own_bytes = n_own sizeof(T).
// COMB (uniform coefficients): KF holds the element matrix fac1 L + fac2 M of each record
// class (type | level << 5, [NCLASS][64]); the walk is over classes and a row costs 8
// products instead of 16 plus the two factor products.
template <class T, bool MASS, int MODE, uint32_t XS, bool COMB = false>
__device__ __forceinline__ void eval_rows(const Rec& R, uint32_t own_bytes, int es, const T* __restrict__ KF) {
  if (COMB) {
    const T sc = T(ldexp(1.0, es));
    T xv[8];
    if (MODE != OP_DIAG) {
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[j] = *lds_at<T>(XS + R.l[j]);
    }
    const uint32_t cl = R.mt;
    bool done = false;
    for (;;) {
      const uint64_t pend = __ballot(!done);
      if (pend == 0) break;
      const uint32_t cu = __builtin_amdgcn_readlane(cl, __builtin_ctzll(pend));
      const bool mine = !done && cl == cu;
      const T* Kt = KF + cu * 64u;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        T kr[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) kr[j] = Kt[k * 8 + j];
        if (mine && R.l[k] < own_bytes) {
          T a;
          if (MODE == OP_DIAG) {
            a = kr[k];
          } else {
            a = kr[0] * xv[0];
#pragma unroll
            for (int j = 1; j < 8; ++j) a += kr[j] * xv[j];
          }
          lds_add(lds_at<fx_acc_t<T>>(R.l[k]), fx_term(a, sc, T(0), T(0), false));
        }
      }
      done = done || mine;
    }
    return;
  }
  const T fac1 = T(R.k1), fac2 = T(R.k2);
  const T f1s = T(ldexp(double(fac1), es));
  const T f2s = MASS ? T(ldexp(double(fac2), es)) : T(0);
  T xv[8];
  if (MODE != OP_DIAG) {
#pragma unroll
    for (int j = 0; j < 8; ++j) xv[j] = *lds_at<T>(XS + R.l[j]);
  }
  const uint32_t tp = R.mt & 31u;
  bool done = false;
  for (;;) {
    const uint64_t pend = __ballot(!done);
    if (pend == 0) break;
    const uint32_t tu = __builtin_amdgcn_readlane(tp, __builtin_ctzll(pend));
    const bool mine = !done && tp == tu;
    const T* Kt = KF + tu * KFSTRIDE;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      T lr[8], mr[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        lr[j] = Kt[k * 8 + j];
        if (MASS) mr[j] = Kt[64 + k * 8 + j];
      }
      if (mine && R.l[k] < own_bytes) {
        T a, b = T(0);
        if (MODE == OP_DIAG) {
          a = lr[k];
          if (MASS) b = mr[k];
        } else {
          a = lr[0] * xv[0];
#pragma unroll
          for (int j = 1; j < 8; ++j) a += lr[j] * xv[j];
          if (MASS) {
            b = mr[0] * xv[0];
#pragma unroll
            for (int j = 1; j < 8; ++j) b += mr[j] * xv[j];
          }
        }
        lds_add(lds_at<fx_acc_t<T>>(R.l[k]), fx_term(a, f1s, b, f2s, MASS));
      }
    }
    done = done || mine;
  }
}

// Lane-stencil variant for small levels: each lane reads its own type's rows from the LDS
// copy of the stencil table at kf (byte offset; the row offsets ride in the ds immediate
// field), so a wavefront whose lanes hold several stencil types makes one pass instead of
// one per type (small tiles mix many types in a wavefront; each pass is a chain of eight
// scalar row loads).
template <class T, bool MASS, int MODE, uint32_t XS>
__device__ __forceinline__ void eval_rows_lane(const Rec& R, uint32_t own_bytes, int es, uint32_t kf) {
  const T fac1 = T(R.k1), fac2 = T(R.k2);
  const T f1s = T(ldexp(double(fac1), es));
  const T f2s = MASS ? T(ldexp(double(fac2), es)) : T(0);
  T xv[8];
  if (MODE != OP_DIAG) {
#pragma unroll
    for (int j = 0; j < 8; ++j) xv[j] = *lds_at<T>(XS + R.l[j]);
  }
  const uint32_t rb = kf + (R.mt & 31u) * uint32_t(KFSTRIDE * sizeof(T));
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (R.l[k] < own_bytes) {
      const lds_ptr<T> lr = lds_at<T>(rb + uint32_t(k * 8 * sizeof(T)));
      const lds_ptr<T> mr = lds_at<T>(rb + uint32_t((64 + k * 8) * sizeof(T)));
      T a, b = T(0);
      if (MODE == OP_DIAG) {
        a = lr[k];
        if (MASS) b = mr[k];
      } else {
        a = lr[0] * xv[0];
#pragma unroll
        for (int j = 1; j < 8; ++j) a += lr[j] * xv[j];
        if (MASS) {
          b = mr[0] * xv[0];
#pragma unroll
          for (int j = 1; j < 8; ++j) b += mr[j] * xv[j];
        }
      }
      lds_add(lds_at<fx_acc_t<T>>(R.l[k]), fx_term(a, f1s, b, f2s, MASS));
    }
  }
}

// ---------------------------------------------------------------- factored element product
// The element matrix without stencil rows.  The regular element's matrix is a sum of Kronecker
// products of the 1D matrices [1 -1; -1 1] and [2 1; 1 2]/6, which share the eigenvectors
// (1, 1) and (1, -1): with W the 8x8 Walsh-Hadamard transform, K_0 = W D W / 8, and D depends
// only on the number p of difference axes of a mode.  A hanging element's matrix is
// P_H^T K_0 P_H, P_H the interpolation of its hanging vertices (edge midpoints (x_0 + x_k)/2,
// face centres (x_0 + x_a + x_b + x_k)/4; the 18 child-0 stencils equal these products to
// rounding).  One product costs 24 + 24 additions and 8 multiplications, with or without a
// mass term, plus at most 36 operations for hanging vertices, in one pass of the wavefront
// whatever types its lanes hold, and reads nothing but its record and its x.  Stencil rows cost
// 64 (128 with mass) FMAs per pass over a type or class, and each row's scalar load waits behind
// the LDS additions in flight (they share a counter).  Measured, FP64 / FP32 products, best row
// source before and this form with the next records prefetched, same tilings:
//   9,374 elements        16.4 / 14.7 us ->  9.5 /  8.1 us
//   318,081 elements      19.5 / 17.0    -> 10.2 /  8.9
//   2.1M, kappa only      35.5 / 31.7    -> 26.5 / 21.0
//   10.5M (1787 tiles)   128.6 / 100.4   -> 96.3 / 72.9 us, of which the prefetch 6 to 10%.
// (Launches back to back on the same buffers; with another mesh and vectors each time the last two take
// 26.8 and 98.3 us in FP64.)
// What bounds it now at 10.5M elements: 400 MB per product (records 215, node ids and x 129, y 56)
// at 4.2 TB/s, of the 4.65 a 4 GiB copy reaches; its LDS reads and additions take about as long
// again and overlap only across workgroups.
//   Laplacian on h: kappa h p 2 (1/6)^(p-1) (1/2)^(3-p); mass: m h^3 (1/6)^p (1/2)^(3-p);
// FACT_LAP and FACT_MASS are these over 8 for the factors kappa h/2 and m h^3/8.
__host__ __device__ constexpr double fact_lap(int p) {
  return p == 0 ? 0.0 : p == 1 ? 0.125 : p == 2 ? 1.0 / 12.0 : 1.0 / 24.0;
}
__host__ __device__ constexpr double fact_mass(int p) {
  return p == 0 ? 0.125 : p == 1 ? 1.0 / 24.0 : p == 2 ? 1.0 / 72.0 : 1.0 / 216.0;
}

// d[p]: the mode factors of an element with scaled factors f1 (Laplacian) and f2 (mass)
template <class T, bool MASS>
__device__ __forceinline__ void fact_modes(T f1, T f2, T d[4]) {
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    d[p] = f1 * T(fact_lap(p));
    if (MASS) d[p] = p == 0 ? f2 * T(fact_mass(0)) : d[p] + f2 * T(fact_mass(p));
  }
}

// DGH_NO_SELECT in a branch keeps it one: the compiler otherwise evaluates every vertex and
// selects (75 more vector instructions per 64 records with hanging vertices), where records
// sorted by type leave most wavefronts with few of the six branches taken.
#define DGH_NO_SELECT asm volatile("")
// v[c] <- P_H v[c] for N columns; q = 1/4 (a register: the compiler would otherwise scale by a
// quarter with the slower ldexp)
template <int N, class T>
__device__ __forceinline__ void hang_interp(T (&v)[N][8], uint32_t hb, T q) {
  if (hb == 0u) return;
#define DGH_HANG(bit, expr)                       \
  if (hb & (bit)) {                               \
    DGH_NO_SELECT;                                \
    _Pragma("unroll") for (int c = 0; c < N; ++c) { expr; } \
  }
  DGH_HANG(8u, v[c][3] = q * ((v[c][0] + v[c][1]) + (v[c][2] + v[c][3])))
  DGH_HANG(16u, v[c][5] = q * ((v[c][0] + v[c][1]) + (v[c][4] + v[c][5])))
  DGH_HANG(32u, v[c][6] = q * ((v[c][0] + v[c][2]) + (v[c][4] + v[c][6])))
  DGH_HANG(1u, v[c][1] = T(0.5) * (v[c][0] + v[c][1]))
  DGH_HANG(2u, v[c][2] = T(0.5) * (v[c][0] + v[c][2]))
  DGH_HANG(4u, v[c][4] = T(0.5) * (v[c][0] + v[c][4]))
}
// v[c] <- P_H^T v[c]
template <int N, class T>
__device__ __forceinline__ void hang_interp_t(T (&v)[N][8], uint32_t hb, T q) {
  if (hb == 0u) return;
  DGH_HANG(1u, v[c][0] += T(0.5) * v[c][1]; v[c][1] *= T(0.5))
  DGH_HANG(2u, v[c][0] += T(0.5) * v[c][2]; v[c][2] *= T(0.5))
  DGH_HANG(4u, v[c][0] += T(0.5) * v[c][4]; v[c][4] *= T(0.5))
  DGH_HANG(8u, v[c][0] += q * v[c][3]; v[c][1] += q * v[c][3]; v[c][2] += q * v[c][3]; v[c][3] *= q)
  DGH_HANG(16u, v[c][0] += q * v[c][5]; v[c][1] += q * v[c][5]; v[c][4] += q * v[c][5]; v[c][5] *= q)
  DGH_HANG(32u, v[c][0] += q * v[c][6]; v[c][2] += q * v[c][6]; v[c][4] += q * v[c][6]; v[c][6] *= q)
#undef DGH_HANG
}

// v <- W diag(d[popcount]) W v.  Without a mass term the mean mode's factor is zero.
template <class T, bool MASS>
__device__ __forceinline__ void fact_product(T v[8], const T d[4]) {
#pragma unroll
  for (int b = 1; b < 8; b <<= 1)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (!(i & b)) {
        const T s = v[i] + v[i | b];
        v[i | b] = v[i] - v[i | b];
        v[i] = s;
      }
#pragma unroll
  for (int i = MASS ? 0 : 1; i < 8; ++i) v[i] *= d[(i & 1) + ((i >> 1) & 1) + (i >> 2)];
#pragma unroll
  for (int b = 1; b < 8; b <<= 1)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (!(i & b)) {
        if (!MASS && b == 1 && i == 0) {
          v[0] = v[1];
          v[1] = -v[1];
          continue;
        }
        const T s = v[i] + v[i | b];
        v[i | b] = v[i] - v[i | b];
        v[i] = s;
      }
}

// Fixed-point term of an already scaled value (see FX_BITS).  The low word of the magic
// number's bits is zero, so only the high word is corrected.
__device__ __forceinline__ unsigned long long fx_round(double v) {
  const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(v + FX_MAGIC));
  const uint32_t hi = uint32_t(b >> 32) - uint32_t(FX_MAGIC_BITS >> 32);
  return (static_cast<unsigned long long>(hi) << 32) | uint32_t(b);
}
// the same of v * sc, rounded once
__device__ __forceinline__ unsigned long long fx_round_fma(double v, double sc) {
  const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(__builtin_fma(v, sc, FX_MAGIC)));
  const uint32_t hi = uint32_t(b >> 32) - uint32_t(FX_MAGIC_BITS >> 32);
  return (static_cast<unsigned long long>(hi) << 32) | uint32_t(b);
}
// FP32: halves to even.  Halves up would be one instruction instead of two, but half of the values
// in [2^22, 2^23) are exact halves: the bias made a null-space solve's FP32 V-cycle ten times less
// exact.
__device__ __forceinline__ unsigned int fx_round(float v) {
  return static_cast<unsigned int>(__float2int_rn(v));
}

// One record for the factored product, as loaded (unpacked where it is evaluated, so that it
// holds four registers while the x gather runs), and its element factors (per record).
template <class T>
struct RecF {
  uint4 lp;
  T k1, k2;
};
template <class T, bool MASS, bool UNI>
__device__ __forceinline__ void load_rec_fact(RecF<T>& R, uint32_t g, const uint16_t* __restrict__ lid,
                                              const T* __restrict__ kappa, const T* __restrict__ mass) {
  R.lp = reinterpret_cast<const uint4*>(lid)[g];
  if (!UNI) {
    R.k1 = kappa[g];
    if (MASS) R.k2 = mass[g];
  }
}

// u1 = lap_fac hFac / 2, u2 = mass_fac hFac^3 / 8: the factors of a uniform-coefficient
// element of level lev are u1 2^(maxD - lev) and u2 8^(maxD - lev).  big (uniform): see fx_big; es
// holds FX_UP then.
template <class T, bool MASS, uint32_t XS, bool UNI>
__device__ __forceinline__ void eval_fact(const RecF<T>& R, uint32_t own_bytes, int es, bool big, double u1, double u2,
                                          uint32_t maxD) {
  const uint4 lp = R.lp;
  const uint32_t w[4] = {lp.x, lp.y, lp.z, lp.w};
  uint32_t l[8];   // LDS byte offsets of the vertices
#pragma unroll
  for (int j = 0; j < 8; ++j) l[j] = ((w[j >> 1] >> (16 * (j & 1))) & REC_ID_MASK) * uint32_t(sizeof(T));
  const uint32_t hb = rec_hang(lp);
  T v[1][8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[0][j] = *lds_at<T>(XS + l[j]);
  if (big) {
    DGH_NO_SELECT;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[0][j] *= T(1.0 / (1 << FX_UP));
  }
  T f1, f2 = T(0);
  if (UNI) {
    const int hs = int(maxD - (rec_class(lp) >> 5));
    f1 = T(ldexp(u1, hs + es));
    if (MASS) f2 = T(ldexp(u2, 3 * hs + es));
  } else if constexpr (sizeof(T) == 8) {
    f1 = ldexp(R.k1, es);
    if (MASS) f2 = ldexp(R.k2, es);
  } else {
    f1 = T(ldexp(double(R.k1), es));
    if (MASS) f2 = T(ldexp(double(R.k2), es));
  }
  T d[4];
  fact_modes<T, MASS>(f1, f2, d);
  T q = T(0.25);
  asm("" : "+s"(q));
  hang_interp(v, hb, q);
  fact_product<T, MASS>(v[0], d);
  hang_interp_t(v, hb, q);
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (l[k] < own_bytes) lds_add(lds_at<fx_acc_t<T>>(l[k]), fx_round(v[0][k]));
}

// Touched and owned nodes per thread of a tile, from the plan's bounds (op_own_cap, op_budget):
// at most 5.94 BLOCK touched and 4 BLOCK owned nodes.  One batch of OP_XC gathers therefore
// covers a tile, with every index static: ids and held values stay in registers.
constexpr int OP_XC = 6;
constexpr int OP_OC = 4;

// KF: [18][128] child-0 full stencil rows of precision T (Laplacian, then mass).
// kappa/mass: per record (nullptr: uniform lap_fac / mass_fac).  MASS: mass term present.
// texp[t]: exponent bound of tile t's contributions per unit |x| and log2 bound of the terms
// per node (see FX_BITS).
// node_tab: [ntiles][pitch], each tile's node ids padded with its last one.
// LDS per tile: the fixed layout above (tile_xs_off), fixed-point sums u64 for FP64, u32 for
// FP32; the plan must have been built with op_own_cap(BLOCK).
// UNI: uniform coefficients (kappa and mass unused; lap_fac, mass_fac, maxD and hFac form the
// factors), else per-record factors (lap_fac, mass_fac, maxD and hFac unused).  The two are
// separate instantiations so that neither keeps the other's arguments in scalar registers.
// LANE: per-lane stencil rows from an LDS copy of KF (eval_rows_lane) instead of per-type
// passes through the scalar cache.
// COMB (uniform coefficients, not LANE): KF is the tiling's class matrix table (fac1 L +
// fac2 M per record class, eval_rows' COMB form) and the records' factors are not formed.
// FACT: the factored product (eval_fact) instead of stencil rows; KF and hFac are unused, and
// lap_fac and mass_fac arrive scaled (lap_fac hFac / 2, mass_fac hFac^3 / 8).
template <class T, class TC, bool MASS, int MODE, int BLOCK, bool UNI = false, bool LANE = false, bool COMB = false,
          bool FACT = false>
__global__ void __launch_bounds__(BLOCK)
tile_op_kernel(const TileRec* __restrict__ tiles, const uint32_t* __restrict__ node_tab, const T* __restrict__ x,
               const uint16_t* __restrict__ lid, const int2* __restrict__ texp, int ntiles, uint32_t pitch,
               const TC* __restrict__ kappa, const TC* __restrict__ mass, OpIO<T> io, double lap_fac, double mass_fac,
               uint32_t maxD, double hFac, const T* __restrict__ KF) {
  constexpr int NW = BLOCK / 64;
  static_assert(!COMB || (UNI && !LANE), "class matrices need uniform coefficients and scalar rows");
  static_assert(NW <= 16, "one max |x| word per wavefront in 64 LDS bytes");
  static_assert(sizeof(fx_acc_t<T>) == sizeof(T), "sums and staged x share the byte offsets of a record");
  constexpr uint32_t XS = tile_xs_off<T, BLOCK>();
  static_assert(XS <= 65535u, "staged x must start within the ds immediate offset range");
  const lds_ptr<fx_acc_t<T>> acc = lds_at<fx_acc_t<T>>(0);
  const lds_ptr<T> xs = lds_at<T>(XS);
  const lds_ptr<uint32_t> s_xhi = lds_at<uint32_t>(tile_xhi_off<T, BLOCK>());
  const int t = xcd_tile(blockIdx.x, ntiles);
  if (t >= ntiles) return;
  const TileRec rec = tiles[t];
  // the node ids sit at a fixed pitch (padded with the last node), so their loads do not wait for
  // the tile's record (318k elements 9.3 -> 8.9 us; mixed PCG, 630k elements, 2.19 -> 2.13 ms)
  const uint32_t* nodes = node_tab + size_t(t) * pitch;
  const uint32_t n_own = rec.n_own;
  // first records: their loads are issued before the x gather so both chains overlap
  static_assert(!FACT || (MODE != OP_DIAG && !LANE && !COMB && std::is_same<T, TC>::value),
                "the factored product has no diagonal and reads no rows");
  typename std::conditional<FACT, RecF<T>, Rec>::type R;
  // the wavefront's records: w0, w0 + BLOCK, ... (64 each); lanes past the last record load it
  // again and add nothing
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t w0 = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x - lane)));
  auto load = [&](decltype(R)& r, uint32_t r0) {
    const uint32_t g = rec.elem_off + min(r0 + lane, rec.n_elem - 1u);
    if constexpr (FACT)
      load_rec_fact<T, MASS, UNI>(r, g, lid, kappa, mass);
    else
      load_rec<TC, MASS, sizeof(T), UNI ? 1 : 0, !COMB>(r, g, lid, kappa, mass, lap_fac, mass_fac, maxD, hFac);
  };
  const uint32_t kf = tile_kf_off<T>(XS, rec.n_touch);
  if (LANE) {   // the stencil table, copied while the gather runs (visible after the barrier)
    for (uint32_t i = threadIdx.x; i < KF_ELEMS; i += BLOCK) lds_at<T>(kf)[i] = KF[i];
  }
  // Gather.  Indexes past the end are clamped to the last slot, so a thread's OP_XC id loads,
  // then its x loads, go out together with no branch between them.  Owned nodes lead the list:
  // nid[0 .. OP_OC) are also the ids of the store phase.
  uint32_t nid[OP_XC];
  const uint32_t last = pitch - 1u;
#pragma unroll
  for (int q = 0; q < OP_XC; ++q) nid[q] = nodes[min(threadIdx.x + uint32_t(q * BLOCK), last)];
  load(R, w0);
  // FP32 residual and smoothing: the owned nodes' b and invd are loaded with the gather, so the
  // store phase waits on no global load.  FP64 loads them before the last barrier instead (held
  // from the gather on, they would take the kernel past the 64 VGPRs of eight wavefronts per
  // SIMD).  Lanes past the owned nodes load the first node's.
  constexpr bool SM = MODE == OP_SMOOTH || MODE == OP_SMOOTH0;
  constexpr bool RS = MODE == OP_RESID || SM;
  constexpr bool EARLY = RS && sizeof(T) == 4;
  T own_b[OP_OC], own_d[OP_OC];
  auto load_own = [&] {
    const uint32_t n0 = nodes[0];
#pragma unroll
    for (int q = 0; q < OP_OC; ++q) {
      const uint32_t n = threadIdx.x + uint32_t(q * BLOCK) < n_own ? nid[q] : n0;
      own_b[q] = io.b[n];
      if (SM) own_d[q] = io.invd[n];
    }
  };
  uint32_t own_bdy = 0;   // DIRMV: boundary flags of this thread's owned nodes, one bit each
  uint32_t xhi = 0;       // high word of max |x| over the values this thread staged
  if (MODE != OP_DIAG) {
    T v[OP_XC];
#pragma unroll
    for (int q = 0; q < OP_XC; ++q)
      v[q] = MODE == OP_SMOOTH0 ? T(0) + io.omega * (io.b[nid[q]] * io.invd[nid[q]]) : x[nid[q]];
    if (MODE == OP_DIRMV) {   // flags loaded beside x (both wait on the node ids only)
      uint8_t bf[OP_XC];
#pragma unroll
      for (int q = 0; q < OP_XC; ++q) bf[q] = io.bdy[nid[q]];
#pragma unroll
      for (int q = 0; q < OP_XC; ++q) {
        v[q] = bf[q] ? T(0) : v[q];
        if (q < OP_OC) own_bdy |= (bf[q] ? 1u : 0u) << q;
      }
      // The ids are taken as new values here, so that the store forms its addresses from them again:
      // the compiler otherwise keeps the gather's 64-bit offsets to the end, and the FP64 form with kappa
      // and mass takes 68 registers, above the 64 of two 1024-thread workgroups per CU (56 so: 2.8M
      // elements 45.0 -> 37.7 us, 1.5M 26.3 -> 23.9; 512-thread tiles 37.4 and 23.9).
#pragma unroll
      for (int q = 0; q < OP_OC; ++q) asm volatile("" : "+v"(nid[q]));
    }
    if (EARLY) load_own();
#pragma unroll
    for (int q = 0; q < OP_XC; ++q) {
      const uint32_t i = threadIdx.x + uint32_t(q * BLOCK);
      if (i < rec.n_touch) xs[i] = v[q];
      if constexpr (sizeof(T) == 8)
        xhi = max(xhi, uint32_t(uint64_t(__double_as_longlong(v[q])) >> 32) & 0x7fffffffu);
      else   // the FP32 bits order as |x| does; the maximum is converted once below
        xhi = max(xhi, __float_as_uint(v[q]) & 0x7fffffffu);
    }
  }
#pragma unroll
  for (int q = 0; q < OP_OC; ++q) {
    const uint32_t i = threadIdx.x + uint32_t(q * BLOCK);
    if (i < n_own) acc[i] = 0;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) xhi = max(xhi, uint32_t(__shfl_xor(int(xhi), off)));
  if ((threadIdx.x & 63) == 0) s_xhi[threadIdx.x >> 6] = xhi;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) xhi = max(xhi, s_xhi[w]);
  if constexpr (sizeof(T) == 4)
    xhi = uint32_t(uint64_t(__double_as_longlong(double(__uint_as_float(xhi)))) >> 32);
  // max |x| < 2^ex; a non-finite x makes every owned output of the tile NaN
  const bool finite = (xhi >> 20) < 0x7ffu;
  const int ex = MODE == OP_DIAG ? 1 : fx_ex<T>(xhi);
  const int es = fx_scale<T>(texp[t], ex);
  const bool big = FACT && fx_big<T>(ex);
  const uint32_t own_bytes = n_own * uint32_t(sizeof(T));
  for (uint32_t r0 = w0; r0 < rec.n_elem; r0 += BLOCK) {
    const bool in = r0 + lane < rec.n_elem;
    if constexpr (FACT) {   // the next records' loads are in flight during the evaluation
      decltype(R) Rn;
      load(Rn, r0 + BLOCK);
      eval_fact<T, MASS, XS, UNI>(R, in ? own_bytes : 0u, big ? es + FX_UP : es, big, lap_fac, mass_fac, maxD);
      R = Rn;
    } else {
      if (in) {
        if constexpr (LANE)
          eval_rows_lane<T, MASS, MODE, XS>(R, own_bytes, es, kf);
        else
          eval_rows<T, MASS, MODE, XS, COMB>(R, own_bytes, es, KF);
      }
      if (r0 + BLOCK < rec.n_elem) load(R, r0 + BLOCK);
    }
  }
  if (RS && !EARLY) load_own();   // in flight while the other wavefronts finish their records
  __syncthreads();
  double dot = 0.0;
#pragma unroll
  for (int q = 0; q < OP_OC; ++q) {
    const uint32_t i = threadIdx.x + uint32_t(q * BLOCK);
    if (i >= n_own) break;
    const uint32_t n = nid[q];
    const T v = finite ? T(fx_value<T>(acc[i], es)) : T(__builtin_nan(""));
    if (MODE == OP_MATVEC) {
      io.y[n] = v;
    } else if (MODE == OP_DIAG) {   // with boundary flags, the Dirichlet diagonal: 1 there
      io.y[n] = (io.bdy && io.bdy[n]) ? T(1) : v;
    } else if (MODE == OP_DIRMV) {
      io.y[n] = (own_bdy >> q) & 1u ? x[n] : v;
    } else if (MODE == OP_RESID) {
      io.y[n] = own_b[q] - v;
    } else if (SM) {
      io.y[n] = xs[i] + io.omega * ((own_b[q] - v) * own_d[q]);   // owned nodes lead the staged x
    } else {
      io.y[n] = v;
      dot += double(xs[i]) * double(v);
    }
  }
  if (MODE == OP_CG) {   // tile partial of p'.y, summed in a fixed order
    __syncthreads();
    const lds_ptr<double> red = lds_at<double>(0);   // over the sums, dead past the barrier
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) dot += __shfl_down(dot, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = dot;
    __syncthreads();
    if (threadIdx.x == 0) {
      double tot = 0.0;
      for (int w = 0; w < NW; ++w) tot += red[w];
      io.part[t] = tot;
    }
  }
}

// Two applications of the operator in one launch, for meshes whose single sweeps are a chain of
// latencies: a sweep x' = x + omega (invd (b - A x)), then PAIR_SMOOTH: another one, y = x'';
// PAIR_RESID: y = x' and r = b - A x'.  A tile (build_pair_tiles) updates all nodes of its own
// records in the first sweep, so neighbouring tiles repeat the sweep on each other's border nodes
// instead of exchanging them through memory and a launch.  A single sweep of a small mesh takes 4.5
// to 5 us in a chain of dependent launches, most of it the launch and two hops to memory; the second
// sweep here adds about 3 (PAIR_MAX_ELEMS has what a solve gains).
enum PairMode { PAIR_SMOOTH = 0, PAIR_RESID = 1 };
template <class T>
struct PairIO {
  T* y;
  T* r;            // PAIR_RESID
  const T* b;
  const T* invd;
  T omega;
};
constexpr int PAIR_BLOCK = 512;
constexpr int PAIR_XC = 4;   // touched and first-sweep nodes per thread, at most
constexpr int PAIR_OC = 3;

template <class T, bool MASS, int MODE, bool UNI>
__global__ void __launch_bounds__(PAIR_BLOCK)
tile_pair_kernel(const TileRec* __restrict__ tiles, const uint32_t* __restrict__ node_tab, const T* __restrict__ x,
                 const uint16_t* __restrict__ lid, const int2* __restrict__ texp, int ntiles, uint32_t pitch,
                 const T* __restrict__ kappa, const T* __restrict__ mass, PairIO<T> io, double u1, double u2,
                 uint32_t maxD) {
  constexpr int BLOCK = PAIR_BLOCK, NW = BLOCK / 64;
  constexpr uint32_t XS = tile_xs_off<T, BLOCK>();
  static_assert(PAIR_OC * BLOCK <= int(op_own_cap(BLOCK)), "the first sweep's sums fit");
  const lds_ptr<fx_acc_t<T>> acc = lds_at<fx_acc_t<T>>(0);
  const lds_ptr<T> xs = lds_at<T>(XS);
  const lds_ptr<uint32_t> s_xhi = lds_at<uint32_t>(tile_xhi_off<T, BLOCK>());
  const int t = xcd_tile(blockIdx.x, ntiles);
  if (t >= ntiles) return;
  const TileRec rec = tiles[t];
  const uint32_t* nodes = node_tab + size_t(t) * pitch;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t w0 = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x - lane)));
  RecF<T> R;
  auto load = [&](RecF<T>& r, uint32_t r0) {
    load_rec_fact<T, MASS, UNI>(r, rec.elem_off + min(r0 + lane, rec.n_elem - 1u), lid, kappa, mass);
  };
  // slots past the end are clamped to the last node, as in tile_op_kernel
  uint32_t nid[PAIR_XC];
  const uint32_t last = pitch - 1u;
#pragma unroll
  for (int q = 0; q < PAIR_XC; ++q) nid[q] = nodes[min(threadIdx.x + uint32_t(q * BLOCK), last)];
  load(R, w0);
  T v[PAIR_XC], ob[PAIR_OC], od[PAIR_OC];
#pragma unroll
  for (int q = 0; q < PAIR_XC; ++q) v[q] = x[nid[q]];
#pragma unroll
  for (int q = 0; q < PAIR_OC; ++q) {
    ob[q] = io.b[nid[q]];
    od[q] = io.invd[nid[q]];
  }
  uint32_t xhi = 0;
  auto take = [&](T val) {   // FP32 bits order as |x| does, converted by max_x
    if constexpr (sizeof(T) == 8)
      xhi = max(xhi, uint32_t(uint64_t(__double_as_longlong(val)) >> 32) & 0x7fffffffu);
    else
      xhi = max(xhi, __float_as_uint(val) & 0x7fffffffu);
  };
  auto wave_max = [&] {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) xhi = max(xhi, uint32_t(__shfl_xor(int(xhi), off)));
    if (lane == 0) s_xhi[threadIdx.x >> 6] = xhi;
  };
  auto max_x = [&] {   // high word of the tile's max |x|
#pragma unroll
    for (int w = 0; w < NW; ++w) xhi = max(xhi, s_xhi[w]);
    if constexpr (sizeof(T) == 4)
      xhi = uint32_t(uint64_t(__double_as_longlong(double(__uint_as_float(xhi)))) >> 32);
  };
#pragma unroll
  for (int q = 0; q < PAIR_XC; ++q) {
    const uint32_t i = threadIdx.x + uint32_t(q * BLOCK);
    if (i < rec.n_touch) xs[i] = v[q];
    take(v[q]);
  }
#pragma unroll
  for (int q = 0; q < PAIR_OC; ++q) {
    const uint32_t i = threadIdx.x + uint32_t(q * BLOCK);
    if (i < rec.n_own) acc[i] = 0;
  }
  wave_max();
  __syncthreads();
  max_x();
  bool finite = (xhi >> 20) < 0x7ffu;
  int ex = fx_ex<T>(xhi), es = fx_scale<T>(texp[t], ex);
  auto sweep = [&](uint32_t n_elem, uint32_t n_own) {
    const uint32_t own_bytes = n_own * uint32_t(sizeof(T));
    const bool big = fx_big<T>(ex);
    for (uint32_t r0 = w0; r0 < n_elem; r0 += BLOCK) {
      RecF<T> Rn;
      // the last round loads the first records again, for the next sweep
      load(Rn, r0 + BLOCK < n_elem ? r0 + BLOCK : w0);
      eval_fact<T, MASS, XS, UNI>(R, r0 + lane < n_elem ? own_bytes : 0u, big ? es + FX_UP : es, big, u1, u2, maxD);
      R = Rn;
    }
  };
  sweep(rec.n_elem, rec.n_own);
  __syncthreads();
  xhi = 0;
#pragma unroll
  for (int q = 0; q < PAIR_OC; ++q) {
    const uint32_t i = threadIdx.x + uint32_t(q * BLOCK);
    if (i < rec.n_own) {
      const T a = finite ? T(fx_value<T>(acc[i], es)) : T(__builtin_nan(""));
      const T xn = xs[i] + io.omega * ((ob[q] - a) * od[q]);
      xs[i] = xn;
      acc[i] = 0;
      take(xn);
    }
  }
  wave_max();
  __syncthreads();
  max_x();
  finite = (xhi >> 20) < 0x7ffu;
  ex = fx_ex<T>(xhi);
  es = fx_scale<T>(texp[t], ex);
  sweep(rec.n_elem2, rec.n_own2);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PAIR_OC; ++q) {
    const uint32_t i = threadIdx.x + uint32_t(q * BLOCK);
    if (i >= rec.n_own2) break;
    const T a = finite ? T(fx_value<T>(acc[i], es)) : T(__builtin_nan(""));
    if (MODE == PAIR_SMOOTH) {
      io.y[nid[q]] = xs[i] + io.omega * ((ob[q] - a) * od[q]);
    } else {
      io.y[nid[q]] = xs[i];
      io.r[nid[q]] = ob[q] - a;
    }
  }
}

// f_out[j] = f_in[j] + sum_k W[s][pos][k] c[cnl[k]] for every fine node j (prolongation
// P = R^T): the coarse shape functions of the coarse element holding node j.
template <class T>
__global__ void __launch_bounds__(256)
prolong_kernel(uint32_t nf, const uint32_t* __restrict__ celem, const uint8_t* __restrict__ pos,
               const uint32_t* __restrict__ cnl, const uint8_t* __restrict__ cs,
               const T* __restrict__ W, const T* __restrict__ c, const T* __restrict__ f_in,
               T* __restrict__ f_out, const uint8_t* __restrict__ cbdy = nullptr,
               const uint8_t* __restrict__ fbdy = nullptr) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nf) return;
  const uint32_t ce = celem[j];
  const T* w = W + (size_t(cs[ce]) * 27 + pos[j]) * 8;
  const uint4 a = reinterpret_cast<const uint4*>(cnl)[2 * ce];
  const uint4 b = reinterpret_cast<const uint4*>(cnl)[2 * ce + 1];
  const uint32_t idx[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  // the 8 coarse values are loaded whatever the weights (they sit in L2): the loads then wait
  // on the vertex ids only, not on the weights as well; zero weights still add nothing
  T cv[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) cv[k] = c[idx[k]];
  if (cbdy) {   // Dirichlet: no entry from a boundary coarse node
#pragma unroll
    for (int k = 0; k < 8; ++k) cv[k] = cbdy[idx[k]] ? T(0) : cv[k];
  }
  T acc = T(0);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const T wk = w[k];
    acc += (wk != T(0)) ? wk * cv[k] : T(0);
  }
  if (fbdy && fbdy[j]) acc = T(0);   // Dirichlet: no entry into a boundary fine node
  f_out[j] = (f_in ? f_in[j] : T(0)) + acc;
}

// c[i] = sum_p w_p f[col_p] over row i of R = P^T (CSR built on the host; gather, no
// atomics).  RLANES lanes share a row (rows hold about 4-30 entries) and combine their
// partial sums with shuffles; the sum order is fixed.
constexpr int RLANES = 4;
// With x1 given, also the coarse level's first smoothing sweep from a zero guess:
// x1 = omega (c * invd), as smooth_first_kernel forms it.
template <class T>
__global__ void __launch_bounds__(256)
restrict_kernel(uint32_t nc, const uint32_t* __restrict__ rowptr, const uint32_t* __restrict__ col,
                const float* __restrict__ w, const T* __restrict__ f, T* __restrict__ c, T omega = T(0),
                const T* __restrict__ invd = nullptr, T* __restrict__ x1 = nullptr,
                const uint8_t* __restrict__ cbdy = nullptr, const uint8_t* __restrict__ fbdy = nullptr) {
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t i = gid / RLANES, lane = gid % RLANES;
  T acc = T(0);
  if (i < nc) {
    const uint32_t p1 = rowptr[i + 1];
    // RU entries of a lane per step: their column loads, then their f loads, go out together
    // (the sum still runs over the lane's entries in order)
    constexpr int RU = 8;
    for (uint32_t p0 = rowptr[i] + lane; p0 < p1; p0 += RU * RLANES) {
      uint32_t e[RU];
      T fv[RU], wv[RU];
#pragma unroll
      for (int u = 0; u < RU; ++u) {
        const uint32_t p = p0 + u * RLANES;
        e[u] = p < p1 ? col[p] : 0u;
        wv[u] = p < p1 ? T(w[p]) : T(0);
      }
#pragma unroll
      for (int u = 0; u < RU; ++u) fv[u] = p0 + u * RLANES < p1 ? f[e[u]] : T(0);
      if (fbdy) {   // Dirichlet: no entry from a boundary fine node
#pragma unroll
        for (int u = 0; u < RU; ++u)
          if (p0 + u * RLANES < p1 && fbdy[e[u]]) fv[u] = T(0);
      }
#pragma unroll
      for (int u = 0; u < RU; ++u) {
        if (p0 + u * RLANES >= p1) break;
        acc += wv[u] * fv[u];
      }
    }
  }
#pragma unroll
  for (int off = RLANES / 2; off > 0; off >>= 1) acc += __shfl_down(acc, off, RLANES);
  if (i < nc && lane == 0) {
    if (cbdy && cbdy[i]) acc = T(0);   // Dirichlet: no entry into a boundary coarse node
    c[i] = acc;
    if (x1) x1[i] = T(0) + omega * (acc * invd[i]);
  }
}

// ---------------------------------------------------------------- transfers through LDS
// Both transfers as sparse products whose workgroups gather the distinct columns of their rows once
// into LDS (build_gather).  The forms above chase three dependent loads (a row's place, its columns,
// their values) and issue up to 12 scattered loads per fine node, 40% of them for zero weights; here
// the column lists and the rows' entries (2 bytes each) arrive together, then the values, and the
// products read LDS.  NS: column slots per thread.  The zero slot past the list takes unused
// entries, so whole rows are read without a count.
constexpr uint32_t GE_ID = (1u << GATHER_BITS) - 1u;
template <class T>
__device__ __forceinline__ T gather_weight(uint32_t e) {
  return T(float((e >> GATHER_BITS) + 1u) * 0.03125f);
}
// stages the values of the block's columns (0 where zero flags one), and the zero slot
template <class T, int NS>
__device__ __forceinline__ void gather_stage(T* xs, uint32_t pitch, const uint32_t* __restrict__ list,
                                             const T* __restrict__ x, const uint8_t* __restrict__ zero) {
  uint32_t id[NS];
  T v[NS];
#pragma unroll
  for (int q = 0; q < NS; ++q) id[q] = list[min(threadIdx.x + uint32_t(q) * blockDim.x, pitch - 1u)];
#pragma unroll
  for (int q = 0; q < NS; ++q) v[q] = x[id[q]];
  if (zero) {
#pragma unroll
    for (int q = 0; q < NS; ++q) v[q] = zero[id[q]] ? T(0) : v[q];
  }
#pragma unroll
  for (int q = 0; q < NS; ++q) {
    const uint32_t i = threadIdx.x + uint32_t(q) * blockDim.x;
    if (i < pitch) xs[i] = v[q];
  }
  if (threadIdx.x == 0) xs[pitch] = T(0);
}

// f_out = f_in + P c: a thread per fine node, its up to 8 entries in 16 bytes.
constexpr int PT_ROWS = 256;
template <class T, int NS>
__global__ void __launch_bounds__(PT_ROWS)
prolong_tile_kernel(uint32_t nf, uint32_t pitch, const uint32_t* __restrict__ list, const uint4* __restrict__ ent,
                    const T* __restrict__ c, const T* __restrict__ f_in, T* __restrict__ f_out,
                    const uint8_t* __restrict__ cbdy, const uint8_t* __restrict__ fbdy) {
  extern __shared__ __align__(16) unsigned char gather_lds[];
  T* xs = reinterpret_cast<T*>(gather_lds);
  const uint32_t j = blockIdx.x * PT_ROWS + threadIdx.x, jc = min(j, nf - 1u);
  const uint4 e4 = ent[jc];
  const T f = f_in ? f_in[jc] : T(0);
  gather_stage<T, NS>(xs, pitch, list + size_t(blockIdx.x) * pitch, c, cbdy);
  const bool out0 = fbdy && fbdy[jc];   // Dirichlet: no entry into a boundary fine node
  __syncthreads();
  if (j >= nf) return;
  const uint32_t e[4] = {e4.x, e4.y, e4.z, e4.w};
  T acc = T(0);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint32_t ek = (e[k >> 1] >> (16 * (k & 1))) & 0xffffu;
    acc += gather_weight<T>(ek) * xs[ek & GE_ID];
  }
  f_out[j] = f + (out0 ? T(0) : acc);
}

// c = P^T f and x1 (see restrict_kernel): RT_LANES lanes for each of RT_ROWS coarse nodes.  Where the
// launch does not fill the device 64 rows, FP64 with 8 lanes (FP64 V-cycle 149.6 -> 147.7 us, of 11k
// elements 84.2 -> 81.9), FP32 with the 4 of restrict_kernel, whose sums it keeps; from RT_LARGE coarse
// nodes on 128 rows with 2 lanes and two partial sums each, the same sums: there fewer workgroups and
// shuffles count.  Both transfers in turn on the same buffers, FP32 / FP64 us, in one run: 461k fine and
// 135k coarse nodes, 2 lanes 8.5 / 10.4, 4 lanes 9.1 / 12.1, 8 lanes 10.5 / 13.3, the general kernels 11.3
// / 14.6; 5.5M and 2.1M: 70 / 89, 104 / 124, 127 / 152 and 95 / 137.  Against the kernels before (general,
// the restriction with packed entries): 10.5 / 13.4 -> 8.9 / 10.6 and 84 / 121 -> 67 / 83; with another
// mesh and vectors each time, FP32, 461k nodes, 11.4 -> 10.1.  The restriction's column lists are padded
// to the largest block's (1447 columns on this mesh, 605 on average), which is most of what is left.
constexpr uint32_t RT_ROWS_SMALL = 64, RT_ROWS_LARGE = 128;
constexpr uint32_t RT_LARGE = 80000;
template <class T, int NS, int RT_LANES, int RT_ROWS>
__global__ void __launch_bounds__(RT_LANES * RT_ROWS)
restrict_tile_kernel(uint32_t nc, uint32_t pitch, const uint32_t* __restrict__ list,
                     const uint32_t* __restrict__ rowptr, const uint16_t* __restrict__ ent, const T* __restrict__ f,
                     T* __restrict__ c, T omega, const T* __restrict__ invd, T* __restrict__ x1,
                     const uint8_t* __restrict__ cbdy, const uint8_t* __restrict__ fbdy) {
  extern __shared__ __align__(16) unsigned char gather_lds[];
  T* xs = reinterpret_cast<T*>(gather_lds);
  const uint32_t i = blockIdx.x * RT_ROWS + threadIdx.x / RT_LANES, lane = threadIdx.x % RT_LANES;
  const uint32_t ic = min(i, nc - 1u);
  const uint32_t p0 = rowptr[ic] + lane, p1 = rowptr[ic + 1];
  const T dv = x1 ? invd[ic] : T(0);
  gather_stage<T, NS>(xs, pitch, list + size_t(blockIdx.x) * pitch, f, fbdy);
  constexpr int RU = 32 / RT_LANES;   // a row of up to 32 entries in one step
  uint32_t e[RU];
#pragma unroll
  for (int u = 0; u < RU; ++u) e[u] = p0 + u * RT_LANES < p1 ? uint32_t(ent[p0 + u * RT_LANES]) : pitch;
  __syncthreads();
  constexpr int NA = RT_LANES < RLANES ? RLANES / RT_LANES : 1;   // partial sums per lane, in restrict_kernel's order
  T part[NA];
#pragma unroll
  for (int a = 0; a < NA; ++a) part[a] = T(0);
#pragma unroll
  for (int u = 0; u < RU; ++u) part[u % NA] += gather_weight<T>(e[u]) * xs[e[u] & GE_ID];
  for (uint32_t p = p0 + RU * RT_LANES; p < p1; p += NA * RT_LANES)
#pragma unroll
    for (int a = 0; a < NA; ++a)
      if (p + a * RT_LANES < p1) {
        const uint32_t ep = ent[p + a * RT_LANES];
        part[a] += gather_weight<T>(ep) * xs[ep & GE_ID];
      }
  T acc = part[0];
#pragma unroll
  for (int a = 1; a < NA; ++a) acc += part[a];
#pragma unroll
  for (int off = RT_LANES / 2; off > 0; off >>= 1) acc += __shfl_down(acc, off, RT_LANES);
  if (i < nc && lane == 0) {
    if (cbdy && cbdy[i]) acc = T(0);
    c[i] = acc;
    if (x1) x1[i] = T(0) + omega * (acc * dv);
  }
}

template <class T>
__global__ void fill_kernel(T* __restrict__ v, T val, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = val;
}

}  // namespace dgh
