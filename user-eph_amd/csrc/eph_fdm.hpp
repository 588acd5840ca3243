// eph_fdm.hpp -- device functions of the T_e stencil (EPH_FDM::solve,
// eph_fdm.h:315-395), shared by the single-grid and the batched kernels.
#pragma once

#include "eph_devfn.hpp"

namespace eph {

// A divisor used for many quotients: its reciprocal rounded to 53 bits and the
// rest to about 106.  The IEEE division the compiler emits is about ten
// dependent instructions with a quarter-rate reciprocal among them; with the
// reciprocal known, the same rounded quotient takes four.  q0 = x rd + x rl is
// within one ulp of x / d, and then q0 + (x - q0 d) rd with rd = RN(1/d) is
// RN(x / d) (P. Markstein, IBM J. Res. Dev. 34 (1990) 111).  The remainder has
// to be exact, so this holds for operands away from the ends of the exponent
// range; a zero dividend may come out as a zero of either sign.
struct Divisor {
  double d = 1.0, rd = 1.0, rl = 0.0;
};
static __host__ __device__ __forceinline__ Divisor divisor(double d) {
  Divisor v;
  v.d = d;
  v.rd = 1.0 / d;
  v.rl = __builtin_fma(-v.rd, d, 1.0) * v.rd;
  return v;
}
static __device__ __forceinline__ double div_fast(const double x, const Divisor& v) {
  const double q = __builtin_fma(x, v.rd, x * v.rl);
  return __builtin_fma(__builtin_fma(-q, v.d, x), v.rd, q);
}
// x is zero or 2^-e <= |x| < 2^e
static __host__ __device__ __forceinline__ bool in_range(const double x, const int e) {
  union { double d; uint64_t u; } b;
  b.d = x;
  const unsigned ex = static_cast<unsigned>(b.u >> 52) & 0x7ffu;
  return (ex - (1023u - e) < 2u * e) | (x == 0.0);
}
// Operands for which every quotient of a sub-step can be formed by div_fast:
// spacings within 2^+-20, the update's divisor and kappa (or 0) within 2^+-60,
// temperatures, dT_e and S (or 0) within 2^+-500.  A sum or difference of such
// temperatures is 0 or at least 2^-552, and what the stencil makes of it 0 or
// at least 2^-760, so no quotient, remainder or correction leaves the range of
// normal numbers.
static __host__ __device__ __forceinline__ bool fdm_range_T(const double T) { return in_range(T, 500); }

// A cell's values that stay as they are over the sub-steps of a solve: its
// neighbours after the wall rule, kappa, dT_e, S and the divisor of the
// update (rho C, or rho where the cell is temperature dependent).  flat: the
// two neighbours of every dimension have equal kappa.
struct FdmCell {
  int p[3], q[3];
  double kr, dT, S;
  Divisor div;
  int flag;
  bool flat, tdyn;
};
static __host__ __device__ __forceinline__ bool fdm_range_cell(const FdmCell& c) {
  return in_range(c.kr, 60) & in_range(c.dT, 500) & in_range(c.S, 500) & in_range(c.div.d, 60) &
         (c.div.d > 0.0);
}
static __host__ __device__ __forceinline__ bool fdm_range_grid(const Divisor* d3) {
  return in_range(d3[0].d, 20) & in_range(d3[1].d, 20) & in_range(d3[2].d, 20) & (d3[0].d > 0.0) &
         (d3[1].d > 0.0) & (d3[2].d > 0.0);
}

// One explicit sub-step of one cell (eph_fdm.h:315-395): the 7-point
// variable-kappa stencil in the reference's order, the update and the clamp.
// MODE 0: uniform material without walls; 1: values per cell; 2: also
// temperature-dependent cells.  T and kappa are indexed by r, p and q.
// fast: every operand is in the ranges above; divisions otherwise.
//
// The stencil sum starts at +0 and so never becomes -0: zero terms (the first
// term of a flat dimension) can be left out and zero quotients may have either
// sign without changing a bit.
template <int MODE>
static __device__ __forceinline__ double fdm_advance(const FdmCell& c, const Divisor* d3,
                                                     const GridView& g, const double* T,
                                                     const double* kappa, const int r,
                                                     const double inner_dt, const bool fast) {
  const double Tr = T[r], Tr2 = 2.0 * Tr;
  double a[3], b[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    a[d] = T[c.q[d]];
    b[d] = T[c.p[d]];
  }
  const bool curved = MODE != 0 && !c.flat;
  double ddT = 0.0, rate;
  if (fast) {
    double y[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) y[d] = div_fast(div_fast(a[d] + b[d] - Tr2, d3[d]), d3[d]);
    if (!curved) {
#pragma unroll
      for (int d = 0; d < 3; ++d) ddT += c.kr * y[d];
    } else {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double t = (kappa[c.q[d]] - kappa[c.p[d]]) * (a[d] - b[d]);
        ddT += div_fast(div_fast(t, d3[d]), d3[d]) / 4.0;
        ddT += c.kr * y[d];
      }
    }
    if (MODE != 0 && c.flag == kCellZeroDerivative) ddT = 0.0;
    rate = div_fast(ddT + c.dT + c.S, c.div);
  } else {
    if (MODE == 0 || c.flag != kCellZeroDerivative) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double h = d3[d].d;
        const double dk = MODE != 0 ? kappa[c.q[d]] - kappa[c.p[d]] : 0.0;
        const double t = dk * (a[d] - b[d]);
        if (t != 0.0) ddT += t / h / h / 4.0;
        ddT += c.kr * ((a[d] + b[d] - Tr2) / h / h);
      }
    }
    rate = (ddT + c.dT + c.S) / c.div.d;
  }
  double t = Tr;
  if (MODE == 0 || c.flag == kCellDynamic) {
    if (MODE == 2 && c.tdyn) {
      double E = linear_fwd(g, t);
      E += rate * inner_dt;
      t = linear_rev(g, E);
    } else {
      t += rate * inner_dt;
    }
  }
  if (t < 0.0) t = 0.0;
  return t;
}

// the wall rule on a cell's neighbours, and what it leaves of kappa
static __device__ __forceinline__ void fdm_walls(FdmCell& c, const int r, const int8_t* flag,
                                                 const double* kappa) {
  c.flat = true;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (flag[c.q[d]] == kCellZeroDerivative) c.q[d] = r;
    else if (flag[c.p[d]] == kCellZeroDerivative) c.p[d] = r;
    c.flat = c.flat && kappa[c.q[d]] - kappa[c.p[d]] == 0.0;
  }
}

// the cell's own values from the grid's cell r (neighbours apart); RECIP: with
// the reciprocal of the update's divisor
template <int MODE, bool RECIP = true>
static __device__ __forceinline__ void fdm_load(FdmCell& c, const GridView& g, const int r) {
  c.dT = g.dT[r];
  if (MODE == 0) return;
  c.kr = g.kappa[r];
  c.S = g.S[r];
  c.flag = g.flag[r];
  c.tdyn = MODE == 2 && g.tdyn[r] == 1;
  const double div = c.tdyn ? g.rho[r] : g.rho[r] * g.C[r];
  if (RECIP) c.div = divisor(div);
  else c.div.d = div;
}

// periodic neighbours of cell r in i + j nx + k nx ny order
static __device__ __forceinline__ void fdm_neighbours(const int r, const int nx, const int ny,
                                                      const int nz, int* p, int* q) {
  const int i = r % nx, j = (r / nx) % ny, k = r / (nx * ny), pl = nx * ny;
  p[0] = i > 0 ? r - 1 : r + (nx - 1);
  q[0] = i < nx - 1 ? r + 1 : r - (nx - 1);
  p[1] = j > 0 ? r - nx : r + (ny - 1) * nx;
  q[1] = j < ny - 1 ? r + nx : r - (ny - 1) * nx;
  p[2] = k > 0 ? r - pl : r + (nz - 1) * pl;
  q[2] = k < nz - 1 ? r + pl : r - (nz - 1) * pl;
}

// one explicit sub-step of EPH_FDM::solve (eph_fdm.h:315-395) for cell r, from
// Tin into Tout
template <bool TDYN>
__device__ __forceinline__ void fdm_cell(const GridView& g, const double* __restrict__ Tin,
                                         double* __restrict__ Tout, const int r,
                                         const double inner_dt) {
  constexpr int MODE = TDYN ? 2 : 1;
  FdmCell c;
  fdm_neighbours(r, g.nx, g.ny, g.nz, c.p, c.q);
  fdm_load<MODE, false>(c, g, r);
  fdm_walls(c, r, g.flag, g.kappa);
  // one quotient per divisor: a reciprocal would be the division over again
  Divisor d3[3];
  d3[0].d = g.dx; d3[1].d = g.dy; d3[2].d = g.dz;
  Tout[r] = fdm_advance<MODE>(c, d3, g, Tin, g.kappa, r, inner_dt, false);
}

}  // namespace eph
