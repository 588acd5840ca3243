// eph_adjoint.hip -- reverse-mode (adjoint) kernels of one MD step with the
// fix: vector-Jacobian products of the FDM stencil, the deposit, the Verlet
// kicks, pair lj/cut, the force sweep (stages 2 + 3 of force_prl), the w sweep
// (stage 1), alpha(rho) and the density sweep.  Forward expressions are those
// of eph_kernels.hip (fix_eph.cpp:431-466, 702-836, 364-390; eph_fdm.h:315-395);
// each pair term is differentiated by hand.  The neighbour sweeps gather; only
// the T_e cells and the table gradient are added to with FP64 atomics, so
// gradients are deterministic up to the order of those additions.
#include "eph_adjoint.hpp"
#include "eph_devfn.hpp"

namespace eph {

namespace {

// value and d/dr^2 of rho(r^2) of element e at x = r^2 (the interval and cubic
// of rho_r2_at, interleaved tables)
__device__ __forceinline__ void rho_r2_vd(const TablesView& t, int e, double x, double* v, double* dv) {
  int i = static_cast<int>(x * t.inv_dr2);
  i = i < 0 ? 0 : (i < t.n_rho - 1 ? i : t.n_rho - 1);
  const double4 c = t.rho_r2[i * t.n_elem + e];
  *v = c.x + x * (c.y + x * (c.z + x * c.w));
  *dv = c.y + x * (2.0 * c.z + 3.0 * x * c.w);
}

inline int nblk(long n) { return static_cast<int>((n + kBlock - 1) / kBlock); }

}  // namespace

// ------------------------------------------------------------------ FDM
// one sub-step of k_fdm_substep in reverse:
// Tb_in += (dT_out/dT_in)^T Tb_out, dTb += (dT_out/d dT)^T Tb_out, and with
// temperature-dependent cells (TDYN) kb += (dT_out/d kappa)^T Tb_out.  A
// temperature-dependent cell updates in energy space, T_out =
// E^-1(E(T_in) + (ddT + dT + S) / rho dt_in), whose derivatives are the
// slopes of the two piecewise-linear lookups; the others update
// T_out = T_in + (ddT + dT + S) / (rho C) dt_in.
template <bool TDYN>
__global__ __launch_bounds__(kBlock) void k_adj_fdm(GridView g, const double* __restrict__ Tin,
                                                    const double* __restrict__ Tb_out,
                                                    double* Tb_in, double* dTb, double* kb,
                                                    double inner_dt, int G) {
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r >= G) return;
  const double tb = Tb_out[r];
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int i = r % nx, j = (r / nx) % ny, k = r / (nx * ny);
  const int fr = g.flag[r];
  // forward value before the clamp
  double ddT = 0.0;
  int pp[3], qq[3];
  const double dd[3] = {g.dx, g.dy, g.dz};
  if (fr != kCellZeroDerivative) {
    int p, q;
    p = i > 0 ? r - 1 : r + (nx - 1);
    q = i < nx - 1 ? r + 1 : r - (nx - 1);
    if (g.flag[q] == kCellZeroDerivative) q = r;
    else if (g.flag[p] == kCellZeroDerivative) p = r;
    pp[0] = p; qq[0] = q;
    p = j > 0 ? r - nx : r + (ny - 1) * nx;
    q = j < ny - 1 ? r + nx : r - (ny - 1) * nx;
    if (g.flag[q] == kCellZeroDerivative) q = r;
    else if (g.flag[p] == kCellZeroDerivative) p = r;
    pp[1] = p; qq[1] = q;
    const int pl = nx * ny;
    p = k > 0 ? r - pl : r + (nz - 1) * pl;
    q = k < nz - 1 ? r + pl : r - (nz - 1) * pl;
    if (g.flag[q] == kCellZeroDerivative) q = r;
    else if (g.flag[p] == kCellZeroDerivative) p = r;
    pp[2] = p; qq[2] = q;
    const double Tr = Tin[r], kr = g.kappa[r];
    for (int d = 0; d < 3; ++d) {
      const int P = pp[d], Q = qq[d];
      ddT += (g.kappa[Q] - g.kappa[P]) * (Tin[Q] - Tin[P]) / dd[d] / dd[d] / 4.0;
      ddT += kr * ((Tin[Q] + Tin[P] - 2.0 * Tr) / dd[d] / dd[d]);
    }
  }
  double T = Tin[r];
  double kfac = 0.0;  // dT_out / d ddT (= dT_out / d dT)
  double sfac = 1.0;  // dT_out / dT_in through the cell's own update
  if (fr == kCellDynamic) {
    if (TDYN && g.tdyn[r] == 1) {
      const double E = linear_fwd(g, T) + (ddT + g.dT[r] + g.S[r]) / g.rho[r] * inner_dt;
      const double inv = linear_rev_slope(g, E);
      sfac = inv * linear_fwd_slope(g, T);
      kfac = inv * inner_dt / g.rho[r];
      T = linear_rev(g, E);
    } else {
      kfac = inner_dt / (g.rho[r] * g.C[r]);
      T += (ddT + g.dT[r] + g.S[r]) / (g.rho[r] * g.C[r]) * inner_dt;
    }
  }
  if (T < 0.0 || tb == 0.0) return;  // clamped to 0 K: no dependence
  atomicAdd(&Tb_in[r], tb * sfac);
  if (fr != kCellDynamic) return;
  atomicAdd(&dTb[r], tb * kfac);
  const double kr = g.kappa[r];
  for (int d = 0; d < 3; ++d) {
    const int P = pp[d], Q = qq[d];
    const double h2 = dd[d] * dd[d];
    const double cq = (g.kappa[Q] - g.kappa[P]) / h2 / 4.0 + kr / h2;
    const double cp = -(g.kappa[Q] - g.kappa[P]) / h2 / 4.0 + kr / h2;
    atomicAdd(&Tb_in[Q], tb * kfac * cq);
    atomicAdd(&Tb_in[P], tb * kfac * cp);
    atomicAdd(&Tb_in[r], tb * kfac * (-2.0 * kr / h2));
    if (TDYN) {
      // ddT's dependence on kappa at q, p and the cell itself
      const double dq = (Tin[Q] - Tin[P]) / h2 / 4.0;
      atomicAdd(&kb[Q], tb * kfac * dq);
      atomicAdd(&kb[P], -tb * kfac * dq);
      atomicAdd(&kb[r], tb * kfac * ((Tin[Q] + Tin[P] - 2.0 * Tin[r]) / h2));
    }
  }
}

// kappa(T) of the temperature-dependent cells is evaluated once per solve at
// the solve's starting T_e (eph_fdm.h:280-287): its gradient, gathered over
// the sub-steps in kb, goes to that T_e through the spline's slope
__global__ __launch_bounds__(kBlock) void k_adj_kappa_T(GridView g, const double* __restrict__ T0,
                                                        const double* __restrict__ kb, double* Tb,
                                                        int G) {
  const int c = blockIdx.x * kBlock + threadIdx.x;
  if (c >= G || !g.tdyn[c] || kb[c] == 0.0) return;
  Tb[c] += kb[c] * cubic_slope(g.kappa_T, g.n_kT, g.inv_dT_k, T0[c]);
}

// ------------------------------------------------------------- deposit
// dE_i = -(f_i . v'_i) dt for the friction and random parts; each feeds the
// tally (weight Eb) and dT_e of its cell (weight dTb / (dV dt))
__global__ __launch_bounds__(kBlock) void k_adj_deposit(AdjStepView s, GridView g, AtomsView a,
                                                        double dt, int fric, int rnd, double Eb,
                                                        const double* __restrict__ dTb,
                                                        AdjBuffers b) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.nlocal || !(a.mask[i] & a.groupbit)) return;
  const double4 x = s.rec[i].p;
  const double4 v = s.vn[i];
  const int c = cell_of(g, x.x, x.y, x.z);
  const double w = Eb + (dTb ? dTb[c] / (g.dV * dt) : 0.0);
  const int fs = s.fstride;
  double4 vb = b.vnb[i];
  if (fric) {
    const double fx = s.fE[i], fy = s.fE[fs + i], fz = s.fE[2 * fs + i];
    double4 fb = b.fEb[i];
    fb.x -= w * dt * v.x; fb.y -= w * dt * v.y; fb.z -= w * dt * v.z;
    b.fEb[i] = fb;
    vb.x -= w * dt * fx; vb.y -= w * dt * fy; vb.z -= w * dt * fz;
  }
  if (rnd) {
    const double fx = s.fR[i], fy = s.fR[fs + i], fz = s.fR[2 * fs + i];
    double4 fb = b.fRb[i];
    fb.x -= w * dt * v.x; fb.y -= w * dt * v.y; fb.z -= w * dt * v.z;
    b.fRb[i] = fb;
    vb.x -= w * dt * fx; vb.y -= w * dt * fy; vb.z -= w * dt * fz;
  }
  b.vnb[i] = vb;
}

// ------------------------------------------------------ final integrate
// v' = vh + (dtf / m) f  (group atoms; others keep vh)
__global__ __launch_bounds__(kBlock) void k_adj_final(AtomsView a, StepParams p, int noint,
                                                      AdjBuffers b) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.nlocal) return;
  const double4 vn = b.vnb[i];
  double4 vh = b.vhb[i];
  vh.x += vn.x; vh.y += vn.y; vh.z += vn.z;
  b.vhb[i] = vh;
  if (!noint && (a.mask[i] & a.groupbit)) {
    const double c = p.dtf / p.mass[a.type[i]];
    double4 ft = b.ftb[i];
    ft.x += c * vn.x; ft.y += c * vn.y; ft.z += c * vn.z;
    b.ftb[i] = ft;
  }
}

// ------------------------------------------------- neighbour sweeps
// The full lists are symmetric: when j (or a ghost of it) is in i's list, an
// image of i at the opposite vector is in j's.  So atom i gathers everything
// its pairs contribute to it, both as the centre (i, j) and as the neighbour
// of (j, i), whose terms depend on e only through its sign; nothing is
// scattered, ghosts collect no adjoint, and every sum has one owner.  (All
// atoms of the harness share one mask, so the group holds all of them or
// none.)  kLanes lanes share an atom's list and add up at the end.
// On 32,000 atoms the scattering form, one thread per atom with 6 to 9 FP64
// atomics per pair, took 415 (force), 332 (w), 243 (lj) and 171 us (rho);
// the gather takes 33, 29, 37 and 15 us.  Bound by the latency of the
// neighbour records' loads.
constexpr int kLanes = 8;

__device__ __forceinline__ double lanes_sum(double v) {
#pragma unroll
  for (int o = 1; o < kLanes; o <<= 1) v += __shfl_xor(v, o);
  return v;
}

// the local atom whose values atom j carries
__device__ __forceinline__ int owner_of(const AdjStepView& s, int nlocal, int j) {
  return j < nlocal ? j : s.owner[j - nlocal];
}

// -------------------------------------------------------------- lj/cut
// x_b,i += sum_j H(d) (ftb_i - ftb_j), H u = F u + 2 F' (u.d) d
__global__ __launch_bounds__(kBlock) void k_adj_lj(AdjStepView s, AtomsView a, double lj1,
                                                   double lj2, double rc2, AdjBuffers b) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int i = t / kLanes, sub = t % kLanes;
  if (i >= a.nlocal) return;
  const double4 ui = b.ftb[i];
  const double4 pi = s.pv[i].p;
  const int n = s.ljn[i];
  double bx = 0.0, by = 0.0, bz = 0.0;
  for (int k = sub; k < n; k += kLanes) {
    const int j = s.lj[k * a.stride + i];
    const double4 pj = s.pv[j].p;
    const double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (!(r2 < rc2)) continue;
    const double4 uj = b.ftb[owner_of(s, a.nlocal, j)];
    const double ux = ui.x - uj.x, uy = ui.y - uj.y, uz = ui.z - uj.z;
    // F(r^2) = lj1 r^-14 - lj2 r^-8 (the fpair of k_lj), dF/d(r^2)
    const double r2i = 1.0 / r2;
    const double r4i = r2i * r2i, r6i = r4i * r2i, r8i = r4i * r4i;
    const double F = r6i * (lj1 * r6i - lj2) * r2i;
    const double dF = -7.0 * lj1 * r8i * r8i + 4.0 * lj2 * r8i * r2i;
    const double q = 2.0 * dF * (ux * dx + uy * dy + uz * dz);
    bx += F * ux + q * dx;
    by += F * uy + q * dy;
    bz += F * uz + q * dz;
  }
  bx = lanes_sum(bx); by = lanes_sum(by); bz = lanes_sum(bz);
  if (sub != 0) return;
  double4 x = b.xb[i];
  x.x += bx; x.y += by; x.z += bz;
  b.xb[i] = x;
}

// ------------------------------------------------- force sweep (2 + 3)
// f_E,i = -sum_j [B_ij (e.w_i) - B_ji (e.w_j)] e,
// f_R,i = eta sqrt(T_i) sum_j [B_ij (e.xi_i) - B_ji (e.xi_j)] e,
// B_ij = alpha_i rho_{t_j}(r^2) / (rho_i r^2), e = x_j - x_i.

// per atom: uE = dL/df_E, uS = eta sqrt(T) dL/df_R (dL/d of the sum before the
// factor), and T_e's part through the factor
__global__ __launch_bounds__(kBlock) void k_adj_force_in(AdjStepView s, AtomsView a, GridView g,
                                                         StepParams p, int fric, int rnd, int addE,
                                                         int addR, AdjBuffers b) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.nlocal) return;
  double4 uE = make_double4(0, 0, 0, 0), uS = uE;
  if ((a.mask[i] & a.groupbit) && s.rec[i].rw.w > 0.0) {
    const double4 pi = s.rec[i].p;
    const double4 ft = b.ftb[i];
    if (fric) uE = b.fEb[i];
    if (rnd) uS = b.fRb[i];
    if (addE && fric) { uE.x += ft.x; uE.y += ft.y; uE.z += ft.z; }
    if (addR && rnd) { uS.x += ft.x; uS.y += ft.y; uS.z += ft.z; }
    // f_R = eta sqrt(T) S -> S_bar = eta sqrt(T) uR, T_bar += uR.f_R / (2 T)
    if (rnd) {
      const int c = cell_of(g, pi.x, pi.y, pi.z);
      const double Te = g.T[c];
      const double f = p.eta * sqrt(Te);
      const int fs = s.fstride;
      if (Te > 0.0) {
        const double fr = uS.x * s.fR[i] + uS.y * s.fR[fs + i] + uS.z * s.fR[2 * fs + i];
        atomicAdd(b.Tb + c, fr / (2.0 * Te));
      }
      uS.x *= f; uS.y *= f; uS.z *= f;
    }
  }
  b.fEb[i] = uE;
  b.fRb[i] = uS;
}

// Primed quantities are those of the pair (j, i): e' = -e, B1' = B2, B2' = B1,
// a1' = -a2, a2' = -a1, and the same bracket.
__global__ __launch_bounds__(kBlock) void k_adj_force(AdjStepView s, AtomsView a, TablesView t,
                                                      int fric, int rnd, AdjBuffers b) {
  const int th = blockIdx.x * kBlock + threadIdx.x;
  const int i = th / kLanes, sub = th % kLanes;
  if (i >= a.nlocal) return;
  const ForceRec ri = s.rec[i];
  const double rho_i = ri.rw.w;
  const double4 pi = ri.p, wi = ri.rw, xi = ri.xa;
  const double alpha_i = xi.w;
  const double4 uE = b.fEb[i], uS = b.fRb[i];
  const bool multi = t.n_elem > 1;
  const int ei = multi ? static_cast<int>(pi.w) : 0;
  double wbx = 0, wby = 0, wbz = 0, abi = 0, rbi = 0, xbx = 0, xby = 0, xbz = 0;
  const int na = (a.mask[i] & a.groupbit) && rho_i > 0.0 ? s.nact[i] : 0;
  for (int k = sub; k < na; k += kLanes) {
    const int j = s.act[k * a.stride + i];
    const double4 pj = s.rec[j].p, wj = s.rec[j].rw, xj = s.rec[j].xa;
    const int o = owner_of(s, a.nlocal, j);
    const double4 uEj = b.fEb[o], uSj = b.fRb[o];
    const double rho_j = wj.w;
    if (!(rho_j > 0.0)) continue;
    const double alpha_j = xj.w;
    const double ex = pj.x - pi.x, ey = pj.y - pi.y, ez = pj.z - pi.z;
    const double r2 = ex * ex + ey * ey + ez * ez;
    const int ej = multi ? static_cast<int>(pj.w) : 0;
    double vji, dvji, vij, dvij;
    rho_r2_vd(t, ej, r2, &vji, &dvji);
    if (multi) {
      rho_r2_vd(t, ei, r2, &vij, &dvij);
    } else {
      vij = vji;
      dvij = dvji;
    }
    const double qi = 1.0 / (rho_i * r2), qj = 1.0 / (rho_j * r2);
    const double B1 = alpha_i * vji * qi, B2 = alpha_j * vij * qj;
    double b1 = 0, b2 = 0;             // d/dB1, d/dB2 of both pairs
    double gx = 0, gy = 0, gz = 0;     // d/de - d/de'
    if (fric) {
      const double a1 = ex * wi.x + ey * wi.y + ez * wi.z;
      const double a2 = ex * wj.x + ey * wj.y + ez * wj.z;
      const double sc = -(B1 * a1 - B2 * a2);
      const double ds = (uE.x - uEj.x) * ex + (uE.y - uEj.y) * ey + (uE.z - uEj.z) * ez;
      gx += sc * (uE.x - uEj.x); gy += sc * (uE.y - uEj.y); gz += sc * (uE.z - uEj.z);
      b1 -= ds * a1;
      b2 += ds * a2;
      const double v1 = -ds * B1, v2 = ds * B2;
      wbx += v1 * ex; wby += v1 * ey; wbz += v1 * ez;
      gx += v1 * wi.x + v2 * wj.x;
      gy += v1 * wi.y + v2 * wj.y;
      gz += v1 * wi.z + v2 * wj.z;
    }
    if (rnd) {
      const double a1 = ex * xi.x + ey * xi.y + ez * xi.z;
      const double a2 = ex * xj.x + ey * xj.y + ez * xj.z;
      const double sc = B1 * a1 - B2 * a2;
      const double ds = (uS.x - uSj.x) * ex + (uS.y - uSj.y) * ey + (uS.z - uSj.z) * ez;
      gx += sc * (uS.x - uSj.x); gy += sc * (uS.y - uSj.y); gz += sc * (uS.z - uSj.z);
      b1 += ds * a1;
      b2 -= ds * a2;
      const double v1 = ds * B1, v2 = -ds * B2;
      gx += v1 * xi.x + v2 * xj.x;
      gy += v1 * xi.y + v2 * xj.y;
      gz += v1 * xi.z + v2 * xj.z;
    }
    // B1 = alpha_i v_ji / (rho_i r2), B2 = alpha_j v_ij / (rho_j r2)
    abi += b1 * vji * qi;
    rbi -= b1 * B1 / rho_i;
    const double r2b = (b1 * alpha_i * (dvji * r2 - vji) * qi + b2 * alpha_j * (dvij * r2 - vij) * qj) / r2;
    xbx -= gx + 2.0 * r2b * ex;
    xby -= gy + 2.0 * r2b * ey;
    xbz -= gz + 2.0 * r2b * ez;
  }
  wbx = lanes_sum(wbx); wby = lanes_sum(wby); wbz = lanes_sum(wbz);
  abi = lanes_sum(abi); rbi = lanes_sum(rbi);
  xbx = lanes_sum(xbx); xby = lanes_sum(xby); xbz = lanes_sum(xbz);
  if (sub != 0) return;
  b.wb[i] = make_double4(wbx, wby, wbz, 0.0);
  b.ab[i] = abi;
  b.rb[i] = rbi;
  double4 x = b.xb[i];
  x.x += xbx; x.y += xby; x.z += xbz;
  b.xb[i] = x;
}

// --------------------------------------------------- w sweep (stage 1)
// w_i = sum_j B_ij (e.vh_i - e.vh_j) e over the active list (no rho_j test)
__global__ __launch_bounds__(kBlock) void k_adj_w(AdjStepView s, AtomsView a, TablesView t,
                                                  AdjBuffers b) {
  const int th = blockIdx.x * kBlock + threadIdx.x;
  const int i = th / kLanes, sub = th % kLanes;
  if (i >= a.nlocal || !(a.mask[i] & a.groupbit)) return;
  const double rho_i = s.rec[i].rw.w, alpha_i = s.rec[i].xa.w;
  const double4 W = b.wb[i];
  const double4 pi = s.pv[i].p, vi = s.pv[i].v;
  const bool multi = t.n_elem > 1;
  const int ei = multi ? static_cast<int>(pi.w) : 0;
  double vbx = 0, vby = 0, vbz = 0, abi = 0, rbi = 0, xbx = 0, xby = 0, xbz = 0;
  const int na = s.nact[i];
  for (int k = sub; k < na; k += kLanes) {
    const int j = s.act[k * a.stride + i];
    const double4 pj = s.pv[j].p, vj = s.pv[j].v;
    const double rho_j = s.rec[j].rw.w, alpha_j = s.rec[j].xa.w;
    const double4 Wj = b.wb[owner_of(s, a.nlocal, j)];
    const double ex = pj.x - pi.x, ey = pj.y - pi.y, ez = pj.z - pi.z;
    const double r2 = ex * ex + ey * ey + ez * ez;
    const int ej = multi ? static_cast<int>(pj.w) : 0;
    const double ux = vi.x - vj.x, uy = vi.y - vj.y, uz = vi.z - vj.z;
    const double dc = ex * ux + ey * uy + ez * uz;
    double vji, dvji, vij, dvij;
    rho_r2_vd(t, ej, r2, &vji, &dvji);
    if (multi) {
      rho_r2_vd(t, ei, r2, &vij, &dvij);
    } else {
      vij = vji;
      dvij = dvji;
    }
    double gx = 0, gy = 0, gz = 0, r2b = 0, vb = 0;
    if (rho_i > 0.0) {  // (i, j)
      const double q = 1.0 / (rho_i * r2);
      const double B = alpha_i * vji * q;
      const double sb = W.x * ex + W.y * ey + W.z * ez;
      gx += B * dc * W.x; gy += B * dc * W.y; gz += B * dc * W.z;
      vb += sb * B;
      const double Bb = sb * dc;
      abi += Bb * vji * q;
      rbi -= Bb * B / rho_i;
      r2b += Bb * alpha_i * (dvji * r2 - vji) * q / r2;
    }
    if (rho_j > 0.0) {  // (j, i)
      const double q = 1.0 / (rho_j * r2);
      const double B = alpha_j * vij * q;
      const double sb = Wj.x * ex + Wj.y * ey + Wj.z * ez;
      gx -= B * dc * Wj.x; gy -= B * dc * Wj.y; gz -= B * dc * Wj.z;
      vb -= sb * B;
      r2b -= sb * dc * alpha_j * (dvij * r2 - vij) * q / r2;
    }
    vbx += vb * ex; vby += vb * ey; vbz += vb * ez;
    xbx -= gx + vb * ux + 2.0 * r2b * ex;
    xby -= gy + vb * uy + 2.0 * r2b * ey;
    xbz -= gz + vb * uz + 2.0 * r2b * ez;
  }
  vbx = lanes_sum(vbx); vby = lanes_sum(vby); vbz = lanes_sum(vbz);
  abi = lanes_sum(abi); rbi = lanes_sum(rbi);
  xbx = lanes_sum(xbx); xby = lanes_sum(xby); xbz = lanes_sum(xbz);
  if (sub != 0) return;
  double4 v = b.vhb[i];
  v.x += vbx; v.y += vby; v.z += vbz;
  b.vhb[i] = v;
  b.ab[i] += abi;
  b.rb[i] += rbi;
  double4 x = b.xb[i];
  x.x += xbx; x.y += xby; x.z += xbz;
  b.xb[i] = x;
}

// ------------------------------------------------------------ alpha(rho)
// alpha_i = a + rho (b + rho (c + rho d)) on the interval of rho_i: rho_b +=
// alpha_b alpha', table gradient Gb[e][k] += alpha_b (1, rho, rho^2, rho^3).
// The atoms of a crystal mostly sit on one or two knots, and an atomic on an
// address that all blocks share takes some 50 ns: 32,000 atoms took 27 us with
// one per knot and wave (1.5 ms with one per atom).

// rho_b and the four terms of atom i; its knot, -1 for none
__device__ __forceinline__ int adj_alpha_atom(const int i, const AdjStepView& s, const AtomsView& a,
                                              const TablesView& t, const AdjBuffers& b, double* g) {
  if (i >= a.nlocal || !(a.mask[i] & a.groupbit)) return -1;
  const double rho = s.rec[i].rw.w, ab = b.ab[i];
  if (!(rho > 0.0) || rho > t.rho_cut || ab == 0.0) return -1;
  const int e = t.n_elem > 1 ? static_cast<int>(s.rec[i].p.w) : 0;
  int k = static_cast<int>(rho * t.inv_drho);
  k = k < 0 ? 0 : (k < t.n_beta - 1 ? k : t.n_beta - 1);
  const int key = e * t.n_beta + k;
  const double4 c = t.alpha[key];
  b.rb[i] += ab * (c.y + rho * (2.0 * c.z + 3.0 * rho * c.w));
  g[0] = ab; g[1] = ab * rho; g[2] = ab * rho * rho; g[3] = ab * rho * rho * rho;
  return key;
}

// Tables whose gradient fits the LDS (9 us for those atoms): a few large blocks sum it there
// and add each touched coefficient once.
constexpr int kAlphaThreads = 1024, kAlphaBlocks = 32;
constexpr size_t kAlphaLds = 64 * 1024;
__global__ __launch_bounds__(kAlphaThreads) void k_adj_alpha_lds(AdjStepView s, AtomsView a, TablesView t,
                                                                 AdjBuffers b, int ncoef) {
  extern __shared__ double s_g[];
  for (int q = threadIdx.x; q < ncoef; q += kAlphaThreads) s_g[q] = 0.0;
  __syncthreads();
  for (int i = blockIdx.x * kAlphaThreads + threadIdx.x; i < a.nlocal; i += gridDim.x * kAlphaThreads) {
    double g[4];
    const int key = adj_alpha_atom(i, s, a, t, b, g);
    if (key >= 0)
      for (int q = 0; q < 4; ++q) atomicAdd(s_g + 4 * key + q, g[q]);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < ncoef; q += kAlphaThreads)
    if (s_g[q] != 0.0) atomicAdd(b.Gb + q, s_g[q]);
}

// any table: summed over the wave per distinct knot, all lanes taking part
__global__ __launch_bounds__(kBlock) void k_adj_alpha(AdjStepView s, AtomsView a, TablesView t,
                                                      AdjBuffers b) {
  double g[4] = {0.0, 0.0, 0.0, 0.0};
  const int key = adj_alpha_atom(blockIdx.x * kBlock + threadIdx.x, s, a, t, b, g);
  const int lane = static_cast<int>(threadIdx.x) & (warpSize - 1);
  unsigned long long left = __ballot(key >= 0);
  while (left) {
    const int lead = __ffsll(static_cast<long long>(left)) - 1;
    const int k0 = __shfl(key, lead);
    const bool mine = key == k0;
    double s0 = mine ? g[0] : 0.0, s1 = mine ? g[1] : 0.0, s2 = mine ? g[2] : 0.0, s3 = mine ? g[3] : 0.0;
    for (int off = warpSize / 2; off > 0; off >>= 1) {
      s0 += __shfl_xor(s0, off);
      s1 += __shfl_xor(s1, off);
      s2 += __shfl_xor(s2, off);
      s3 += __shfl_xor(s3, off);
    }
    if (lane == lead) {
      double* G = b.Gb + 4 * static_cast<long>(k0);
      atomicAdd(G + 0, s0);
      atomicAdd(G + 1, s1);
      atomicAdd(G + 2, s2);
      atomicAdd(G + 3, s3);
    }
    left &= ~__ballot(mine);
  }
}

// ------------------------------------------------------- density sweep
// rho_i = sum_j rho_{t_j}(r^2) over the active list
__global__ __launch_bounds__(kBlock) void k_adj_rho(AdjStepView s, AtomsView a, TablesView t,
                                                    AdjBuffers b) {
  const int th = blockIdx.x * kBlock + threadIdx.x;
  const int i = th / kLanes, sub = th % kLanes;
  if (i >= a.nlocal || !(a.mask[i] & a.groupbit)) return;
  const double rb = b.rb[i];
  const double4 pi = s.rec[i].p;
  const bool multi = t.n_elem > 1;
  const int ei = multi ? static_cast<int>(pi.w) : 0;
  double xbx = 0, xby = 0, xbz = 0;
  const int na = s.nact[i];
  for (int k = sub; k < na; k += kLanes) {
    const int j = s.act[k * a.stride + i];
    const double4 pj = s.rec[j].p;
    const double rbj = b.rb[owner_of(s, a.nlocal, j)];
    const double ex = pj.x - pi.x, ey = pj.y - pi.y, ez = pj.z - pi.z;
    const double r2 = ex * ex + ey * ey + ez * ez;
    double v, dvj, dvi;
    rho_r2_vd(t, multi ? static_cast<int>(pj.w) : 0, r2, &v, &dvj);
    if (multi) rho_r2_vd(t, ei, r2, &v, &dvi);
    else dvi = dvj;
    const double q = 2.0 * (rb * dvj + rbj * dvi);
    xbx -= q * ex; xby -= q * ey; xbz -= q * ez;
  }
  xbx = lanes_sum(xbx); xby = lanes_sum(xby); xbz = lanes_sum(xbz);
  if (sub != 0) return;
  double4 x = b.xb[i];
  x.x += xbx; x.y += xby; x.z += xbz;
  b.xb[i] = x;
}

// ---------------------------------------------------- initial integrate
// vh = v + (dtf / m) f_prev, x' = x + dtv vh  (group atoms)
__global__ __launch_bounds__(kBlock) void k_adj_initial(AtomsView a, StepParams p, int noint,
                                                        AdjBuffers b) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.nlocal) return;
  const double4 xb = b.xb[i];
  double4 vh = b.vhb[i];
  double4 ft = make_double4(0, 0, 0, 0);
  if (!noint && (a.mask[i] & a.groupbit)) {
    vh.x += p.dtv * xb.x; vh.y += p.dtv * xb.y; vh.z += p.dtv * xb.z;
    const double c = p.dtf / p.mass[a.type[i]];
    ft = make_double4(c * vh.x, c * vh.y, c * vh.z, 0.0);
  }
  // the previous step's v' and total force
  b.vnb[i] = make_double4(vh.x, vh.y, vh.z, 0.0);
  b.ftb[i] = ft;
  b.vhb[i] = make_double4(0, 0, 0, 0);
}

// ------------------------------------------------------------ wrappers
hipError_t launch_adj_fdm(const GridView& g, const double* Tin, const double* Tb_out, double* Tb_in,
                          double* dTb, double* kb, double inner_dt, hipStream_t s) {
  const int G = g.nx * g.ny * g.nz;
  if (kb) k_adj_fdm<true><<<nblk(G), kBlock, 0, s>>>(g, Tin, Tb_out, Tb_in, dTb, kb, inner_dt, G);
  else k_adj_fdm<false><<<nblk(G), kBlock, 0, s>>>(g, Tin, Tb_out, Tb_in, dTb, nullptr, inner_dt, G);
  return hipGetLastError();
}

hipError_t launch_adj_kappa_T(const GridView& g, const double* T0, const double* kb, double* Tb,
                              hipStream_t s) {
  const int G = g.nx * g.ny * g.nz;
  k_adj_kappa_T<<<nblk(G), kBlock, 0, s>>>(g, T0, kb, Tb, G);
  return hipGetLastError();
}

hipError_t launch_adj_step(const AdjStepView& sv, const AtomsView& a, const TablesView& t,
                           const GridView& g, const StepParams& p, const AdjStepFlags& f,
                           const double* dTb, const AdjBuffers& b, hipStream_t s) {
  const int nl = a.nlocal;
  if (nl == 0) return hipSuccess;
  const int nb = nblk(nl), nbl = nblk(static_cast<long>(nl) * kLanes);
  if (f.fric || f.rnd)
    k_adj_deposit<<<nb, kBlock, 0, s>>>(sv, g, a, p.dt, f.fric, f.rnd, 1.0, dTb, b);
  k_adj_final<<<nb, kBlock, 0, s>>>(a, p, f.noint, b);
  k_adj_lj<<<nbl, kBlock, 0, s>>>(sv, a, f.lj1, f.lj2, f.ljrc2, b);
  if (f.model4 && (f.fric || f.rnd)) {
    k_adj_force_in<<<nb, kBlock, 0, s>>>(sv, a, g, p, f.fric, f.rnd, f.addE, f.addR, b);
    k_adj_force<<<nbl, kBlock, 0, s>>>(sv, a, t, f.fric, f.rnd, b);
  }
  if (f.fric) k_adj_w<<<nbl, kBlock, 0, s>>>(sv, a, t, b);
  const int ncoef = 4 * t.n_elem * t.n_beta;
  if (ncoef * sizeof(double) <= kAlphaLds) {
    const int blocks = static_cast<int>((a.nlocal + kAlphaThreads - 1l) / kAlphaThreads);
    k_adj_alpha_lds<<<blocks < kAlphaBlocks ? blocks : kAlphaBlocks, kAlphaThreads, ncoef * sizeof(double), s>>>(
        sv, a, t, b, ncoef);
  } else {
    k_adj_alpha<<<nb, kBlock, 0, s>>>(sv, a, t, b);
  }
  k_adj_rho<<<nbl, kBlock, 0, s>>>(sv, a, t, b);
  k_adj_initial<<<nb, kBlock, 0, s>>>(a, p, f.noint, b);
  return hipGetLastError();
}

}  // namespace eph
