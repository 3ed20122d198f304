// lp_adjoint.hpp -- kernels of the discrete adjoint of the frozen-coefficient step
// (main.f90:252-826 with Nu_t and the wall u* of a base run held fixed), binary64.
// Each kernel is the transpose of a forward kernel, written as a gather (every output
// point sums the contributions that reach it), so no atomics are needed.  Levels k are
// 0-based (Fortran jz = k+1); only the physical columns x < nx carry adjoint values.
#pragma once
#include "lp_droplets.hpp"
#include "lp_kernels.hpp"

namespace lp {

struct AdjGeo {
  int nx, ny, nz, ld;
  long np;
};

__device__ __forceinline__ bool adj_phys(const AdjGeo &g, long i, int &k, int &x) {
  k = (int)(i / g.np);
  x = (int)(i % g.ld);
  return x < g.nx;
}

// forcing.f90:145-292 (velocity correction, boundary values) and main.f90:795-803
// (RHS -= grad p), transposed.  au/av/aw: adjoint of the step's u, v, w; rb*: adjoint of
// the RHS it leaves.  Writes the adjoints of u* (us), of dpdx/dpdy/dpdz (ap*), of the
// RHS before the pressure gradient (ar*), and of filt_da's u, v at the top level (af*:
// the top level of u, v is filt_da's value unless the mean forcing copies it).
__global__ void k_adj_project(const double *__restrict__ au, const double *__restrict__ av,
                              const double *__restrict__ aw, const double *__restrict__ rbx,
                              const double *__restrict__ rby, const double *__restrict__ rbz,
                              double *__restrict__ usx, double *__restrict__ usy, double *__restrict__ usz,
                              double *__restrict__ apx, double *__restrict__ apy, double *__restrict__ apz,
                              double *__restrict__ arx, double *__restrict__ ary, double *__restrict__ arz,
                              double *__restrict__ afu, double *__restrict__ afv, AdjGeo g, double dt,
                              int mean_force, int stress_free) {
  const long i = gtid();
  if (i >= g.np * g.nz) return;
  int k, x;
  const bool ph = adj_phys(g, i, k, x);
  const long r = i - (long)k * g.np;
  // boundary values: u(top) = u(top-1) with the mean forcing, u(0) = u(1) stress-free
  auto bc = [&](const double *a, long j, int kk) -> double {
    double v = a[j];
    if (kk == g.nz - 1) return 0.0;  // the top level is not a velocity the correction writes
    if (mean_force && kk == g.nz - 2) v += a[(long)(g.nz - 1) * g.np + r];
    if (stress_free && kk == 0) v = 0.0;
    if (stress_free && kk == 1) v += a[r];
    return v;
  };
  double ux = 0, uy = 0, uz = 0, px = 0, py = 0, pz = 0, rx = 0, ry = 0, rz = 0, fu = 0, fv = 0;
  if (ph && k <= g.nz - 2) {
    const double a_u = bc(au, i, k), a_v = bc(av, i, k);
    const double a_w = (k >= 1) ? aw[i] : 0.0;  // w(0) = 0 is a boundary value
    ux = a_u; uy = a_v; uz = a_w;
    px = -1.5 * dt * a_u - rbx[i];
    py = -1.5 * dt * a_v - rby[i];
    pz = -1.5 * dt * a_w - rbz[i];
    rx = rbx[i]; ry = rby[i]; rz = rbz[i];
  }
  if (ph && k == g.nz - 1 && !mean_force) { fu = au[i]; fv = av[i]; }
  usx[i] = ux; usy[i] = uy; usz[i] = uz;
  apx[i] = px; apy[i] = py; apz[i] = pz;
  arx[i] = rx; ary[i] = ry; arz[i] = rz;
  afu[i] = fu; afv[i] = fv;
}

// dpdz = (p(k+1) - p(k))/dz on levels 0..nz-2 (main.f90:789-791), transposed: the
// adjoint of p on planes 0..nz-1 (plane nz of p is not an output)
__global__ void k_adj_dpdz(const double *__restrict__ apz, double *__restrict__ ap, AdjGeo g, double idz) {
  const long i = gtid();
  if (i >= g.np * g.nz) return;
  int k, x;
  double v = 0.0;
  if (adj_phys(g, i, k, x)) {
    if (k >= 1) v += apz[i - g.np] * idz;
    if (k <= g.nz - 2) v -= apz[i] * idz;
  }
  ap[i] = v;
}

// forward intermediates of the adjoint's base state: the wall-level dudz, dvdz of the
// wall law (u / (zl denom), wallstress.f90:176-183 with the frozen u*) and the vorticity
// of convec.f90:100-133 (jz = 1 on the uvp node)
__global__ void k_adj_base(const double *__restrict__ uf, const double *__restrict__ vf,
                           const double *__restrict__ uz, const double *__restrict__ vz, const double *__restrict__ uy, const double *__restrict__ vx,
                           const double *__restrict__ wx, const double *__restrict__ wy, double *__restrict__ om1,
                           double *__restrict__ om2, double *__restrict__ om3, AdjGeo g, double wfac, int wall) {
  const long i = gtid();
  if (i >= g.np * g.nz) return;
  int k, x;
  if (!adj_phys(g, i, k, x)) { om1[i] = 0; om2[i] = 0; om3[i] = 0; return; }
  const double a_uz = k == 0 ? (wall ? uf[i] * wfac : 0.0) : uz[i];
  const double a_vz = k == 0 ? (wall ? vf[i] * wfac : 0.0) : vz[i];
  const long up = (k == 0) ? g.np : 0;
  const double wyv = k == 0 ? 0.5 * (wy[i] + wy[i + up]) : wy[i];
  const double wxv = k == 0 ? 0.5 * (wx[i] + wx[i + up]) : wx[i];
  om1[i] = wyv - a_vz;
  om2[i] = a_uz - wxv;
  om3[i] = vx[i] - uy[i];
}

// the AB2 predictor (main.f90:716-728), the RHS assembly (:433-439) and the Euler start
// (:577-584), transposed, together with the pressure's contributions: us* (projection)
// + h* (H back-transformed) is the adjoint of u*; wall / lid rows (bwb, twb planes) go to
// divtz.  Outputs the adjoints of filt_da's u, v, w (af*, initialised here), of the
// convective terms (ac*), of the stress divergences (ad*) and of RHS_f (rb*, in place).
__global__ void k_adj_ab2(const double *__restrict__ usx, const double *__restrict__ usy,
                          const double *__restrict__ usz, const double *__restrict__ hx, const double *__restrict__ hy,
                          const double *__restrict__ hz, const double *__restrict__ arx,
                          const double *__restrict__ ary, const double *__restrict__ arz,
                          const double *__restrict__ afu_top, const double *__restrict__ afv_top,
                          const double *__restrict__ bwb, const double *__restrict__ twb, double *__restrict__ afu,
                          double *__restrict__ afv, double *__restrict__ afw, double *__restrict__ acx,
                          double *__restrict__ acy, double *__restrict__ acz, double *__restrict__ adx,
                          double *__restrict__ ady, double *__restrict__ adz, double *__restrict__ rbx,
                          double *__restrict__ rby, double *__restrict__ rbz, AdjGeo g, double dt, int first) {
  const long i = gtid();
  if (i >= g.np * g.nz) return;
  int k, x;
  const bool ph = adj_phys(g, i, k, x);
  const long r = i - (long)k * g.np;
  double fu = 0, fv = 0, fw = 0, cx_ = 0, cy_ = 0, cz_ = 0, dx_ = 0, dy_ = 0, dz_ = 0, ox = 0, oy = 0, oz = 0;
  if (ph && k <= g.nz - 2) {
    const double sx = usx[i] + hx[i], sy = usy[i] + hy[i], sz = usz[i] + hz[i];
    const double tr = first ? 1.0 : 1.5;
    fu = sx; fv = sy; fw = sz;
    const double rx = arx[i] + tr * dt * sx, ry = ary[i] + tr * dt * sy, rz = arz[i] + tr * dt * sz;
    ox = first ? 0.0 : -0.5 * dt * sx;
    oy = first ? 0.0 : -0.5 * dt * sy;
    oz = first ? 0.0 : -0.5 * dt * sz;
    cx_ = -rx; dx_ = -rx;
    cy_ = -ry; dy_ = -ry;
    cz_ = k >= 1 ? -rz : 0.0;
    dz_ = -rz;
  }
  if (ph && k == 0) dz_ += bwb[r];
  if (ph && k == g.nz - 1) {
    dz_ += twb[r];
    fu = afu_top[i];
    fv = afv_top[i];
  }
  afu[i] = fu; afv[i] = fv; afw[i] = fw;
  acx[i] = cx_; acy[i] = cy_; acz[i] = cz_;
  adx[i] = dx_; ady[i] = dy_; adz[i] = dz_;
  rbx[i] = ox; rby[i] = oy; rbz[i] = oz;
}

// convec.f90:138-279 products on the 3/2 grid, transposed (gather over the levels whose
// products read level k).  p*: adjoint of the products (times the truncation's transpose
// scale tt); U, O: base velocities and vorticity on the 3/2 grid (nz levels, npb points).
__global__ void k_adj_products(const double *__restrict__ px, const double *__restrict__ py,
                               const double *__restrict__ pz, const double *__restrict__ U1,
                               const double *__restrict__ U2, const double *__restrict__ U3,
                               const double *__restrict__ O1, const double *__restrict__ O2,
                               const double *__restrict__ O3, double *__restrict__ aU1, double *__restrict__ aU2,
                               double *__restrict__ aU3, double *__restrict__ aO1, double *__restrict__ aO2,
                               double *__restrict__ aO3, long npb, int nz, double tt) {
  const long a = gtid();
  if (a >= npb * nz) return;
  const int k = (int)(a / npb);
  const long m = a - npb, b = a + npb;
  auto P = [&](const double *p, long j, int kk, int lo) -> double {  // tt p(kk), kk in lo..nz-2
    return (kk >= lo && kk <= nz - 2) ? tt * p[j] : 0.0;
  };
  const double pxk = P(px, a, k, 0), pyk = P(py, a, k, 0), pzk = P(pz, a, k, 1);
  const double pxm = P(px, m, k - 1, 0), pym = P(py, m, k - 1, 0);
  const double pzp = P(pz, b, k + 1, 1);
  const double u1 = U1[a], u2 = U2[a], u3 = U3[a], o1 = O1[a], o2 = O2[a], o3 = O3[a];
  const double u1m = k >= 1 ? U1[m] : 0.0, u2m = k >= 1 ? U2[m] : 0.0;
  const double o1p = k + 1 <= nz - 1 ? O1[b] : 0.0, o2p = k + 1 <= nz - 1 ? O2[b] : 0.0;
  const bool in = k >= 1;  // the [k >= 1] terms of px, py at level k
  aU1[a] = o3 * pyk - 0.5 * o2 * pzk - 0.5 * o2p * pzp;
  aU2[a] = -o3 * pxk + 0.5 * o1 * pzk + 0.5 * o1p * pzp;
  aU3[a] = 0.5 * o2 * pxm + (in ? 0.5 * o2 * pxk : 0.0) - 0.5 * o1 * pym - (in ? 0.5 * o1 * pyk : 0.0);
  aO1[a] = -0.5 * u3 * pym - (in ? 0.5 * u3 * pyk : 0.0) + 0.5 * (u2 + u2m) * pzk;
  aO2[a] = 0.5 * u3 * pxm + (in ? 0.5 * u3 * pxk : 0.0) - 0.5 * (u1 + u1m) * pzk;
  aO3[a] = -u2 * pxk + u1 * pyk;
}

// divstress_uv / divstress_w (z parts) and the stresses with the frozen Nu_t
// (sgs_stag.f90:254-325), transposed: the adjoints of S11..S33 from the adjoints of the
// divergences (ad*) and of their x / y derivative parts (d*: Dx ad, Dy ad, already
// computed; the derivatives are antisymmetric so they enter with a minus sign).
// qw: the wall-law coefficient times the adjoint of txz(1), tyz(1) is written to
// wtx / wty (plane) for the test filter.
__global__ void k_adj_tau(const double *__restrict__ adx, const double *__restrict__ ady,
                          const double *__restrict__ adz, const double *__restrict__ dxa,
                          const double *__restrict__ dya, const double *__restrict__ dxb,
                          const double *__restrict__ dyb, const double *__restrict__ dxc,
                          const double *__restrict__ dyc, const double *__restrict__ nut,
                          const double *__restrict__ ust, double *__restrict__ aS11, double *__restrict__ aS12,
                          double *__restrict__ aS13, double *__restrict__ aS22, double *__restrict__ aS23,
                          double *__restrict__ aS33, double *__restrict__ wtx, double *__restrict__ wty, AdjGeo g,
                          double idz, double qfac, int wall) {
  const long i = gtid();
  if (i >= g.np * g.nz) return;
  int k, x;
  if (!adj_phys(g, i, k, x)) {
    aS11[i] = 0; aS12[i] = 0; aS13[i] = 0; aS22[i] = 0; aS23[i] = 0; aS33[i] = 0;
    return;
  }
  const int nz = g.nz;
  const long np = g.np;
  // adjoints of the stresses at level kk (this column)
  auto atxx = [&](int kk) { return -dxa[i + (long)(kk - k) * np]; };
  auto atxy = [&](int kk) { const long j = i + (long)(kk - k) * np; return -dya[j] - dxb[j]; };
  auto atyy = [&](int kk) { return -dyb[i + (long)(kk - k) * np]; };
  auto atxz = [&](int kk) {
    const long j = i + (long)(kk - k) * np;
    double v = -dxc[j];
    if (kk - 1 >= 0 && kk - 1 <= nz - 2) v += adx[j - np] * idz;
    if (kk <= nz - 2) v -= adx[j] * idz;
    return v;
  };
  auto atyz = [&](int kk) {
    const long j = i + (long)(kk - k) * np;
    double v = -dyc[j];
    if (kk - 1 >= 0 && kk - 1 <= nz - 2) v += ady[j - np] * idz;
    if (kk <= nz - 2) v -= ady[j] * idz;
    return v;
  };
  auto atzz = [&](int kk) {
    const long j = i + (long)(kk - k) * np;
    double v = 0.0;
    if (kk >= 1 && kk <= nz - 2) v += adz[j] * idz;
    if (kk + 1 >= 1 && kk + 1 <= nz - 2) v -= adz[j + np] * idz;
    return v;
  };
  auto cc = [&](int kk) { const long j = i + (long)(kk - k) * np; return 0.5 * (nut[j] + nut[j + np]); };
  double s11 = 0, s12 = 0, s13 = 0, s22 = 0, s23 = 0, s33 = 0;
  if (k == 0) {
    const double n0 = nut[i];
    s11 = -2.0 * n0 * atxx(0); s12 = -2.0 * n0 * atxy(0); s22 = -2.0 * n0 * atyy(0); s33 = -2.0 * n0 * atzz(0);
    if (wall) {  // txz(1) = q G(u(1)), q = -u* kappa / denom (frozen)
      wtx[i] = -ust[i] * qfac * atxz(0);
      wty[i] = -ust[i] * qfac * atyz(0);
    }
  } else {
    if (k <= nz - 2) {
      const double c0 = cc(k);
      s11 = -c0 * atxx(k); s12 = -c0 * atxy(k); s22 = -c0 * atyy(k); s33 = -c0 * atzz(k);
      s13 = -2.0 * nut[i] * atxz(k);
      s23 = -2.0 * nut[i] * atyz(k);
    }
    if (k - 1 >= 1 && k - 1 <= nz - 2) {
      const double c1 = cc(k - 1);
      s11 += -c1 * atxx(k - 1); s12 += -c1 * atxy(k - 1); s22 += -c1 * atyy(k - 1); s33 += -c1 * atzz(k - 1);
    }
  }
  aS11[i] = s11; aS12[i] = s12; aS13[i] = s13; aS22[i] = s22; aS23[i] = s23; aS33[i] = s33;
}

// the strain rates (sgs_stag.f90:49-125), the vorticity (convec.f90:100-133) and the z
// derivatives (ddz_uv, ddz_w, the wall law's dudz) transposed: the adjoints of filt_da's
// u, v, w gain the z-derivative parts here (af*, in place), and those of the x and y
// derivatives are written (a*x, a*y).  ao*: adjoint of the vorticity.
__global__ void k_adj_strain(const double *__restrict__ aS11, const double *__restrict__ aS12,
                             const double *__restrict__ aS13, const double *__restrict__ aS22,
                             const double *__restrict__ aS23, const double *__restrict__ aS33,
                             const double *__restrict__ ao1, const double *__restrict__ ao2,
                             const double *__restrict__ ao3, double *__restrict__ aux, double *__restrict__ auy,
                             double *__restrict__ avx, double *__restrict__ avy, double *__restrict__ awx,
                             double *__restrict__ awy, double *__restrict__ afu, double *__restrict__ afv,
                             double *__restrict__ afw, AdjGeo g, double idz, double wfac, int wall) {
  const long i = gtid();
  if (i >= g.np * g.nz) return;
  int k, x;
  if (!adj_phys(g, i, k, x)) {
    aux[i] = 0; auy[i] = 0; avx[i] = 0; avy[i] = 0; awx[i] = 0; awy[i] = 0;
    return;
  }
  const int nz = g.nz;
  const long np = g.np, r = i - (long)k * np;
  auto at = [&](const double *a, int kk) { return a[r + (long)kk * np]; };
  const bool hasp = k + 1 <= nz - 1;
  // x and y derivatives
  aux[i] = (k == 0 ? at(aS11, 0) : 0.5 * at(aS11, k)) + (hasp ? 0.5 * at(aS11, k + 1) : 0.0);
  const double s12 = (k == 0 ? 0.5 * at(aS12, 0) : 0.25 * at(aS12, k)) + (hasp ? 0.25 * at(aS12, k + 1) : 0.0);
  auy[i] = s12 - at(ao3, k);
  avx[i] = s12 + at(ao3, k);
  avy[i] = (k == 0 ? at(aS22, 0) : 0.5 * at(aS22, k)) + (hasp ? 0.5 * at(aS22, k + 1) : 0.0);
  awx[i] = (k <= 1 ? 0.25 * at(aS13, 0) - 0.5 * at(ao2, 0) : 0.0) + (k >= 1 ? 0.5 * at(aS13, k) - at(ao2, k) : 0.0);
  awy[i] = (k <= 1 ? 0.25 * at(aS23, 0) + 0.5 * at(ao1, 0) : 0.0) + (k >= 1 ? 0.5 * at(aS23, k) + at(ao1, k) : 0.0);
  // z derivatives: auz, avz at level kk; awz at level kk
  auto auz = [&](int kk) { return (kk == 0 ? 0.5 * at(aS13, 0) : 0.5 * at(aS13, kk)) + at(ao2, kk); };
  auto avz = [&](int kk) { return (kk == 0 ? 0.5 * at(aS23, 0) : 0.5 * at(aS23, kk)) - at(ao1, kk); };
  auto awz = [&](int kk) {
    return (kk == 0 ? at(aS33, 0) : 0.5 * at(aS33, kk)) + (kk + 1 <= nz - 1 ? 0.5 * at(aS33, kk + 1) : 0.0);
  };
  double fu = afu[i], fv = afv[i], fw = afw[i];
  // dudz(k) = (u(k) - u(k-1))/dz on 1..nz-2; dudz(0) = u(0) wfac (wall law)
  if (k >= 1 && k <= nz - 2) { fu += auz(k) * idz; fv += avz(k) * idz; }
  if (k + 1 >= 1 && k + 1 <= nz - 2) { fu -= auz(k + 1) * idz; fv -= avz(k + 1) * idz; }
  if (k == 0 && wall) { fu += auz(0) * wfac; fv += avz(0) * wfac; }
  // dwdz(k) = (w(k+1) - w(k))/dz on 0..nz-2
  if (k >= 1) fw += awz(k - 1) * idz;
  if (k <= nz - 2) fw -= awz(k) * idz;
  afu[i] = fu; afv[i] = fv; afw[i] = fw;
}

// out = a - b - c on the physical columns, zero on the padding (filt_da transposed:
// F(af) - Dx(ax) - Dy(ay)); with wall plane add: af(0) += gw before (the wall-law term)
__global__ void k_adj_combine(double *__restrict__ out, const double *__restrict__ fu, const double *__restrict__ fv,
                              const double *__restrict__ fw, const double *__restrict__ ux,
                              const double *__restrict__ vx, const double *__restrict__ wx,
                              const double *__restrict__ uy, const double *__restrict__ vy,
                              const double *__restrict__ wy, long nv, AdjGeo g) {
  const long i = gtid();
  if (i >= g.np * g.nz) return;
  const int q = blockIdx.y;
  const double *a = q == 0 ? fu : q == 1 ? fv : fw, *b = q == 0 ? ux : q == 1 ? vx : wx;
  const double *c = q == 0 ? uy : q == 1 ? vy : wy;
  int k, x;
  out[q * nv + i] = adj_phys(g, i, k, x) ? a[i] - b[i] - c[i] : 0.0;
}

// a0 += b0, a1 += b1, a2 += b2 (blockIdx.y)
__global__ void k_add_plane3(double *__restrict__ a0, double *__restrict__ a1, double *__restrict__ a2,
                             const double *__restrict__ b0, const double *__restrict__ b1,
                             const double *__restrict__ b2, long n) {
  const long i = gtid();
  if (i >= n) return;
  const int q = blockIdx.y;
  double *a = q == 0 ? a0 : q == 1 ? a1 : a2;
  a[i] += (q == 0 ? b0 : q == 1 ? b1 : b2)[i];
}

}  // namespace lp

namespace lp {

// wallstress.f90:101-185 with the wall u* of a base run (frozen coefficient):
// txz = -(u*^2/|U|) u1 = -(u* kappa/denom) u1, dudz = u/(zl denom); u1, v1 test-filtered
template <typename T>
__global__ void k_wallstress_frozen(const T *__restrict__ u1, const T *__restrict__ v1, const double *__restrict__ u,
                                    const double *__restrict__ v, T *__restrict__ txz, T *__restrict__ tyz,
                                    T *__restrict__ dudz, T *__restrict__ dvdz, T *__restrict__ ust,
                                    const T *__restrict__ frz_ust, Geo g, double denom, double zl, double vonk) {
  long i = gtid();
  if (i >= g.np) return;
  int x = (int)(i % g.ld);
  if (x >= g.nx) return;
  const double q = -(double)frz_ust[i] * vonk / denom;
  txz[i] = (T)(q * (double)u1[i]);
  tyz[i] = (T)(q * (double)v1[i]);
  dudz[i] = (T)(u[i] / (zl * denom));
  dvdz[i] = (T)(v[i] / (zl * denom));
  ust[i] = frz_ust[i];
}

// sgs_stag.f90:254-325, 391-394 with the Nu_t of a base run (frozen coefficient): the
// stresses of k_nut_tau from the strain rates and a given Nu_t (copied to Nu_t)
template <typename T>
__global__ void k_tau_frozen(const T *__restrict__ S11, const T *__restrict__ S12, const T *__restrict__ S13,
                             const T *__restrict__ S22, const T *__restrict__ S23, const T *__restrict__ S33,
                             const T *__restrict__ frz, T *__restrict__ Nu_t, T *__restrict__ txx,
                             T *__restrict__ txy, T *__restrict__ txz, T *__restrict__ tyy, T *__restrict__ tyz,
                             T *__restrict__ tzz, Geo g) {
  long i = gtid();
  if (i >= g.np * g.nz) return;
  int k = (int)(i / g.np), x = (int)(i % g.ld);
  const T nu = frz[i];
  if (x < g.nx) Nu_t[i] = nu;
  if (k == g.nz - 1) {
    txz[i] = T(0);
    tyz[i] = T(0);
    return;
  }
  if (x >= g.nx) return;
  const T m2 = T(-2), h = T(0.5);
  if (k == 0) {
    txx[i] = m2 * nu * S11[i];
    txy[i] = m2 * nu * S12[i];
    tyy[i] = m2 * nu * S22[i];
    tzz[i] = m2 * nu * S33[i];
  } else {
    const long p = i + g.np;
    const T c = h * (nu + frz[p]);
    txx[i] = m2 * c * h * (S11[i] + S11[p]);
    txy[i] = m2 * c * h * (S12[i] + S12[p]);
    tyy[i] = m2 * c * h * (S22[i] + S22[p]);
    tzz[i] = m2 * c * h * (S33[i] + S33[p]);
    txz[i] = m2 * nu * S13[i];
    tyz[i] = m2 * nu * S23[i];
  }
}

// ------------------------------------------------------------------------------------
// droplets (pollen_all_in_one2, scalars_module_crossflow_mod.f90:1494-1786, with
// pollen_RHS_calc2 :1894-4472, calcbeta_pcon :1795-1843, step_pollen2 :4481-4508), all
// bins in one launch per pass, the faces' adjoints summed over a run of bins in registers and
// over the runs at the end.  Frozen: Kc_t (from Nu_t).  The transport is linear in C on each branch
// of the SMART limiter: its transpose uses the branch the base C selects.  The three
// directions are gathers (a thread per cell adds what the line scan of the fluxes
// transposed would scatter into it, in the scan's order), so no pass needs atomics.
// ------------------------------------------------------------------------------------

// step_pollen2 and calcbeta_pcon transposed (every point of every bin):
// lb, lr the adjoints of the step's PCon and RHS_PCon (lr becomes that of the RHS_PCon the
// step reads); mu = adjoint of this step's RHS_PCon; ac = adjoint of the old PCon through
// the update and the buoyancy (the transport adds to it)
__global__ void k_adj_drop_update(const double *__restrict__ lb_all, double *__restrict__ lr_all,
                                  const double *__restrict__ arz, const double *__restrict__ vfac, int active,
                                  double *__restrict__ mu_all, double *__restrict__ ac_all, DropGeo g, double dt,
                                  int euler) {
  const long t = gtid();
  if (t >= g.nv * g.npc) return;
  const int b = (int)(t / g.nv);
  const long s = t % g.nv, ob = (long)b * g.nv;
  const double *lb = lb_all + ob;
  double *lr = lr_all + ob, *mu = mu_all + ob, *ac = ac_all + ob;
  const int k = (int)(s / g.np), x = (int)(s % g.ld);
  if (k == g.nz - 1 || x >= g.nx) {
    mu[s] = 0.0; ac[s] = 0.0; lr[s] = 0.0;
    return;
  }
  const double l = lb[s] + (k == g.nz - 2 ? lb[s + g.np] : 0.0);  // the top level copies nz-2
  mu[s] = lr[s] + (euler ? dt : 1.5 * dt) * l;
  ac[s] = l + (active ? vfac[b] * arz[s] : 0.0);
  lr[s] = euler ? 0.0 : -0.5 * dt * l;
}

struct DropAdjP {
  double idx, idy, idz, idx2, idy2, idz2;
  int bc_x, bc_y, settling;
};

// The branch that smart_face takes at a face with the difference num across it and den across
// the face before it (downstream of the upwind cell), as the coefficients of the upwind, the
// second upwind and the downwind cell: (1, 0, 0), (0, 0, 1), QUICK (3/4, -1/8, 3/8) or psi = 4
// (3, -2, 0); all have a zero low word.
struct SmartBranch {
  bool up, dn, qk;
  __device__ __forceinline__ SmartBranch(double num, double den) {
    const unsigned long long m = den > 0.0 ? 0ull : 0x8000000000000000ull;
    const double n = __longlong_as_double(__double_as_longlong(num) ^ m), d = fabs(den);
    const double q = 0.375 * n + 0.125 * d, t = fmin(fmin(n, q), d + d);
    up = !(t > 0.0);
    dn = t == n;
    qk = t == q;
  }
  __device__ __forceinline__ static double hi(int h) { return __hiloint2double(h, 0); }
  __device__ __forceinline__ double au() const { return hi(up ? 0x3ff00000 : (dn ? 0 : (qk ? 0x3fe80000 : 0x40080000))); }
  __device__ __forceinline__ double auu() const { return hi(up || dn ? 0 : (qk ? 0xbfc00000 : 0xc0000000)); }
  __device__ __forceinline__ double ad() const { return hi(up ? 0 : (dn ? 0x3ff00000 : (qk ? 0x3fd80000 : 0))); }
};

// the inputs of one line (x or y) through a cell that do not depend on the bin
struct DropLine {
  unsigned o[6];       // byte offsets within a level of cells c-3 .. c-1, c+1 .. c+3 (ghosts: as nb_x below)
  double U[4];         // faces c-1 .. c+2
  double u0, un;       // faces 0 and n (bc 0 and 2)
  double Hm, Hp;       // Kc_t on the faces of the cell
};

// The x (Y false) or y (Y true) transport of one bin transposed in gather form for one cell.  A
// cell adds the terms the line scan of the fluxes transposed scatters into it, in the scan's
// order: the interior faces c-1, c, c+1, c+2, then the end faces, the Kc diffusion of cells
// c-1, c, c+1 (ghosts at the line ends), and last the folds of the ghosts' adjoints at the two
// end cells.  The terms of a face are recomputed by each cell that reads them; cell c adds face
// c's adjoint to af, the end cells the far end's to ae.
template <bool Y>
__device__ __forceinline__ double drop_line_cell(double A, int c, const DropLine &L, const double *__restrict__ Cl,
                                                 const double *__restrict__ Ml, unsigned lvb, unsigned o, double Cc,
                                                 double Mc, const double *__restrict__ Ul, unsigned o0, double &af, double &ae,
                                                 const DropGeo &g, const DropAdjP &P) {
  const int n = Y ? g.ny : g.nx, bc = Y ? P.bc_y : P.bc_x;
  const double id = Y ? P.idy : P.idx, id2 = Y ? P.idy2 : P.idx2;
  double Cw[7], Mw[5];  // cells c-3 .. c+3 with the ghosts, c-2 .. c+2
#pragma unroll
  for (int d = 0; d < 7; ++d) Cw[d] = d == 3 ? Cc : buf_load(Cl, lvb, L.o[d < 3 ? d : d - 1]);
#pragma unroll
  for (int d = 0; d < 5; ++d) Mw[d] = d == 2 ? Mc : buf_load(Ml, lvb, L.o[d < 2 ? d + 1 : d]);
  const double s0 = signbit(L.u0) ? 1.0 : 0.0, s1 = signbit(-L.u0) ? 1.0 : 0.0;
  if (bc == 2) {
#pragma unroll
    for (int d = 0; d < 7; ++d) {
      const int q = c + d - 3;
      Cw[d] *= q < 0 ? s0 : (q >= n ? s1 : 1.0);
    }
  }
  double a[4], D[6];
#pragma unroll
  for (int d = 0; d < 4; ++d) a[d] = L.U[d] * id * (Mw[d + 1] - Mw[d]);
#pragma unroll
  for (int d = 0; d < 6; ++d) D[d] = Cw[d + 1] - Cw[d];
  bool pos[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) pos[d] = L.U[d] >= 0.0;
  // face c + d - 1 lies between cells c + d - 2 and c + d - 1, with D[d + 1] across it
  auto branch = [&](int d) { return SmartBranch(D[d + 1], pos[d] ? D[d] : D[d + 2]); };
  const SmartBranch B0 = branch(0), B1 = branch(1), B2 = branch(2), B3 = branch(3);
  if (c >= 2 && !pos[0]) A += B0.auu() * a[0];
  if (c >= 1) {
    A += (pos[1] ? B1.ad() : B1.au()) * a[1];
    af += smart_between(L.U[1], Cw[2], Cw[3], D[1], D[2], D[3]) * id * (Mw[2] - Mw[1]);
  }
  if (c <= n - 2) A += (pos[2] ? B2.au() : B2.ad()) * a[2];
  if (c <= n - 3 && pos[3]) A += B3.auu() * a[3];
  // faces 0 and n: they reach cells 0, 1, n-2 and n-1 only
  const unsigned st = Y ? 8u * g.ld : 8u;  // o0: cell 0 of the line
  auto Cv = [&](int q) { return buf_load(Cl, lvb, o0 + q * st); };
  auto Mv = [&](int q) { return buf_load(Ml, lvb, o0 + q * st); };
  double a0 = 0.0, aL = 0.0;
  if (bc == 0) {
    if (c <= 1 || c >= n - 2) {
      const double m0 = Mv(0), mL = -Mv(n - 1);
      a0 = L.u0 * id * m0; aL = L.un * id * mL;
      int iu, iuu, idn;
      if (L.u0 >= 0.0) { iu = n - 1; iuu = n - 2; idn = 0; }
      else { iu = 0; iuu = 1; idn = n - 1; }
      const double cu = Cv(iu), cuu = Cv(iuu), cd = Cv(idn);
      const SmartBranch B(cd - cu, cu - cuu);
      if (c == iu || c == iuu || c == idn) A += (c == iu ? B.au() : c == iuu ? B.auu() : B.ad()) * (a0 + aL);
      if (c == 0) {
        const double f0 = smart_face(cu, cuu, cd);
        af += f0 * id * m0;
        ae += f0 * id * mL;
      }
    }
  } else if (bc == 1) {  // x: face 0 carries nothing, face n the last cell; y: the mirror
    if (Y && c == 0) { af += Cc * id * Mc; A += L.U[1] * id * Mc; }
    if (!Y && c == n - 1) { ae += Cc * id * -Mc; A += L.U[2] * id * -Mc; }
  } else {
    a0 = L.U[1] * id * Mc;  // used at the near end only
    aL = L.U[2] * id * -Mc;
    if (c == 0) {  // the ghosts are the end faces
      af += Cw[2] * id * Mc;
      ae += Cv(n - 1) * s1 * id * -Mv(n - 1);
    }
  }
  if (c >= 1) A += L.Hm * (Mw[1] * id2);
  A -= (L.Hp + L.Hm) * (Mc * id2);
  if (c <= n - 2) A += L.Hp * (Mw[3] * id2);
  // the ghosts' adjoints, summed in the scan's order: that of cell -1 is read by cell 0 (its
  // face 1 and diffusion are cell 0's), of cell n by cell n-1; periodic, they are the other end
  if (bc == 0) {
    if (c == n - 1) {
      const double c0 = Cv(0), c1 = Cv(1), u1 = buf_load(Ul, lvb + 8 * g.ld, o0 + st), m0 = Mv(0);
      double ag = 0.0;
      if (u1 >= 0.0) ag += SmartBranch(c1 - c0, c0 - Cc).auu() * (u1 * id * (Mv(1) - m0));
      A += ag + L.Hp * (m0 * id2);
    } else if (c == 0) {
      const double cn1 = Cv(n - 1), cn2 = Cv(n - 2), un1 = buf_load(Ul, lvb + 8 * g.ld, o0 + (n - 1) * st), mn = Mv(n - 1);
      double ag = 0.0;
      if (!(un1 >= 0.0)) ag += SmartBranch(cn1 - cn2, Cc - cn1).auu() * (un1 * id * (mn - Mv(n - 2)));
      A += ag + L.Hm * (mn * id2);
    }
  }
  else if (c == 0 && (Y || bc == 2)) {
    double ag = pos[2] ? B2.auu() * a[2] : 0.0;
    if (bc == 2) ag += a0;
    ag += L.Hm * (Mc * id2);
    A += bc == 2 ? s0 * ag : ag;
  } else if (c == n - 1 && (!Y || bc == 2)) {
    double ag = pos[1] ? 0.0 : B1.auu() * a[1];
    if (bc == 2) ag += aL;
    ag += L.Hp * (Mc * id2);
    A += bc == 2 ? s1 * ag : ag;
  }
  return A;
}

// z in gather form for one cell of one bin: w faces 1..nz-1 (face 0 carries nothing, face nz-1
// repeats nz-2, face 1 is central for upward flow).  A face adds to three distinct cells, so cell
// c takes the terms of faces c-1 .. c+2 and then the Kc diffusion terms of levels c-1, c, c+1, in
// the order of the level scan; cell c adds the adjoint of w face c to af, cell nz-2 also face
// nz-1's to ae.  c is uniform over the block.  W: faces c-1 .. c+3; Hm, Hp: Kc_t on the faces.
__device__ __forceinline__ double drop_z_cell(double A, int c, const double *__restrict__ C,
                                              const double *__restrict__ M, unsigned lvb, unsigned o, double Cc,
                                              double Mc, const double (&W)[5], double Hm, double Hp, double ws,
                                              double &af, double &ae, const DropGeo &g, const DropAdjP &P) {
  const int nz = g.nz;
  auto lv = [&](const double *F, int q) { return buf_load(F + (long)min(max(q, 0), nz - 1) * g.np, lvb, o); };
  double Cw[7], Mw[5];  // cells c-3 .. c+3, c-2 .. c+2 (clamped: those off the column go unused)
#pragma unroll
  for (int d = 0; d < 7; ++d) Cw[d] = d == 3 ? Cc : lv(C, c + d - 3);
#pragma unroll
  for (int d = 0; d < 5; ++d) Mw[d] = d == 2 ? Mc : lv(M, c + d - 2);
#pragma unroll
  for (int d = 0; d < 4; ++d) {  // faces k = c-1 .. c+2 within 1 .. nz-2
    const int k = c + d - 1;
    if (k < 1 || k > nz - 2) continue;
    const double wk = W[d] - ws;
    const bool pos = wk >= 0.0, mid = k == 1 && pos;
    const double m = Mw[d + 1] - Mw[d];
    double at = wk * P.idz * m;
    if (k == nz - 2) at += (W[d + 1] - 0.0) * P.idz * (-Mw[d + 1]);  // face nz-1 joins nz-2
    const double D0 = Cw[d + 1] - Cw[d], D1 = Cw[d + 2] - Cw[d + 1], D2 = Cw[d + 3] - Cw[d + 2];
    const SmartBranch B(D1, pos ? D0 : D2);
    if (d == 0) A += pos ? 0.0 : B.auu() * at;
    if (d == 1) {
      const double face = mid ? 0.5 * (Cw[3] + Cw[2]) : smart_between(wk, Cw[2], Cw[3], D0, D1, D2);
      af += face * P.idz * m;
      if (k == nz - 2) ae += face * P.idz * (-Mw[2]);
      A += (mid ? 0.5 : (pos ? B.ad() : B.au())) * at;
    }
    if (d == 2) A += (mid ? 0.5 : (pos ? B.au() : B.ad())) * at;
    if (d == 3) A += pos ? B.auu() * at : 0.0;
  }
  if (c >= 1 && c - 1 <= nz - 3) A += Hm * (Mw[1] * P.idz2);  // level c-1
  if (c <= nz - 2) {                                          // level c
    const double m = Mc * P.idz2;
    if (c <= nz - 3) A -= Hp * m;
    if (c >= 1) A -= Hm * m;
  }
  if (c + 1 <= nz - 2) A += Hp * (Mw[3] * P.idz2);            // level c+1
  return A;
}

// The three directions for one cell and a run of bins: x, then y (levels below nz-1), then z,
// each as above; blocks of 64 x by 4 y cells, grid z over level + nz group.  The face
// velocities, Kc_t and offsets are read once for all bins, and the faces' adjoints summed over
// the bins in index order: aui, avi, awi hold a face array or volume per group, zero where
// nothing is written here; ac is read, cb (the adjoint of PCon) written.  Bound by its loads
// through L1, 33 per cell and bin; one bin per thread took 78, and the face arrays of each bin
// were cleared, added to and summed by further passes.  128x128x65 with 15 bins: 496 us, with
// the clearing, the sums and a copy 520; 868 and 1090 before.  Two wavefronts per SIMD 545
// us, four 534 (spills).  Beyond the L2s it reads 1.32 GB and writes 0.25 (3.2 TB/s; C, mu, ac and
// cb once are 0.52).
__global__ void __launch_bounds__(256, 3) k_adj_drop_xyz(const double *__restrict__ C, const double *__restrict__ mu,
                                                      const double *__restrict__ ac, double *__restrict__ cb,
                                                      const double *__restrict__ ui0,
                                                      const double *__restrict__ vi0, const double *__restrict__ w,
                                                      double *__restrict__ aui, double *__restrict__ avi,
                                                      double *__restrict__ awi, const double *__restrict__ kc,
                                                      const double *__restrict__ wsb, DropGeo g, DropAdjP P, int ngrp) {
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.nx || j >= g.ny) return;
  const int grp = (int)blockIdx.z / g.nz, k = (int)blockIdx.z - grp * g.nz;
  const int b0 = (int)((long)grp * g.npc / ngrp), b1 = (int)((long)(grp + 1) * g.npc / ngrp);
  const int nx = g.nx, ny = g.ny, nz = g.nz, ld = g.ld;
  const unsigned lvb = 8u * (unsigned)g.np, lvf = lvb + 8u * ld;
  const unsigned r0 = 8u * (j * ld), c0 = 8u * i, o = r0 + c0;
  // cells of a line around c: wrapped when periodic; else the end cell, or for an inlet's zero
  // ghost an offset past the level
  auto nb = [](int q, int n, int bc, int zero) -> int {
    const int v = bc == 0 ? (q < 0 ? q + n : (q >= n ? q - n : q)) : min(max(q, 0), n - 1);
    return bc == 1 && ((zero < 0 && q < 0) || (zero > 0 && q >= n)) ? -1 : v;
  };
  const long lv = (long)k * g.np;
  DropLine X, Y;
#pragma unroll
  for (int d = 0; d < 6; ++d) {
    const int e = d < 3 ? d - 3 : d - 2, qx = nb(i + e, nx, P.bc_x, -1), qy = nb(j + e, ny, P.bc_y, 1);
    X.o[d] = qx < 0 ? kGone : r0 + 8u * qx;
    Y.o[d] = qy < 0 ? kGone : c0 + 8u * (qy * ld);
  }
  const double *ul = ui0 + (long)k * g.fp, *vl = vi0 + (long)k * g.fp, *kl = kc + lv;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    X.U[d] = buf_load(ul, lvf, r0 + 8u * min(max(i + d - 1, 0), nx));
    Y.U[d] = buf_load(vl, lvf, c0 + 8u * (min(max(j + d - 1, 0), ny) * ld));
  }
  X.u0 = buf_load(ul, lvf, r0);
  X.un = buf_load(ul, lvf, r0 + 8u * nx);
  Y.u0 = buf_load(vl, lvf, c0);
  Y.un = buf_load(vl, lvf, c0 + 8u * (ny * ld));
  const double K = buf_load(kl, lvb, o);
  X.Hm = 0.5 * (K + buf_load(kl, lvb, r0 + 8u * (i ? i - 1 : nx - 1)));
  X.Hp = 0.5 * (K + buf_load(kl, lvb, r0 + 8u * (i + 1 < nx ? i + 1 : 0)));
  Y.Hm = 0.5 * (K + buf_load(kl, lvb, c0 + 8u * ((j ? j - 1 : ny - 1) * ld)));
  Y.Hp = 0.5 * (K + buf_load(kl, lvb, c0 + 8u * ((j + 1 < ny ? j + 1 : 0) * ld)));
  const double Zm = 0.5 * (K + buf_load(kc + (long)max(k - 1, 0) * g.np, lvb, o));
  const double Zp = 0.5 * (K + buf_load(kc + (long)min(k + 1, nz - 1) * g.np, lvb, o));
  double W[5];
#pragma unroll
  for (int d = 0; d < 5; ++d) W[d] = buf_load(w + (long)min(max(k + d - 1, 0), nz - 1) * g.np, lvb, o);
  double ax = 0.0, axe = 0.0, ay = 0.0, aye = 0.0, az = 0.0, aze = 0.0;
  for (int b = b0; b < b1; ++b) {
    const double *Cb = C + (long)b * g.nv, *Mb = mu + (long)b * g.nv;
    const double Cc = buf_load(Cb + lv, lvb, o), Mc = buf_load(Mb + lv, lvb, o);
    double A = buf_load(ac + (long)b * g.nv + lv, lvb, o);
    if (k < nz - 1) {
      A = drop_line_cell<false>(A, i, X, Cb + lv, Mb + lv, lvb, o, Cc, Mc, ul, r0, ax, axe, g, P);
      A = drop_line_cell<true>(A, j, Y, Cb + lv, Mb + lv, lvb, o, Cc, Mc, vl, c0, ay, aye, g, P);
    }
    A = drop_z_cell(A, k, Cb, Mb, lvb, o, Cc, Mc, W, Zm, Zp, P.settling ? wsb[b] : 0.0, az, aze, g, P);
    double *out = cb + (long)b * g.nv + lv + o / 8;
    out[0] = A;
    if (i == nx - 1)
      for (int q = 1; q <= ld - nx; ++q) out[q] = 0.0;  // the padding columns
  }
  const long fz = g.fp * nz;
  double *au = aui + grp * fz + (long)k * g.fp, *av = avi + grp * fz + (long)k * g.fp;
  double *aw = awi + (long)grp * g.nv + lv;
  if (k < nz - 1) {
    au[o / 8] = ax;
    if (P.bc_x == 1 ? i == nx - 1 : i == 0) au[r0 / 8 + nx] = axe;
    av[o / 8] = ay;
    if (P.bc_y != 1 && j == 0) av[c0 / 8 + (long)ny * ld] = aye;
  }
  if (k >= 1 && k <= nz - 2) aw[o / 8] = az;
  if (k == nz - 2) aw[o / 8 + g.np] = aze;
}

// the face-velocity reconstruction transposed, along x:
// ui0(i) = mean(u) + P(i) - mean(P), P(i) = sum_{m<i} dx dudx(m), ui0(nx) = ui0(0).  With
// l the adjoint of the faces (face nx folded into 0) and S = sum l:
//   adjoint of dudx(m), m < nx-1: dx (sum_{i>m} l(i) - S (nx-1-m)/nx);  of u(m): S/nx.
// The same along y.
// The face adjoints of all groups of bins summed (from zero), for k_adj_face_line: one
// coalesced pass instead of strided loads per group inside the line passes.
__global__ void k_adj_face_bins(const double *__restrict__ aui, const double *__restrict__ avi,
                                double *__restrict__ lu, double *__restrict__ lv, DropGeo g, int ngrp) {
  const long fz = g.fp * g.nz;
  const long s = gtid();
  if (s >= fz) return;
  double a = 0.0, b = 0.0;
  for (int q = 0; q < ngrp; ++q) {
    a += aui[(long)q * fz + s];
    b += avi[(long)q * fz + s];
  }
  lu[s] = a;
  lv[s] = b;
}

// lsum: k_adj_face_bins's sums.  One line per wave (x: a (y, level) row, y: an (x, level)
// column, consecutive waves at consecutive x): S by a wave sum, the tails sum_{i>m} l(i)
// by suffix scans over 64-face chunks from the end of the line.
template <bool Y>
__global__ void __launch_bounds__(256) k_adj_face_line(const double *__restrict__ lsum, double *__restrict__ ad,
                                                       double *__restrict__ af, DropGeo g, double d) {
  const int lane = threadIdx.x & 63;
  const long line = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int nlat = Y ? g.nx : g.ny;
  if (line >= (long)nlat * g.nz) return;  // uniform over the wave
  const int k = (int)(line / nlat), q = (int)(line % nlat), n = Y ? g.ny : g.nx;
  const long st = Y ? g.ld : 1, ol = Y ? (long)q : (long)q * g.ld;
  const double *L0 = lsum + (long)k * g.fp + ol;
  const long o = (long)k * g.np + ol;
  double part = 0.0;
  for (int i = 1 + lane; i < n; i += 64) part += L0[i * st];
  for (int sh = 32; sh > 0; sh >>= 1) part += __shfl_xor(part, sh, 64);
  const double S = (L0[0] + L0[(long)n * st]) + part;  // face n folded into face 0
  double carry = 0.0;
  for (int base = (n - 1) / 64 * 64; base >= 0; base -= 64) {
    const int m = base + lane;
    double v = m + 1 <= n - 1 ? L0[(long)(m + 1) * st] : 0.0;
    for (int sh = 1; sh < 64; sh <<= 1) {
      const double y = __shfl_down(v, sh, 64);
      if (lane + sh < 64) v += y;
    }
    const double tail = v + carry;  // sum_{i > m} l(i)
    carry = __shfl(tail, 0, 64);
    if (m < n - 1) ad[o + m * st] += d * (tail - S * (double)(n - 1 - m) / n);
    if (m < n) af[o + m * st] += S / n;
  }
}

// afw += the w-face adjoints summed over the groups of bins
__global__ void k_adj_face_w(const double *__restrict__ awi, double *__restrict__ afw, DropGeo g, int ngrp) {
  const long s = gtid();
  if (s >= g.nv) return;
  double v = 0.0;
  for (int b = 0; b < ngrp; ++b) v += awi[(long)b * g.nv + s];
  afw[s] += v;
}

}  // namespace lp
