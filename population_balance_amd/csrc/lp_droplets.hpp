// lp_droplets.hpp -- kernels of the multi-bin droplet concentration step
// (scalars_module_crossflow_mod.f90:1494-1843, 1894-4508: pollen_all_in_one2 with
// pollen_RHS_calc2, calcbeta_pcon, step_pollen2) and of the acceleration update that
// feeds its inertia term (main.f90:864-898).
//
// The droplet state (PCon, RHS_PCon, RHS_PCon_f, Rhs_pbe) and all droplet arithmetic are
// binary64 in both precisions, and so are u, v, w; T is the type of the other fields.  Bin b of a droplet field
// is the (ld, ny, nz) volume at offset b*nv.
#pragma once
#include "lp_kernels.hpp"

namespace lp {

struct DropGeo {
  int nx, ny, nz, ld, npc;
  long np;  // ld*ny
  long nv;  // ld*ny*nz
  long fp;  // ld*(ny+1): one level of a face-velocity array
};

// face velocity reconstruction, :2054-2081 (u) and :2088-2122 (v).  The reference forms
// u_int0 = matrix_x^T (dx dudx(1:nx-1), sum u); that matrix product is
//   u_int0(i) = mean(u) + P(i) - mean(P),  P(i) = sum_{m<i} dx dudx(m),
// i.e. the exclusive prefix sum of dx dudx shifted to the mean of u.  u_int0(nx+1) =
// u_int0(1).  One 64-lane wavefront per (y, z) row, four rows per block.
template <typename T>
__global__ __launch_bounds__(256) void k_face_u(const double *__restrict__ u, const T *__restrict__ dudx,
                                                double *__restrict__ ui0, DropGeo g, double dx) {
  const int lane = threadIdx.x & 63;
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= (long)g.ny * g.nz) return;
  const int k = (int)(row / g.ny), j = (int)(row % g.ny);
  const double *ur = u + (long)k * g.np + (long)j * g.ld;
  const T *er = dudx + (long)k * g.np + (long)j * g.ld;
  double *dst = ui0 + (long)k * g.fp + (long)j * g.ld;
  double su = 0.0, sp = 0.0, carry = 0.0;
  for (int m0 = 0; m0 < g.nx; m0 += 64) {
    const int m = m0 + lane;
    const double e = (m < g.nx - 1) ? dx * (double)er[m] : 0.0;
    double x = e;  // inclusive scan over the 64 lanes
    for (int off = 1; off < 64; off <<= 1) {
      double y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    const double P = carry + (x - e);
    if (m < g.nx) {
      dst[m] = P;
      sp += P;
      su += (double)ur[m];
    }
    carry += __shfl(x, 63, 64);
  }
  for (int off = 32; off >= 1; off >>= 1) {
    su += __shfl_xor(su, off, 64);
    sp += __shfl_xor(sp, off, 64);
  }
  const double A = su / g.nx - sp / g.nx;
  for (int m = lane; m < g.nx; m += 64) dst[m] = A + dst[m];
  if (lane == 0) dst[g.nx] = A + 0.0;
}

// the same reconstruction along y.  A block takes 64 x-columns of one level (coalesced
// over x); its kFaceSeg wavefronts scan consecutive y segments, and the segment sums
// are combined through LDS.
static constexpr int kFaceSeg = 8;
template <typename T>
__global__ __launch_bounds__(64 * kFaceSeg) void k_face_v(const double *__restrict__ v, const T *__restrict__ dvdy,
                                                         double *__restrict__ vi0, DropGeo g, double dy) {
  __shared__ double E[kFaceSeg][64], SU[kFaceSeg][64], SP[kFaceSeg][64];
  const int x = threadIdx.x & 63, seg = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + x, k = blockIdx.y;
  const bool on = i < g.nx;
  const int L = (g.ny + kFaceSeg - 1) / kFaceSeg;
  const int m0 = seg * L, m1 = m0 + L < g.ny ? m0 + L : g.ny;
  const double *vc = v + (long)k * g.np + (on ? i : 0);
  const T *ec = dvdy + (long)k * g.np + (on ? i : 0);
  auto e_at = [&](int m) -> double { return (m < g.ny - 1) ? dy * (double)ec[(long)m * g.ld] : 0.0; };
  double P = 0.0, su = 0.0, sp = 0.0;  // segment-local exclusive prefix and sums
  for (int m = m0; m < m1; ++m) {
    sp += P;
    su += (double)vc[(long)m * g.ld];
    P += e_at(m);
  }
  E[seg][x] = P;
  SU[seg][x] = su;
  SP[seg][x] = sp;
  __syncthreads();
  double off = 0.0, tsu = 0.0, tsp = 0.0, run = 0.0;
  for (int q = 0; q < kFaceSeg; ++q) {
    const int n0 = q * L, n1 = n0 + L < g.ny ? n0 + L : g.ny;
    const int n = n1 > n0 ? n1 - n0 : 0;
    if (q == seg) off = run;
    tsu += SU[q][x];
    tsp += SP[q][x] + (double)n * run;
    run += E[q][x];
  }
  const double A = tsu / g.ny - tsp / g.ny;
  if (!on) return;
  double *dst = vi0 + (long)k * g.fp + i;
  P = off;
  for (int m = m0; m < m1; ++m) {
    dst[(long)m * g.ld] = A + P;
    P += e_at(m);
  }
  if (seg == 0) dst[(long)g.ny * g.ld] = A + 0.0;
}

// :3482-3496 Kc_t = Nu_t on cell centres / Sc (zero outside the cells);
// :2135-2138 magS(:,:,nz) = magS(:,:,nz-1)
template <typename T>
__global__ void k_kc(const T *__restrict__ nut, T *__restrict__ magS, double *__restrict__ kc, DropGeo g,
                     double Sc) {
  const long s = gtid();
  if (s >= g.nv) return;
  const int k = (int)(s / g.np), x = (int)(s % g.ld);
  if (k == g.nz - 1) magS[s] = magS[s - g.np];
  if (k == g.nz - 1 || x >= g.nx) {
    kc[s] = 0.0;
    return;
  }
  const double kv = (k == 0 || k == g.nz - 2) ? (double)nut[s] : ((double)nut[s] + (double)nut[s + g.np]) / 2.0;
  kc[s] = kv / Sc;
}

// SMART face value (:2877-3475) from the upwind cell, the cell upwind of it and the
// downwind cell; a zero upwind gradient takes the upwind value
__device__ __forceinline__ double smart_face(double cup, double cupup, double cdn) {
  // cup + psi(r) den / 2 with r = num / den, psi(r) = max(0, min(2r, 0.75 r + 0.25, 4)),
  // without the division: psi(r) den is max(0, min(2 num, 0.75 num + 0.25 den, 4 den))
  // for den > 0, and min(0, max(...)) of the same three for den < 0
  const double den = cup - cupup;
  if (den == 0.0) return cup;
  const double num = cdn - cup;
  const double a = 2.0 * num, b = 0.75 * num + 0.25 * den, c = 4.0 * den;
  const double pd = den > 0.0 ? fmax(0.0, fmin(fmin(a, b), c)) : fmin(0.0, fmax(fmax(a, b), c));
  return cup + pd / 2.0;
}

__device__ __forceinline__ double sign1(double x) { return signbit(x) ? -1.0 : 1.0; }

struct PollenParams {
  double idx, idy, idz;     // 1/dx, 1/dy, 1/dz
  double idx2, idy2, idz2;  // 1/dx^2 ...
  double psf;               // surface flux (lbcp = 1 keeps only negative values)
  double frac, frac1;       // source shares of levels src_k and src_k+1
  int bc_x, bc_y;           // 0 periodic, 1 inlet, 2 upwind-sign ghosts
  int settling;
  int src_on, src_k0;       // source active this step; its lower level (0-based)
  int runs;                 // runs of levels
  int per;                  // tiles per XCD; 0: tiles in the order of the blocks; -1: runs split over XCDs
};

// Half of the SMART face's correction, psi(r) den / 2 (smart_face): num and den with the sign
// that makes den positive, and the result with its sign again; 0 where den is 0.
__device__ __forceinline__ double smart_half(double num, double den) {
  const unsigned long long m = den > 0.0 ? 0ull : 0x8000000000000000ull;
  const double n = __longlong_as_double(__double_as_longlong(num) ^ m), d = fabs(den);
  const double t = fmax(0.0, fmin(fmin(n, 0.375 * n + 0.125 * d), d + d));
  return __longlong_as_double(__double_as_longlong(t) ^ m);
}

// The SMART value at the face between cells L and R = L + d0, with the differences across
// the faces before (dm) and after (dp): smart_face(L, LL, R) for flow from L, and
// smart_face(R, RR, L) otherwise, where num and den both change sign.
__device__ __forceinline__ double smart_between(double vel, double L, double R, double dm, double d0, double dp) {
  const bool fwd = vel >= 0.0;
  const double h = smart_half(d0, fwd ? dm : dp);
  return fwd ? L + h : R - h;
}

// A value at a 32-bit byte offset from a uniform address (the address in scalar registers, no
// 64-bit vector arithmetic); offsets at or past n bytes read as 0.
template <typename V> __device__ __forceinline__ V buf_load(const V *base, unsigned n, unsigned bytes) {
  const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<V *>(base), 0, (int)n, 0x00027000);
  if constexpr (sizeof(V) == 8) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(V, (u2)__builtin_amdgcn_raw_buffer_load_b64(r, (int)bytes, 0, 0));
  } else {
    return __builtin_bit_cast(V, (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)bytes, 0, 0));
  }
}

// pollen_RHS_calc2 at the cells of a run of levels for a group of kPollenBins bins: face
// velocities of the bin (:2243-2276), ghosts (:2478-2590), SMART faces (:2877-3475), flux
// divergence and SGS diffusion (:3559-3677) and the point source (:4222-4256).
//
// A thread takes one (x, y) and marches up the run of levels blockIdx.z - 1 with the
// concentrations, differences, face values and diffusive fluxes of the last level of its
// bins (blockIdx.y = group) in registers: a level loads one new value along z and computes
// one z face instead of two; the bin-independent inputs (face velocities, accelerations,
// Kc_t) are loaded once per group.  A periodic row or column needs no end cases (its end
// faces use the face-1 velocity, which is that of face n + 1 too): the neighbours are read
// at wrapped indices, and the ghosts of the other boundary conditions are loads too.
// Offsets within a level are 32-bit bytes from uniform addresses.  With kPollenXcd tiles of
// pollen_tile(nx) x (256 / pollen_tile(nx)) points or more, XCD q (blockIdx.x % 8) takes
// consecutive ones (P.per), so that the rows above and below are in its L2, and three of four in
// the CU's L1; fewer would leave XCDs without work (4 tiles at 32x32: 38 us for 33 levels and 16
// bins, in the order of the blocks 20) and go in order.  Fewer tiles than XCDs and kPollenRuns
// runs or more: an XCD takes consecutive runs, the levels of a tile staying in its L2 (32x32x300,
// 4 bins: 28 us, in the order of the blocks 40 to 55).
// Points outside the cells keep the values of the previous RHS: when the caller has moved
// it to RF (RHS_PCon_f = RHS_PCon, :1521, done by exchanging the two buffers) the blocks of
// blockIdx.z = 0 copy them back from RF, otherwise (RF null) they are left alone.
//
// 192x192x128, 15 bins with inertia: 700 us for 2.80 GB beyond the L2s (2.18 read, 0.62
// written, 4.0 TB/s; the concentrations once and their right-hand side are 1.14).  One
// point per thread with both faces of each direction and the end cells by branches was
// bound by its vector instructions (630 per point and bin, now 190) and took 1155 us.  Now
// the loads bound it (9 through L1 per point and bin and 23 per point and group): without
// the arithmetic it takes 700 us, without the neighbours along x 590, along y 620, without
// both 470.  Groups of 3 bins 752, of 4 724, of 5 705 (more do not fit three wavefronts per
// SIMD); the value two levels up or the next bin's loads in flight early: no gain.
static constexpr int kPollenBins = 5;   // bins per thread
__host__ __device__ inline int pollen_tile(int nx) { return nx % 64 == 0 ? 64 : 32; }  // nx % 32 == 0
static constexpr unsigned kGone = 0xfffffff0u;  // past any level: reads 0
// levels per run, at most (8: 745 us, 32: 770, 64: 875 at 192x192x128)
static constexpr int kPollenLevels = 16;
static constexpr int kPollenXcd = 64;   // tiles from which an XCD's are consecutive
static constexpr int kPollenRuns = 64;  // runs from which an XCD's are, with fewer than 8 tiles
template <typename T, bool SIGNS, bool INERT>
__global__ __launch_bounds__(256, SIGNS ? 2 : 3) void k_pollen_rhs(
    const double *__restrict__ PC, double *__restrict__ RH, const double *__restrict__ RF,
    const double *__restrict__ ui0, const double *__restrict__ vi0, const double *__restrict__ w,
    const T *__restrict__ dudt, const T *__restrict__ dvdt, const T *__restrict__ dwdt, const double *__restrict__ kc,
    const double *__restrict__ wsb, const double *__restrict__ qsrc, const double *__restrict__ foot, DropGeo g,
    PollenParams P) {
  constexpr int G = kPollenBins;
  constexpr unsigned D = sizeof(double), S = sizeof(T);
  const int nx = g.nx, ny = g.ny, nz = g.nz, ld = g.ld, np = (int)g.np;
  const int b0 = blockIdx.y * G;  // first bin of the group (uniform)
  const int nb = g.npc - b0 < G ? g.npc - b0 : G;
  if (blockIdx.z == 0) {  // points outside the cells: the padding columns, then the top level
    if (!RF) return;
    const int pad = ld - nx, lev = pad * ny, cols = lev * (nz - 1);
    for (int t = (int)(blockIdx.x * 256 + threadIdx.x); t < cols + np; t += (int)gridDim.x * 256) {
      const int k = t / lev, q = t % lev;
      const long o = t < cols ? (long)k * np + (q / pad) * ld + nx + q % pad : (long)(nz - 1) * np + (t - cols);
      for (int bb = 0; bb < nb; ++bb) RH[(long)(b0 + bb) * g.nv + o] = RF[(long)(b0 + bb) * g.nv + o];
    }
    return;
  }
  const int tw = pollen_tile(nx), ntx = nx / tw;
  const int xcd = (int)(blockIdx.x & 7), xi = (int)(blockIdx.x >> 3);
  int tile, run;
  if (P.per >= 0) {
    tile = P.per ? xcd * P.per + xi : (int)blockIdx.x;
    run = (int)blockIdx.z - 1;
  } else {
    const int ntile = ntx * ((ny + 256 / tw - 1) / (256 / tw));
    tile = xi % ntile;
    run = xcd * ((P.runs + 7) / 8) + xi / ntile;
    if (run >= P.runs) return;
  }
  const int kb = (int)((long)run * (nz - 1) / P.runs), ke = (int)((long)(run + 1) * (nz - 1) / P.runs);
  const int i = tile % ntx * tw + (int)threadIdx.x % tw, j = tile / ntx * (256 / tw) + (int)threadIdx.x / tw;
  if (j >= ny) return;
  const int p = j * ld + i;
  const unsigned lvb = (unsigned)(D * np);  // bytes of a level
  auto at = [&](const double *base, unsigned bytes) -> double { return buf_load<double>(base, lvb + D * ld, bytes); };
  auto att = [&](const T *base, unsigned bytes) -> double { return (double)buf_load<T>(base, lvb, bytes); };
  // byte offsets of binary64 values within a level: this cell, its neighbours around the row
  // and the column (Kc_t, accelerations)
  const int r0 = j * ld;
  const unsigned o = D * p;
  const unsigned kxm = D * (i == 0 ? r0 + nx - 1 : p - 1), kxp = D * (i == nx - 1 ? r0 : p + 1);
  const unsigned kym = D * (j == 0 ? (ny - 1) * ld + i : p - ld), kyp = D * (j == ny - 1 ? i : p + ld);
  // and of the concentrations, the ghosts included: the periodic cell; for an inlet the ghost
  // is 0 (an offset past the level) or the end cell, for the upwind-sign ghosts the end cell
  // times 0 or 1 (ghost_x, ghost_y)
  const int wx = P.bc_x == 0 ? nx : 0, wy = P.bc_y == 0 ? ny : 0;
  const bool inx = P.bc_x == 1, iny = P.bc_y == 1;
  auto nb_x = [&](int q) -> unsigned {
    const int lo = wx ? q + wx : 0, hi = wx ? q - wx : nx - 1, v = q < 0 ? lo : (q >= nx ? hi : q);
    return (inx & (q < 0)) ? kGone : D * (r0 + v);
  };
  auto nb_y = [&](int q) -> unsigned {
    const int lo = wy ? q + wy : 0, hi = wy ? q - wy : ny - 1, v = q < 0 ? lo : (q >= ny ? hi : q);
    return (iny & (q >= ny)) ? kGone : D * (v * ld + i);
  };
  const unsigned oxmm = nb_x(i - 2), oxm = nb_x(i - 1), oxp = nb_x(i + 1), oxpp = nb_x(i + 2);
  const unsigned oymm = nb_y(j - 2), oym = nb_y(j - 1), oyp = nb_y(j + 1), oypp = nb_y(j + 2);
  // the end faces of a row or column that is not periodic carry the ghost
  const bool xb = P.bc_x != 0 && i == 0, xt = P.bc_x != 0 && i == nx - 1;
  const bool yb = P.bc_y != 0 && j == 0, yt = P.bc_y != 0 && j == ny - 1;
  // the z face k of a bin: velocity, value (:3340, :3356: face 0 carries no flux, face 1 is
  // central for upward flow, the top face nz-1 repeats the value of face nz-2)
  auto w_at = [&](int k, double wk, T az, double ws, double f) {  // settling at faces 2..nz-1 of the reference
    const bool in = k >= 1 && k <= nz - 2;  // uniform
    return wk - (in ? ws : 0.0) - (double)az * (in ? f : 0.0);
  };
  auto z_face = [&](int k, double wf, double L, double R, double dm, double d0, double dp) {
    const double c = smart_between(wf, L, R, dm, d0, dp);
    return k == 1 && wf >= 0.0 ? (R + L) / 2.0 : c;
  };
  // state of the run at the bottom face of level kb
  double c0[G], c1[G], d0z[G], zf[G], zd[G];
  double K0 = at(kc + (long)kb * np, o), w0 = at(w + (long)kb * np, o);
  T az0 = INERT ? buf_load<T>(dwdt + (long)kb * np, lvb, o / (D / S)) : T(0);
  const double Kz0 = kb > 0 ? at(kc + (long)(kb - 1) * np, o) : 0.0;
#pragma unroll
  for (int bb = 0; bb < G; ++bb) {
    c0[bb] = c1[bb] = d0z[bb] = zf[bb] = zd[bb] = 0.0;
    if (bb < nb) {
      const double *C = PC + (long)(b0 + bb) * g.nv;
      const double cm2 = at(C + (long)(kb >= 2 ? kb - 2 : 0) * np, o);
      const double cm1 = at(C + (long)(kb >= 1 ? kb - 1 : 0) * np, o);
      c0[bb] = at(C + (long)kb * np, o);
      c1[bb] = at(C + (long)(kb + 1) * np, o);
      d0z[bb] = c0[bb] - cm1;
      if (kb > 0) {
        zf[bb] = z_face(kb, w_at(kb, w0, az0, P.settling ? wsb[b0 + bb] : 0.0, INERT ? wsb[g.npc + b0 + bb] : 0.0), cm1, c0[bb], cm1 - cm2, d0z[bb], c1[bb] - c0[bb]);
        zd[bb] = ((K0 + Kz0) / 2.0) * d0z[bb];
      }
    }
  }
  double rp = 0.0, *Rp = nullptr;  // a value that is still to be stored, and its level
  auto put = [&]() {
    if (Rp) *reinterpret_cast<double *>(reinterpret_cast<char *>(Rp) + o) = rp;
  };
  for (int k = kb; k < ke; ++k) {
    // hidden from the passes that would keep an address for each load in the loop
    int ku = k;
    asm volatile("" : "+s"(ku));
    const long lv = (long)ku * np;  // uniform
    // bin-independent inputs: faces i, i+1 and 1 of the row / column
    const double *ul = ui0 + (long)ku * g.fp, *vl = vi0 + (long)ku * g.fp;
    const double u0 = at(ul, o), u1 = at(ul, o + D);
    const double v0 = at(vl, o), v1 = at(vl, o + D * ld);
    const double w1 = at(w + lv + np, o);
    const double Kxm = at(kc + lv, kxm), Kxp = at(kc + lv, kxp);
    const double Kym = at(kc + lv, kym), Kyp = at(kc + lv, kyp);
    const double K1 = at(kc + lv + np, o);  // used below the top cell only
    T az1 = T(0);
    double ax0 = 0.0, ax1 = 0.0, ay0 = 0.0, ay1 = 0.0, axF = 0.0, ayF = 0.0;
    if constexpr (INERT) {  // accelerations on the faces (:2255-2270); the row's end faces are one
      const T *a = dudt + lv, *b = dvdt + lv;
      const double a0 = att(a, o / (D / S)), e0 = att(b, o / (D / S));
      ax0 = 0.5 * (att(a, kxm / (D / S)) + a0);
      ax1 = 0.5 * (a0 + att(a, kxp / (D / S)));
      ay0 = 0.5 * (att(b, kym / (D / S)) + e0);
      ay1 = 0.5 * (e0 + att(b, kyp / (D / S)));
      az1 = buf_load<T>(dwdt + lv + np, lvb, o / (D / S));
    }
    double uF = 0.0, vF = 0.0;
    if (SIGNS && P.bc_x == 2) {
      uF = at(ul, D * r0);
      if (INERT) axF = 0.5 * (att(dudt + lv, S * (r0 + nx - 1)) + att(dudt + lv, S * r0));
    }
    if (SIGNS && P.bc_y == 2) {
      vF = at(vl, D * i);
      if (INERT) ayF = 0.5 * (att(dvdt + lv, S * ((ny - 1) * ld + i)) + att(dvdt + lv, S * i));
    }
    const double Hxm = (K0 + Kxm) / 2.0, Hxp = (K0 + Kxp) / 2.0, Hym = (K0 + Kym) / 2.0, Hyp = (K0 + Kyp) / 2.0;
    const double Hzp = (K1 + K0) / 2.0;
    const bool top = k == nz - 2;
    double q[9];  // the bin's new values: x and y neighbours, the cell two levels up
    auto load_bin = [&](int bb) {
      const double *C = PC + (long)(b0 + bb) * g.nv + lv;
      q[0] = at(C, oxmm); q[1] = at(C, oxm); q[2] = at(C, oxp); q[3] = at(C, oxpp);
      q[4] = at(C, oymm); q[5] = at(C, oym); q[6] = at(C, oyp); q[7] = at(C, oypp);
      q[8] = at(C + (top ? 1 : 2) * (long)np, o);  // not used at the top cell
    };
#pragma unroll
    for (int bb = 0; bb < G; ++bb) {
      if (bb >= nb) break;
      load_bin(bb);
      put();  // the last bin's value, behind this bin's loads: waiting for them does not wait for it
      double xm2 = q[0], xm1 = q[1], xp1 = q[2], xp2 = q[3], ym2 = q[4], ym1 = q[5], yp1 = q[6], yp2 = q[7];
      const double c2 = q[8];
      // settling velocity and its time scale, read again for each level (scalar loads)
      const double ws = P.settling ? wsb[b0 + bb + (ku - k)] : 0.0, f = INERT ? wsb[g.npc + b0 + bb + (ku - k)] : 0.0;
      const double ci = c0[bb];
      const double uf0 = u0 - ax0 * f, uf1 = u1 - ax1 * f;
      const double vf0 = v0 - ay0 * f, vf1 = v1 - ay1 * f;
      const double wf0 = w_at(k, w0, az0, ws, f), wf1 = w_at(k + 1, w1, az1, ws, f);
      if constexpr (SIGNS) {  // bc 2: the ghosts as cells 0 and n - 1, times (1 -+ sign of face 1) / 2
        const double ufF = uF - axF * f, vfF = vF - ayF * f;
        const double sx0 = P.bc_x == 2 ? (1 - sign1(ufF)) / 2 : 1.0, sxL = P.bc_x == 2 ? (1 - sign1(-ufF)) / 2 : 1.0;
        const double sy0 = P.bc_y == 2 ? (1 - sign1(vfF)) / 2 : 1.0, syL = P.bc_y == 2 ? (1 - sign1(-vfF)) / 2 : 1.0;
        xm2 *= i < 2 ? sx0 : 1.0;
        xm1 *= i < 1 ? sx0 : 1.0;
        xp1 *= i >= nx - 1 ? sxL : 1.0;
        xp2 *= i >= nx - 2 ? sxL : 1.0;
        ym2 *= j < 2 ? sy0 : 1.0;
        ym1 *= j < 1 ? sy0 : 1.0;
        yp1 *= j >= ny - 1 ? syL : 1.0;
        yp2 *= j >= ny - 2 ? syL : 1.0;
      }
      const double dx0 = ci - xm1, dx1 = xp1 - ci, dy0 = ci - ym1, dy1 = yp1 - ci;
      double cxb = smart_between(uf0, xm1, ci, xm1 - xm2, dx0, dx1);
      double cxt = smart_between(uf1, ci, xp1, dx0, dx1, xp2 - xp1);
      double cyb = smart_between(vf0, ym1, ci, ym1 - ym2, dy0, dy1);
      double cyt = smart_between(vf1, ci, yp1, dy0, dy1, yp2 - yp1);
      cxb = xb ? xm1 : cxb;
      cxt = xt ? xp1 : cxt;
      cyb = yb ? ym1 : cyb;
      cyt = yt ? yp1 : cyt;
      const double d1z = c1[bb] - ci, d2z = c2 - c1[bb];
      // the top face: value, diffusive flux
      const double zs = z_face(k + 1, wf1, ci, c1[bb], d0z[bb], d1z, d2z);
      const double zt = top ? zf[bb] : zs, zg = top ? 0.0 : Hzp * d1z;
      double r = -P.idx * (uf1 * cxt - uf0 * cxb);
      r = r - P.idy * (vf1 * cyt - vf0 * cyb);
      r = r - P.idz * (wf1 * zt - wf0 * zf[bb]);
      r = r + P.idx2 * (Hxp * dx1 - Hxm * dx0);
      r = r + P.idy2 * (Hyp * dy1 - Hym * dy0);
      r = r + P.idz2 * (zg - zd[bb]);
      if (k == 0) r = r + P.idz * P.psf;
      rp = r;
      Rp = RH + (long)(b0 + bb) * g.nv + lv;
      zf[bb] = zt;
      zd[bb] = zg;
      c0[bb] = c1[bb];
      c1[bb] = c2;
      d0z[bb] = d1z;
    }
    K0 = K1;
    w0 = w1;
    az0 = az1;
  }
  put();
  if (P.src_on)
    for (int k = kb; k < ke; ++k)
      if (k == P.src_k0 || k == P.src_k0 + 1) {  // its two levels
        const double fr = (k == P.src_k0) ? P.frac : P.frac1, fsrc = foot[(long)j * nx + i];
        for (int bb = 0; bb < nb; ++bb) RH[(long)(b0 + bb) * g.nv + (long)k * np + p] += fr * qsrc[b0 + bb] * fsrc;
      }
}

// breakage-frequency fit of one bin (:2167-2230): the Ohnesorge-number coefficients and
// the two diameter powers
struct PbeBin {
  double a, b, c, d, e;
  double dpow_tau;  // d^-0.6666667
  double dpow_re;   // d^(4/3)
};
// one (smaller bin i, larger bin j) pair of the transfer (:4356-4448): a drop of bin j
// breaks into bin i with probability beta; the complementary drop of diameter
// (d_j^3 - d_i^3)^(1/3) is split between bins lo and hi with volume weights
struct PbePair {
  int i, j, lo, hi;  // lo/hi < 0: no target
  double beta, wlo, whi;
};

// Rhs_pbe for every bin at one cell; zero outside the cells (the reference clears the
// whole array, :2005-2021).  With feedback, RHS_PCon += Rhs_pbe.  The pair loop of
// :4356-4448 is linear in g_j = gf(j) PCon(j): Rhs_pbe(b) = sum_j A(b, j) g_j with
// A(b, j) = sum over the pairs (i, j) of beta_ij (+1 into i, -1 out of j, + w_lo / w_hi into
// the complementary drop's bins), built on the host.  NB >= npc bins are held in
// registers (loops unrolled, bins >= npc skipped); A is read through the scalar cache.
// pow(Re1, b) and pow(Re1, d) share one logarithm (exp(b ln Re1)) and pow(10, x) is
// exp10(x); both agree with pow to a few ulp.
//
// STEP (pollen_all_in_one2 with the breakup source on): the same pass then does
// calcbeta_pcon and step_pollen2 at the point (as k_beta_step, from the old PCon), and on
// an Euler start first sets RHS_PCon_f = RHS_PCon (:1660-1665).
struct PbeStep {
  double *PCw;           // PCon (the same array as PC), advanced in place at this point
  double *RF;            // RHS_PCon_f
  void *bp;              // beta_pcon (field type)
  const double *vfac;    // buoyancy factor of each bin
  int active, euler;
  double dt;
};
template <typename T, int NB, bool STEP>
__global__ __launch_bounds__(256) void k_pbe(const double *PC, double *__restrict__ PB,
                                             double *__restrict__ RH, const T *__restrict__ dissip,
                                             const PbeBin *__restrict__ bins, const double *__restrict__ A,
                                             DropGeo g, double kpref, double ustar3, double z_i, double nu_c,
                                             int feedback, PbeStep St) {
  const long s = gtid();
  if (s >= g.nv) return;
  const int npc = g.npc;
  const int k = (int)(s / g.np), x = (int)(s % g.ld);
  if (k >= g.nz - 1 || x >= g.nx) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (b < npc) PB[(long)b * g.nv + s] = 0.0;
    if constexpr (STEP) {  // as k_beta_step outside the cells
      T *bp = (T *)St.bp;
      bp[s] = T(0);
      if (k == g.nz - 2)
#pragma unroll
        for (int b = 0; b < NB; ++b)
          if (b < npc) St.PCw[(long)b * g.nv + s + g.np] = St.PCw[(long)b * g.nv + s];
    }
    return;
  }
  const double eps = (double)dissip[s];
  const double ds = eps * ustar3 / z_i;
  const double et = pow(fabs(eps), 0.33333333);
  const double er = pow(fabs(ds), 1.0 / 3.0);
  double gj[NB], pc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    gj[b] = 0.0;
    pc[b] = 0.0;
    if (b < npc) {
      const PbeBin B = bins[b];
      const double tau_c = et * B.dpow_tau;
      const double Re = er * B.dpow_re / nu_c;
      const double Re1 = log10(Re);
      const double fb = 0.5 * (sign1(Re1) + 1.0);
      double pb = 1.0, pd = 1.0;  // pow(Re1, fb b), pow(Re1, fb d): 1 when fb = 0
      if (fb != 0.0) {
        const double lr = log(Re1);
        pb = exp(B.b * lr);
        pd = exp(B.d * lr);
      }
      const double al = B.a * fb * pb;
      const double bl = fb * B.c * pd - B.e;
      const double fit = exp10(al + bl);
      pc[b] = PC[(long)b * g.nv + s];
      gj[b] = kpref * tau_c * fit * pc[b];
    }
  }
  double tb = 0.0;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (b < npc) {
      double acc = 0.0;
#pragma unroll
      for (int j = 0; j < NB; ++j)
        if (j < npc) acc = fma(A[b * npc + j], gj[j], acc);
      const long o = (long)b * g.nv + s;
      PB[o] = acc;
      double rh = RH[o];
      if (feedback) {
        rh = rh + acc;
        RH[o] = rh;
      }
      if constexpr (STEP) {  // calcbeta_pcon from the old PCon, then step_pollen2
        double rf;
        if (St.euler) {
          St.RF[o] = rh;
          rf = rh;
        } else {
          rf = St.RF[o];
        }
        const double c = pc[b];
        tb = tb + St.vfac[b] * c;
        const double cn = c + St.dt * (1.5 * rh - 0.5 * rf);
        St.PCw[o] = cn;
        if (k == g.nz - 2) St.PCw[o + g.np] = cn;
      }
    }
  }
  if constexpr (STEP) {
    T *bp = (T *)St.bp;
    bp[s] = St.active ? (T)tb : T(0);
  }
}

// calcbeta_pcon (:1795-1843; buoyancy of all bins into beta_pcon, zero outside the cells
// or when the droplets are passive) and step_pollen2 (:4481-4508; AB2 in the cells, the
// top level copies level nz-1).  One thread per point of the volume.
// do_beta / do_step select either routine or both (fused: one pass over PCon).
template <typename T>
__global__ void k_beta_step(double *__restrict__ PC, const double *__restrict__ RH, const double *__restrict__ RF,
                            T *__restrict__ bp, const double *__restrict__ vfac, int active, DropGeo g, double dt,
                            int do_beta, int do_step) {
  const long s = gtid();
  if (s >= g.nv) return;
  const int k = (int)(s / g.np), x = (int)(s % g.ld);
  if (k == g.nz - 1) {
    if (do_beta) bp[s] = T(0);
    return;
  }
  if (x >= g.nx) {
    if (do_beta) bp[s] = T(0);
    if (do_step && k == g.nz - 2)
      for (int b = 0; b < g.npc; ++b) PC[(long)b * g.nv + s + g.np] = PC[(long)b * g.nv + s];
    return;
  }
  double tb = 0.0;
  for (int b = 0; b < g.npc; ++b) {
    const long o = (long)b * g.nv + s;
    const double c = PC[o];
    if (do_beta) tb = tb + vfac[b] * c;
    if (do_step) {
      const double cn = c + dt * (1.5 * RH[o] - 0.5 * RF[o]);
      PC[o] = cn;
      if (k == g.nz - 2) PC[o + g.np] = cn;
    }
  }
  if (do_beta) bp[s] = active ? (T)tb : T(0);
}

// energy.f90:23-31 kinetic energy on the uvp nodes (zero outside the cells)
template <typename T>
__global__ void k_energy(const double *__restrict__ u, const double *__restrict__ v, const double *__restrict__ w,
                         T *__restrict__ ke, Geo g) {
  const long i = gtid();
  if (i >= g.np * g.nz) return;
  const int k = (int)(i / g.np), x = (int)(i % g.ld);
  if (k == g.nz - 1 || x >= g.nx) {
    ke[i] = T(0);
    return;
  }
  const double tw = 0.5 * (w[i] + w[i + g.np]);
  ke[i] = (T)(0.5 * (u[i] * u[i] + v[i] * v[i] + tw * tw));
}

// main.f90:883-885 with ddz_uv(dkedz, ke) folded in (ddz_uv.f90:39-57: level 1 and the
// columns beyond nx add nothing)
template <typename T>
__global__ void k_ke_add(T *__restrict__ dudt, T *__restrict__ dvdt, T *__restrict__ dwdt,
                         const T *__restrict__ kex, const T *__restrict__ key, const T *__restrict__ ke, Geo g,
                         T idz) {
  const long i = gtid();
  if (i >= g.np * (g.nz - 1)) return;
  const int k = (int)(i / g.np), x = (int)(i % g.ld);
  dudt[i] += kex[i];
  dvdt[i] += key[i];
  const T kz = (k >= 1 && x < g.nx) ? idz * (ke[i] - ke[i - g.np]) : T(0);
  dwdt[i] += kz;
}

}  // namespace lp
