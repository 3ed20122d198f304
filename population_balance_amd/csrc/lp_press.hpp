// lp_press.hpp -- the pressure's tridiagonal systems, one per (kx, ky) mode, and their
// transposes, with the levels of a mode split over the wavefronts of a block.
//
// Every system of a context has the same coefficients (the grid's), so the elimination
// factors are tabled once (k_press_factors) and the Thomas sweeps become two first-order
// recurrences per mode, u(j) = (r(j) - a(j) u(j-1))/bet(j) upwards and
// p(j) = u(j) - c(j)/bet(j) p(j+1) downwards.  A recurrence over levels is affine in the
// value that enters it, so a block of 16 modes x S segments of rows sweeps every segment
// once from zero (its affine map: a factor and an offset), scans the S maps over LDS, and
// sweeps again from the value that really enters.  The factors of the interior rows are below
// 1 in magnitude (|bet(j)| >= kx^2 + ky^2 + 1/dz^2 by induction), so that their maps shrink what
// they join.  Those of the end rows may be large: the lid row's -1/bet(nz) is -337 for kx = 1,
// dz = 1/256, nz = 257, and in the transposed systems it is 1/(dz^2 bet(nz)), 2.2e7, with -1/dz^2
// for the wall row downwards.  They amplify nothing, because an end row is the last of its sweep:
// no row is entered through its map, and its own value is formed from its neighbour's as in
// the serial sweep.  The rows stay in registers between the two directions.
//
// What bounds it: one thread per mode held 33 K (256 x 256) to 0.5 K (32 x 32) threads, too
// few to keep memory busy, each on a serial chain of 2 (nz + 1) rows with its p_hat written,
// read and written again.  Segments give 8 to 32 times the threads, one read of H and one
// write of p_hat.  16 modes (128 or 256 bytes a row) per block keep every access whole
// 128-byte lines (modes are taken in the spectra's own pitch, not as kx + lh ky), and at
// 122 VGPRs (binary32) two blocks of 512 threads share a CU, so that one block's loads run
// beside the other's sweeps.  RNDS false leaves out the loop over rounds, which would cost
// 60 registers.  Measured, one thread per mode -> this: binary32 spectra 246 -> 94 us at
// 256 x 256 x 257 (H, 1/bet and p_hat: 415 MB, 4.4 TB/s), 94 -> 31 us at 192 x 192 x 128;
// binary64 80 -> 33 us at 128 x 128 x 129, 23 -> 12 us at 32 x 32 x 33; the transposed solve
// 95 -> 19 us at 128 x 128 x 65.
#pragma once
#include "lp_kernels.hpp"

namespace lp {

constexpr int kPsModes = 16;  // modes per block
constexpr int kPsRows = 9;    // rows of a segment held in registers

// segments per block for n rows: the fewest of 8, 16, 32 that hold all rows at once; beyond
// 32 kPsRows = 288 rows a block of 32 takes several rounds and keeps the sweep's values in
// p_hat between them
__host__ __device__ constexpr int press_segs(int n) {
  return n <= 8 * kPsRows ? 8 : n <= 16 * kPsRows ? 16 : 32;
}
__host__ __device__ constexpr bool press_rounds(int n) { return n > 32 * kPsRows; }

// The binary64 solve hands the elimination from segment to segment, so a block of 32 segments,
// which leaves room for no other on its CU, stands still while one of them sweeps.  With a block
// for every CU, 16 segments in rounds are better beyond 144 rows: two blocks share a CU and one
// loads while the other sweeps.  16 against 32 segments: 165 against 242 us at 256 x 256 x 160
// (one thread per mode 162), 226 / 305 at 256 x 256 x 257 (281), 299 / 567 at 300 levels (342), 387
// / 641 at 400 (468), 69 / 102 at 128 x 128 x 257 (158).  With fewer blocks than CUs there is
// nothing to share a CU with: 323 / 274 at 32 x 32 x 2000 (64 blocks), 63 / 63 at 64 x 64 x 300 (192).
// The rounds are equal in length.
__host__ __device__ constexpr int press_segs64(int n, long blocks) {
  return n > 16 * kPsRows && blocks >= 256 ? 16 : press_segs(n);
}
__host__ __device__ constexpr int serial_rounds(int n, int S) { return (n + S * kPsRows - 1) / (S * kPsRows); }
__host__ __device__ constexpr int serial_rows(int n, int S) {
  return (n + S * serial_rounds(n, S) - 1) / (S * serial_rounds(n, S));
}

// press_stag_array.f90:149-329 / tridag_array.f90:30-155: bet(j) of each mode's system
// (a = c = 1/dz^2, b = -(kx^2 + ky^2 + 2/dz^2) inside; the wall row b = -1, c = 1; the lid
// row a = -1, b = 1), bet(j) = b(j) - a(j) (c(j-1)/bet(j-1)), in [(nz+1)][ny][pitch]; inv:
// 1/bet(j) instead.  Modes the solve skips (mean, Nyquist) are left alone.
static __global__ void k_press_factors(const double *__restrict__ kxt, const double *__restrict__ kyt,
                                       double *__restrict__ tab, int lh, int ny, int nz, long pitch, double dz,
                                       int inv) {
  const long m = gtid();
  const long nh = (long)lh * ny;
  if (m >= nh) return;
  const int jx = (int)(m % lh), jy = (int)(m / lh);
  if (jy == ny / 2 || jx == lh - 1 || m == 0) return;
  const long o = (long)jy * pitch + jx, ps = pitch * ny;
  const double kx = kxt[m], ky = kyt[m];
  const double idz2 = 1.0 / (dz * dz);
  const double bi = -(kx * kx + ky * ky + 2.0 / (dz * dz));
  double bet = -1.0, cprev = 1.0;
  tab[o] = bet;
  for (int j = 1; j <= nz; ++j) {
    const double a = j < nz ? idz2 : -1.0, b = j < nz ? bi : 1.0;
    bet = b - a * (cprev / bet);
    tab[(long)j * ps + o] = inv ? 1.0 / bet : bet;
    cprev = idz2;
  }
}

// Addresses.  A volume of spectra may be larger than 4 GiB (256 x 256 modes from 7282 rows of
// 16 bytes on), so a row's place in it takes 64 bits.  The rows of a wavefront's 64 / kPsModes
// segments follow one another: the address of the first (row0) is uniform and stays in scalar
// registers, and a lane adds a 32-bit offset within the next (64 / kPsModes) kPsRows + 1 rows of at
// most 256 x 144 values, 22 MB.  row >= row0.
__host__ __device__ constexpr unsigned row_off(int row, int row0, unsigned ps, unsigned o, unsigned bytes) {
  return ((unsigned)(row - row0) * ps + o) * bytes;
}
__host__ __device__ constexpr long row_base(int row0, unsigned ps) { return (long)row0 * (long)ps; }

template <typename E>
__device__ __forceinline__ E at_row(const E *base, int row, int row0, unsigned ps, unsigned o) {
  return *reinterpret_cast<const E *>(reinterpret_cast<const char *>(base + row_base(row0, ps)) +
                                      row_off(row, row0, ps, o, sizeof(E)));
}

template <typename E>
__device__ __forceinline__ void put_row(E *base, int row, int row0, unsigned ps, unsigned o, E v) {
  *reinterpret_cast<E *>(reinterpret_cast<char *>(base + row_base(row0, ps)) + row_off(row, row0, ps, o, sizeof(E))) = v;
}

// the plane of an H level or gradient, levels 1 .. nz-1 at planes 0 .. nz-2, of row j (clamped)
__host__ __device__ constexpr int press_plane(int j, int nz) { return j < 1 ? 0 : j > nz - 1 ? nz - 2 : j - 1; }

// the first segment of the thread's wavefront
__device__ __forceinline__ int wave_seg() {
  return __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64 * (64 / kPsModes));
}

template <int S> struct SegLds {
  double a[2][S][kPsModes], x[2][S][kPsModes], y[2][S][kPsModes];
};

// v(end) = A v(in) + B of segment s (counted along the sweep) of mode l; returns the value
// that enters segment s when `first` enters segment 0, and the last segment's end in `last`
template <int S>
__device__ __forceinline__ cx<double> seg_enter(SegLds<S> &L, int s, int l, double A, cx<double> B, cx<double> first,
                                                cx<double> &last) {
  int p = 0;
  L.a[p][s][l] = A; L.x[p][s][l] = B.x; L.y[p][s][l] = B.y;
  __syncthreads();
#pragma unroll
  for (int d = 1; d < S; d <<= 1) {
    if (s >= d) {
      const double a2 = L.a[p][s - d][l];
      B = mk<double>(B.x + A * L.x[p][s - d][l], B.y + A * L.y[p][s - d][l]);
      A = A * a2;
    }
    p ^= 1;
    L.a[p][s][l] = A; L.x[p][s][l] = B.x; L.y[p][s][l] = B.y;
    __syncthreads();
  }
  cx<double> r = first;
  if (s > 0) {
    const double a = L.a[p][s - 1][l];
    r = mk<double>(L.x[p][s - 1][l] + a * first.x, L.y[p][s - 1][l] + a * first.y);
  }
  const double a = L.a[p][S - 1][l];
  last = mk<double>(L.x[p][S - 1][l] + a * first.x, L.y[p][S - 1][l] + a * first.y);
  __syncthreads();
  return r;
}

// The two sweeps of one block, u(j) = r(j) - f(j) u(j-1) with rows up, then
// p(j) = u(j) - fb(j, f(j)) p(j+1) down.  load(j0, jw, Lr) fills r and f of this thread's rows
// j0 .. j0 + Lr - 1 (clamped beyond n); out(j, jw, p(j), p(j+1)) takes the solution.  jw is the
// first row of the wavefront's segments (uniform, it may lie beyond n).  u: scratch
// for the rounds but the last (n > S kPsRows), [n][plane], this thread's own rows.
template <int S, bool RNDS, typename Load, typename Fb, typename Out>
__device__ __forceinline__ void seg_solve(SegLds<S> &L, int s, int l, int n, Load load, Fb fb, Out out,
                                          cx<double> (&r)[kPsRows], double (&f)[kPsRows],
                                          cx<double> *__restrict__ u, unsigned plane) {
  const int per = (n + S - 1) / S;
  const int Lr = per < kPsRows ? per : kPsRows;
  const int rounds = RNDS ? (n + S * Lr - 1) / (S * Lr) : 1;
  const int sw = wave_seg();
  cx<double> carry = mk<double>(0.0, 0.0), last;
  for (int rd = 0; rd < rounds; ++rd) {
    const int j0 = (rd * S + s) * Lr, jw = (rd * S + sw) * Lr;
    const int nr = n - j0 < Lr ? n - j0 : Lr;  // rows of this segment (none: <= 0)
    load(j0, jw, Lr);
    double A = 1.0;
    cx<double> B = mk<double>(0.0, 0.0);
#pragma unroll
    for (int q = 0; q < kPsRows; ++q)
      if (q < nr) {
        B = mk<double>(r[q].x - f[q] * B.x, r[q].y - f[q] * B.y);
        A = -f[q] * A;
      }
    cx<double> v = seg_enter<S>(L, s, l, A, B, carry, last);
    carry = last;
#pragma unroll
    for (int q = 0; q < kPsRows; ++q)
      if (q < nr) {
        v = mk<double>(r[q].x - f[q] * v.x, r[q].y - f[q] * v.y);
        r[q] = v;
      }
    if (rd + 1 < rounds)
#pragma unroll
      for (int q = 0; q < kPsRows; ++q)
        if (q < nr) u[(size_t)(j0 + q) * plane] = r[q];
  }
  carry = mk<double>(0.0, 0.0);
  for (int rd = rounds - 1; rd >= 0; --rd) {
    const int j0 = (rd * S + s) * Lr, jw = (rd * S + sw) * Lr;
    const int nr = n - j0 < Lr ? n - j0 : Lr;
    if (rd + 1 < rounds) {
      load(j0, jw, Lr);  // f again; r is replaced by the forward sweep's values
#pragma unroll
      for (int q = 0; q < kPsRows; ++q)
        if (q < nr) r[q] = u[(size_t)(j0 + q) * plane];
    }
    double A = 1.0;
    cx<double> B = mk<double>(0.0, 0.0);
#pragma unroll
    for (int q = kPsRows - 1; q >= 0; --q)
      if (q < nr) {
        const double g = fb(j0 + q, f[q]);
        B = mk<double>(r[q].x - g * B.x, r[q].y - g * B.y);
        A = -g * A;
      }
    cx<double> v = seg_enter<S>(L, S - 1 - s, l, A, B, carry, last);
    carry = last;
#pragma unroll
    for (int q = kPsRows - 1; q >= 0; --q)
      if (q < nr) {
        const double g = fb(j0 + q, f[q]);
        const cx<double> up = v;
        v = mk<double>(r[q].x - g * v.x, r[q].y - g * v.y);
        out(j0 + q, jw, v, up);
      }
  }
}

// x / b rounded as the division rounds it, from rb = 1 / b rounded: the quotient's residual is
// exact in one fused multiply-add, and the correction by it rounds correctly (Markstein 1990).
// That holds for finite x, b, rb and x rb with |x| and |x / b| above 2^-960 or x = 0; below, the
// residual may be subnormal and the last place off, and an infinite x gives NaN where the division
// gives an infinity (a step reports either, in the velocity).  b = 0 is reported on its own (err).
__device__ __forceinline__ double div_by(double x, double b, double rb) {
  const double q = x * rb;
  return fma(fma(-q, b, x), rb, q);
}

// The same solve in the reference's own order of operations (tridag_array.f90:60-80):
// u(j) = (r(j) - a(j) u(j-1))/bet(j), gam(j+1) = c(j)/bet(j), p(j) = u(j) - gam(j+1) p(j+1),
// every segment waiting for the one below (above).  The chain of a row is four operations
// (div_by) instead of a division's fourteen, the loads and the stores of all segments run
// beside it.  f: bet.  num(j, r(j), u(j-1)) = r(j) - a(j) u(j-1) of one component, above(j) = c(j).
template <int S, bool RNDS, typename Load, typename Num, typename Up, typename Out>
__device__ __forceinline__ void seg_solve_serial(cx<double> (&end)[kPsModes], int s, int l, int n, Load load, Num num,
                                                 Up above, Out out, cx<double> (&r)[kPsRows], double (&f)[kPsRows],
                                                 cx<double> *__restrict__ u, unsigned plane) {
  const int rounds = RNDS ? serial_rounds(n, S) : 1;
  const int Lr = serial_rows(n, S);
  const int sw = wave_seg();
  double rb[kPsRows];
  if (s == 0) end[l] = mk<double>(0.0, 0.0);
  for (int rd = 0; rd < rounds; ++rd) {
    const int j0 = (rd * S + s) * Lr, jw = (rd * S + sw) * Lr;
    const int nr = n - j0 < Lr ? n - j0 : Lr;
    load(j0, jw, Lr);
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) rb[q] = 1.0 / f[q];
    __syncthreads();
    for (int sg = 0; sg < S; ++sg) {
      if (sg == s) {
        cx<double> v = end[l];
#pragma unroll
        for (int q = 0; q < kPsRows; ++q)
          if (q < nr) {
            v = mk<double>(div_by(num(j0 + q, r[q].x, v.x), f[q], rb[q]), div_by(num(j0 + q, r[q].y, v.y), f[q], rb[q]));
            r[q] = v;
          }
        end[l] = v;
      }
      __syncthreads();
    }
    if (rd + 1 < rounds)
#pragma unroll
      for (int q = 0; q < kPsRows; ++q)
        if (q < nr) u[(size_t)(j0 + q) * plane] = r[q];
  }
  if (s == 0) end[l] = mk<double>(0.0, 0.0);
  for (int rd = rounds - 1; rd >= 0; --rd) {
    const int j0 = (rd * S + s) * Lr, jw = (rd * S + sw) * Lr;
    const int nr = n - j0 < Lr ? n - j0 : Lr;
    if (rd + 1 < rounds) {
      load(j0, jw, Lr);
#pragma unroll
      for (int q = 0; q < kPsRows; ++q) {
        rb[q] = 1.0 / f[q];
        if (q < nr) r[q] = u[(size_t)(j0 + q) * plane];
      }
    }
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) rb[q] = div_by(above(j0 + q), f[q], rb[q]);  // gam(j + 1)
    __syncthreads();
    for (int sg = S - 1; sg >= 0; --sg) {
      if (sg == s) {
        cx<double> v = end[l];
#pragma unroll
        for (int q = kPsRows - 1; q >= 0; --q)
          if (q < nr) {
            v = mk<double>(r[q].x - rb[q] * v.x, r[q].y - rb[q] * v.y);
            r[q] = v;
          }
        end[l] = v;
      }
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kPsRows; ++q)
      if (q < nr) out(j0 + q, jw, r[q], r[q]);
  }
}

// press_stag_array.f90:149-329 + tridag_array.f90:30-155: the wall row, the interior rows
// and the lid row assembled on the fly, the solve, the gauge-fixed cumulative sum of the
// mean mode (a = -1, 1/bet = 1, no backward sweep), zero on the Nyquist row and column.
// H levels 1..nz-1 at planes 0..nz-2 (complex TH), bw / tw_ one plane, ph planes 0..nz.
template <typename TH, int S, bool RNDS>
__global__ __launch_bounds__(kPsModes *S, RNDS && sizeof(TH) == 4 ? 1 : sizeof(TH) == 4 ? 4 : 3) void k_press_tridiag(
    const cx<TH> *__restrict__ Hx, const cx<TH> *__restrict__ Hy, const cx<TH> *__restrict__ Hz,
    const cx<TH> *__restrict__ bw, const cx<TH> *__restrict__ tw_, const double *__restrict__ kxt,
    const double *__restrict__ kyt, cx<double> *ph, const double *__restrict__ tab, int lh, int ny, int nz,
    long pitch, double dz, int *__restrict__ err) {
  // Binary32 spectra: tab holds 1/bet, r is taken times it, a row of the sweep is one fused
  // multiply-add and the segments are joined by the scan.  Binary64: tab holds bet and the
  // rows go in the reference's order with its rounding (the scan's own rounding, no larger,
  // moved RHSx of 50 steps at 128 x 128 x 129 from 8.0e-13 to 2.7e-12 of the reference).
  constexpr bool DIV = sizeof(TH) == 8;
  const int l = threadIdx.x % kPsModes, s = threadIdx.x / kPsModes;
  const long ps = pitch * ny;
  const long o = (long)blockIdx.x * kPsModes + l;  // ps is a multiple of kPsModes
  const int jy = (int)(o / pitch), jx = (int)(o % pitch);
  const bool store = jx < lh;
  const bool live = jx < lh - 1 && jy != ny / 2;
  const bool mean = o == 0;
  const long oc = live ? o : 0;  // lanes without a mode read mode 0 and drop it
  const unsigned ocu = (unsigned)oc, psu = (unsigned)ps;
  const long m = (long)jy * lh + (store ? jx : 0);
  const double kx = kxt[m], ky = kyt[m];
  const double idz2 = 1.0 / (dz * dz), idz = 1.0 / dz;
  cx<double> r[kPsRows];
  double f[kPsRows];
  bool bad = false;
  // the coefficient below the diagonal: 1/dz^2, -1 in the lid row and for the mean's sum
  auto below = [&](int j) { return !live || j == 0 ? 0.0 : (mean || j == nz) ? -1.0 : idz2; };
  auto load = [&](int j0, int jw, int Lr) {
    cx<TH> hz[kPsRows + 1], hx[kPsRows], hy[kPsRows];
    double ib[kPsRows];
    const int pw = press_plane(jw, nz), tw0 = jw > nz ? nz : jw;
    auto row_of = [&](int q) { return j0 + (q < Lr ? q : Lr - 1); };
    auto at_h = [&](const cx<TH> *H, int j) { return at_row(H, press_plane(j, nz), pw, psu, ocu); };
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) {
      const int j = row_of(q);
      ib[q] = at_row(tab, j > nz ? nz : j, tw0, psu, ocu);
      hz[q] = at_h(Hz, j);
    }
    hz[kPsRows] = at_h(Hz, j0 + Lr);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) hx[q] = at_h(Hx, row_of(q));
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) {  // (Hz(j+1) - Hz(j))/dz, H_z zero at level nz
      const int j = j0 + q;
      const cx<TH> h0 = hz[q], h1 = q + 1 < Lr ? hz[q + 1] : hz[kPsRows];
      const double z1x = j + 1 < nz ? (double)h1.x : 0.0, z1y = j + 1 < nz ? (double)h1.y : 0.0;
      const double dx = z1x - (double)h0.x, dy = z1y - (double)h0.y;
      r[q] = mean ? (DIV ? mk<double>((double)h0.x, (double)h0.y) : mk<double>((double)h0.x * dz, (double)h0.y * dz))
                  : DIV ? mk<double>(dx / dz, dy / dz) : mk<double>(dx * idz, dy * idz);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) hy[q] = at_h(Hy, row_of(q));
    const cx<TH> b0 = bw[oc], t0 = tw_[oc];
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) {
      const int j = j0 + q;
      const bool own = q < Lr && j <= nz;
      if (own && live && !mean && (DIV ? ib[q] == 0.0 : isinf(ib[q]))) bad = true;  // bet(j) == 0
      // i (kx Hx + ky Hy) + (Hz(j+1) - Hz(j))/dz
      const double sx = kx * (double)hx[q].x + ky * (double)hy[q].x;
      const double sy = kx * (double)hx[q].y + ky * (double)hy[q].y;
      cx<double> v = mk<double>(-sy + r[q].x, sx + r[q].y);
      if (mean) {  // :303-312
        v = r[q];
        if (j == 0 || j == nz) v = mk<double>(0.0, 0.0);
        if (j == 1) v = mk<double>(-dz * (double)b0.x, -dz * (double)b0.y);
        ib[q] = 1.0;
      } else {
        if (j == 0) v = mk<double>(-dz * (double)b0.x, -dz * (double)b0.y);
        if (j == nz) v = mk<double>(-(double)t0.x * dz, -(double)t0.y * dz);
      }
      if constexpr (DIV) {
        r[q] = live ? v : mk<double>(0.0, 0.0);
        f[q] = live ? ib[q] : 1.0;
      } else {
        r[q] = live ? mk<double>(v.x * ib[q], v.y * ib[q]) : mk<double>(0.0, 0.0);
        f[q] = below(j) * (live ? ib[q] : 0.0);
      }
    }
  };
  auto out = [&](int j, int jw, cx<double> p, cx<double>) {
    if (store) put_row(ph, j, jw, psu, (unsigned)o, p);
  };
  // above the diagonal 1/dz^2 as below; 1 in the wall row (bet = -1), nothing in the lid row
  if constexpr (DIV) {
    __shared__ cx<double> end[kPsModes];
    auto num = [&](int j, double rj, double v) {  // the mean's rows carry H_z
      return mean && j > 1 && j < nz ? v + rj * dz : rj - below(j) * v;
    };
    auto above = [&](int j) { return mean || j >= nz || !live ? 0.0 : j == 0 ? 1.0 : idz2; };
    seg_solve_serial<S, RNDS>(end, s, l, nz + 1, load, num, above, out, r, f, ph + o, psu);
  } else {
    __shared__ SegLds<S> L;
    auto fb = [&](int j, double fj) { return mean || j == nz || !live ? 0.0 : j == 0 ? -1.0 : fj; };
    seg_solve<S, RNDS>(L, s, l, nz + 1, load, fb, out, r, f, ph + o, psu);
  }
  if (bad) atomicExch(err, 1);
}

// The same, transposed.  Input spectra (forward y transforms of the r2c, pitch `pitch`
// complex per row): Sp[j] of the adjoint of p (planes 0..nz-1), Sx[j-1], Sy[j-1] of the
// adjoints of dpdx, dpdy (j = 1..nz-1).  The adjoint of p_hat is W (Sp - i kx Sx - i ky Sy),
// W = 2 on the interior kx (c2r^T).  The transposed system A^T lambda = that is solved; the
// mean mode is a reverse cumulative sum.  Outputs, already multiplied by the halving of the
// interior kx (r2c^T) and the forward scales (cst/(1.5 dt) for H, cst for the wall and lid
// rows): Hx, Hy, Hz planes 0..nz-2 (H levels 1..nz-1), bw, tw one plane each.  lam: scratch,
// planes 0..nz.
template <int S, bool RNDS>
__global__ __launch_bounds__(kPsModes *S) void k_press_adj(
    const cx<double> *__restrict__ Sp, const cx<double> *__restrict__ Sx, const cx<double> *__restrict__ Sy,
    const double *__restrict__ kxt, const double *__restrict__ kyt, cx<double> *__restrict__ Hx,
    cx<double> *__restrict__ Hy, cx<double> *__restrict__ Hz, cx<double> *__restrict__ bw,
    cx<double> *__restrict__ tw, const double *__restrict__ tab, cx<double> *lam, int lh, int ny, int nz,
    long pitch, double dz, double sH, double sB) {
  __shared__ SegLds<S> L;
  const int l = threadIdx.x % kPsModes, s = threadIdx.x / kPsModes;
  const long ps = pitch * ny;
  const long o = (long)blockIdx.x * kPsModes + l;
  const int jy = (int)(o / pitch), jx = (int)(o % pitch);
  const bool store = jx < lh;
  const bool live = jx < lh - 1 && jy != ny / 2;
  const bool mean = o == 0;
  const unsigned ocu = live ? (unsigned)o : 0u, psu = (unsigned)ps;
  const long m = (long)jy * lh + (store ? jx : 0);
  const double W = (jx == 0) ? 1.0 : 2.0, h = (jx == 0) ? 1.0 : 0.5;
  const double kx = kxt[m], ky = kyt[m];
  const double idz2 = 1.0 / (dz * dz);
  const cx<double> z0 = mk<double>(0.0, 0.0);
  cx<double> r[kPsRows];
  double f[kPsRows];
  auto load = [&](int j0, int jw, int Lr) {
    cx<double> a[kPsRows], b[kPsRows];
    double ib[kPsRows];
    const int pw = press_plane(jw, nz), tw0 = jw > nz ? nz : jw, sw0 = jw > nz - 1 ? nz - 1 : jw;
    auto row_of = [&](int q) {
      const int j = j0 + (q < Lr ? q : Lr - 1);
      return j > nz ? nz : j;
    };
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) {
      const int j = row_of(q);
      ib[q] = at_row(tab, j, tw0, psu, ocu);  // bet
      r[q] = at_row(Sp, j < nz ? j : nz - 1, sw0, psu, ocu);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) a[q] = at_row(Sx, press_plane(row_of(q), nz), pw, psu, ocu);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) b[q] = at_row(Sy, press_plane(row_of(q), nz), pw, psu, ocu);
#pragma unroll
    for (int q = 0; q < kPsRows; ++q) {
      const int j = row_of(q);
      cx<double> v = r[q];
      if (j >= 1)  // -i kx a - i ky b
        v = mk<double>(v.x + kx * a[q].y + ky * b[q].y, v.y - kx * a[q].x - ky * b[q].x);
      v = mk<double>(W * v.x, W * v.y);
      if (j >= nz || !live) v = z0;
      ib[q] = mean ? 1.0 : 1.0 / ib[q];
      // A^T: below the diagonal c(j-1), 1 under the wall row, 1/dz^2 elsewhere
      r[q] = live ? mk<double>(v.x * ib[q], v.y * ib[q]) : z0;
      f[q] = mean || j == 0 || !live ? 0.0 : j == 1 ? ib[q] : idz2 * ib[q];
    }
  };
  // above the diagonal a(j+1): 1/dz^2, -1 over the lid row; the mean mode
  // lambda(j) = r(j) + lambda(j+1)
  auto fb = [&](int j, double fj) {
    if (mean) return -1.0;
    if (!live || j == nz) return 0.0;
    return j == 0 ? -idz2 : j == 1 ? idz2 * fj : j == nz - 1 ? -(dz * dz) * fj : fj;
  };
  auto out = [&](int j, int, cx<double> lj, cx<double> nxt) {
    if (!store) return;
    if (mean) {  // :303-312: p(1) = -dz bw, p(j) = p(j-1) + dz Hz(j)
      if (j == nz) tw[o] = z0;
      if (j >= 1 && j < nz) {
        const long q = (long)(j - 1) * ps + o;
        Hx[q] = z0;
        Hy[q] = z0;
        // H level 1 of the mean mode is not read by the forward
        Hz[q] = j >= 2 ? mk<double>(h * sH * dz * lj.x, h * sH * dz * lj.y) : z0;
      }
      if (j == 0) bw[o] = mk<double>(h * sB * -dz * nxt.x, h * sB * -dz * nxt.y);
      return;
    }
    if (j == nz) tw[o] = mk<double>(h * sB * -dz * lj.x, h * sB * -dz * lj.y);
    if (j >= 1 && j < nz) {  // row j: i (kx Hx(j) + ky Hy(j)) + (Hz(j+1) - Hz(j))/dz
      const long q = (long)(j - 1) * ps + o;
      Hx[q] = mk<double>(h * sH * kx * lj.y, h * sH * -kx * lj.x);  // -i kx lambda
      Hy[q] = mk<double>(h * sH * ky * lj.y, h * sH * -ky * lj.x);
    }
    if (j <= nz - 2) {  // Hz(j+1): +lambda(j)/dz from row j (j >= 1), -lambda(j+1)/dz from row j+1
      const double ax = (j >= 1 ? lj.x : 0.0) - nxt.x, ay = (j >= 1 ? lj.y : 0.0) - nxt.y;
      Hz[(long)j * ps + o] = mk<double>(h * sH * ax / dz, h * sH * ay / dz);
    }
    if (j == 0) bw[o] = mk<double>(h * sB * -dz * lj.x, h * sB * -dz * lj.y);
  };
  seg_solve<S, RNDS>(L, s, l, nz + 1, load, fb, out, r, f, lam + o, psu);
}

}  // namespace lp
