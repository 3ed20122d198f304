// lp_fft.hip -- batched plane FFT passes for gfx950.
//
// A 2-D real transform of an (ld,ny) plane (FFTW2 rfftwnd in-place layout,
// fft.f90:35-46) is split into
//   row_r2c : each x-row of 2M reals -> M+1 complex (half-length complex FFT + split)
//   col_op  : per kx column, complex FFT along y, a spectral map, inverse FFT along y
//   row_c2r : M+1 complex -> 2M reals (merge + half-length inverse FFT), using only the
//             real parts of the kx = 0 and kx = M terms (FFTW2 halfcomplex semantics)
// Every transform is a register-resident four-step FFT (lp_fft4.hpp) with one LDS
// exchange; loads and stores go straight between HBM and registers.
#include <hip/hip_ext.h>

#include <climits>

#include "lp_fft4.hpp"
#include "lp_internal.hpp"

#pragma clang fp contract(off)  // see lp_device.hpp

namespace lp {

// c2r block: 256 threads; 128 in binary64, whose slots (16-byte values) would otherwise
// take 88 KB of LDS per block and leave one block per CU
template <typename T> __host__ __device__ constexpr int row_block() { return sizeof(T) == 8 ? 128 : 256; }

// XCD-aware plane order for the binary64 passes.  Workgroup ids are dealt round-robin to
// the 8 XCDs, each with its own L2.  The column pass and the back-transform give plane p to
// XCD p mod 8, so that a plane written by one is read by the other on the same XCD; the
// column pass takes an XCD's planes last first, the back-transform first first (the
// column pass wrote those last).  In binary32 the same order measured slightly slower
// (its planes are half the size, and more of them are served from the cache behind L2).
// xcd_planes(n, j): the planes of XCD j.
__host__ __device__ constexpr int xcd_planes(int nplanes, int j) { return (nplanes - j + 7) / 8; }
template <typename T> __host__ __device__ constexpr bool xcd_order() { return sizeof(T) == 8; }
static constexpr int kR2cBlock = 128;  // r2c: persistent blocks of 128 threads

template <typename T> __host__ __device__ constexpr bool r2c_persistent() { return sizeof(T) == 4; }

// grid of the r2c pass: persistent (8 blocks per compute unit, at most one per group) or
// one block per group
static unsigned r2c_grid(long ngroups, bool persistent) {
  if (!persistent) return (unsigned)ngroups;
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
      cus = n;
    else
      cus = 256;
  }
  const long g = 8L * cus;
  return (unsigned)(ngroups < g ? ngroups : g);
}

// ---------------------------------------------------------------------------------
// Sets of a launch.  `first` is the first plane of each set in the launch (INT_MAX past the
// last set); a plane's set is found by comparing, on scalars: every wavefront's rows lie in
// one plane (64/P divides the rows of a plane), every column block's columns too.  What a block
// needs of its set lies together, and a launch of one set is a kernel of its own (N = 1) with
// no search and an eighth of the arguments: as one kernel, a lone 64 x 64 plane took 0.5 to
// 2.4 us more in its three passes.
// ---------------------------------------------------------------------------------
template <typename Set, int N> struct Sets {
  int first[N];
  Set s[N];
  __device__ __forceinline__ int of(int plane) const {
    int f = 0;
#pragma unroll
    for (int i = 1; i < N; ++i) f += plane >= first[i] ? 1 : 0;
    return f;
  }
};
template <typename T, typename TI> struct R2cArg {
  const TI *in;
  cx<T> *out;
  TI scale;
  int flag;  // 1: shifted; vorticity: 1 negated, 2 averaged on plane 0
  const T *b;
  double *shift_out;
};
template <typename T, typename TO> struct C2rArg {
  const cx<T> *in;
  TO *out;
  int np;
  int w;  // div: 1 the w-node form
  const TO *tz;
};

// ---------------------------------------------------------------------------------
// row_r2c: real rows of 2M values -> M+1 complex (half-length complex FFT + split)
// ---------------------------------------------------------------------------------
// VORT: the rows are a vorticity component formed from two derivative volumes (convec.f90:
// 100-133): w_y - v_z, u_z - w_x, v_x - u_y; on plane 0 (jz = 1) w_y and w_x are averaged with
// plane 1 onto the uvp node.  b has in's layout.
// TI is the type of `in` (binary64 velocities into a binary32 transform); there, a shifted
// set's rows enter as (in - in[plane, 0, 0]) * scale, which only moves the plane's kx = ky = 0
// mode; the row y = 0 stores that value in shift_out[plane] when shift_out is given.
template <typename T, int M, int N, bool VORT = false, typename TI = T>
__global__ __launch_bounds__(kR2cBlock) void k_row_r2c(Sets<R2cArg<T, TI>, N> A, long in_pitch, long in_plane, unsigned rows,
                                                       unsigned total, long out_pitch, long out_plane, int ncols_out,
                                                       const cx<T> *__restrict__ twM,
                                                       const cx<T> *__restrict__ twN) {
  constexpr int P = row_lanes(M);
  using F = Fft4<T, M, P, -1>;
  constexpr int Q = F::Q;
  static_assert(kR2cBlock % P == 0, "every thread of the block belongs to a row slot");
  constexpr int RB = kR2cBlock / P;
  constexpr int SS = slot_stride(F::SCR > M ? F::SCR : M);
  __shared__ cx<T> lds[RB * SS];
  __shared__ cx<T> tws[2 * M + 1];  // twM[0..M), twN[0..M]: read from LDS by every group
  const int t = threadIdx.x % P, r = threadIdx.x / P;
  const unsigned ngroups = (total + RB - 1) / RB;
  cx<T> *sc = lds + r * SS;
  for (int i = threadIdx.x; i <= 2 * M; i += kR2cBlock) tws[i] = i < M ? twM[i] : twN[i - M];
  __syncthreads();
  using v2 = typename V2<T>::t;
  // plane of this wavefront's rows in group g, and the row (beyond the last: row 0 of plane 0,
  // not stored)
  auto where = [&](unsigned g, unsigned &y) -> int {
    const unsigned grow = g * RB + r;
    const unsigned pl = grow < total ? grow / rows : 0;
    y = grow < total ? grow - pl * rows : 0;
    return __builtin_amdgcn_readfirstlane((int)pl);
  };
  auto load = [&](unsigned g, cx<T> (&v)[Q]) {
    unsigned y;
    const int pg = where(g, y);
    const int f = A.of(pg), plane = pg - A.first[f];
    const R2cArg<T, TI> &S = A.s[f];
    const TI scale = S.scale;
    if constexpr (!VORT) {
      using vi2 = typename V2<TI>::t;
      const TI *src0 = S.in + (long)plane * in_plane;
      const TI *src = src0 + y * in_pitch;
      TI s0 = TI(0);
      if constexpr (sizeof(TI) > sizeof(T)) s0 = S.flag ? src0[0] : TI(0);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const vi2 p = *reinterpret_cast<const vi2 *>(src + 2 * (t + P * q));
        if constexpr (sizeof(TI) > sizeof(T))
          v[q] = mk<T>((T)((p.x - s0) * scale), (T)((p.y - s0) * scale));
        else
          v[q] = mk<T>((T)(p.x * scale), (T)(p.y * scale));
      }
      if constexpr (sizeof(TI) > sizeof(T)) {
        if (S.shift_out && g * RB + r < total && y == 0 && t == 0) S.shift_out[plane] = (double)s0;
      }
    } else {
      const long o = (long)plane * in_plane + y * in_pitch;
      const bool avg = (S.flag & 2) && plane == 0, neg = S.flag & 1;
      const long up = avg ? in_plane : 0;  // clamped: same row above jz = 1
      const T *pa = S.in + o, *pb = S.b + o;
      const T h = T(0.5);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int x = 2 * (t + P * q);
        const v2 a0 = *reinterpret_cast<const v2 *>(pa + x);
        const v2 b0 = *reinterpret_cast<const v2 *>(pb + x);
        const v2 a1 = *reinterpret_cast<const v2 *>(pa + x + up);
        const v2 av{h * (a0.x + a1.x), h * (a0.y + a1.y)};
        const v2 aa = avg ? av : a0;
        const v2 rr = neg ? v2{b0.x - aa.x, b0.y - aa.y} : v2{aa.x - b0.x, aa.y - b0.y};
        v[q] = mk<T>(rr.x * scale, rr.y * scale);
      }
    }
  };
  // binary32: persistent blocks, the next group's loads issued before this group's
  // transform; binary64 (twice the registers per value): one group per block
  constexpr bool PF = r2c_persistent<T>();
  unsigned g = blockIdx.x;
  cx<T> v[Q];
  if (PF && g < ngroups) load(g, v);
  for (; g < ngroups; g += gridDim.x) {
    cx<T> vn[Q];
    if (!PF) load(g, v);
    else if (g + gridDim.x < ngroups) load(g + gridDim.x, vn);
    F::stage1(v, t, sc, tws);
    slot_sync<P>();
    cx<T> a[F::G][P];
    bool ok[F::G];
#pragma unroll
    for (int j = 0; j < F::G; ++j) ok[j] = F::stage2(j, t, sc, a[j]);
    slot_sync<P>();
#pragma unroll
    for (int j = 0; j < F::G; ++j)
      if (ok[j]) {
#pragma unroll
        for (int k1 = 0; k1 < P; ++k1) sc[t + P * j + Q * k1] = a[j][k1];
      }
    slot_sync<P>();
    if (g * RB + r < total) {
      unsigned y;
      const int pg = where(g, y);
      const int f = A.of(pg);
      cx<T> *dst = A.s[f].out + (long)(pg - A.first[f]) * out_plane + y * out_pitch;
      for (int k = t; k <= M && k < ncols_out; k += P) {
        dst[k] = split_r2c<false>(sc[k % M], sc[(M - k) % M], tws[M + k]);
      }
    }
    if (!PF) break;
    slot_sync<P>();
#pragma unroll
    for (int q = 0; q < Q; ++q) v[q] = vn[q];
  }
}

// ---------------------------------------------------------------------------------
// row_c2r: M+1 complex (first ncols_in present; imaginary parts of kx = 0 and kx = M
// ignored, as FFTW2's halfcomplex c2r) -> 2M reals, columns [2M, out_pitch) zeroed
// ---------------------------------------------------------------------------------
// DIV: what is stored is, per set, (divstress_uv.f90:88-89,116-125) the transform plus
// dz^-1 (tz(k+1) - tz(k)), BOGUS on the top level; or (w: divstress_w.f90:35, 46-81 with the
// wall at level 1 and no lid term) the transform plus dz^-1 (tz(k) - tz(k-1)) on levels
// 1..nz-2.  The padding columns are zero (BOGUS on the uv top level).  tz has the layout of
// out.  IKX: the input is multiplied by i*ikx[kx] first, which turns the (kx, y) spectrum of f
// into that of df/dx (ddx.f90:15-24; kx is uniform along y).
template <typename T, typename TO, int M, int N, bool DIV, bool IKX = false>
__global__ __launch_bounds__(row_block<T>()) void k_row_c2r(Sets<C2rArg<T, TO>, N> A, long in_pitch, long in_plane,
                                                       int ncols_in, unsigned rows, unsigned total, long out_pitch,
                                                       long out_plane, const cx<T> *__restrict__ twM,
                                                       const cx<T> *__restrict__ twN, TO cst,
                                                       const double *__restrict__ ikx, int xorder) {
  constexpr int P = row_lanes(M);
  using F = Fft4<T, M, P, +1>;
  constexpr int Q = F::Q;
  static_assert(row_block<T>() % P == 0, "every thread of the block belongs to a row slot");
  constexpr int RB = row_block<T>() / P;
  constexpr int SS = slot_stride(F::SCR);
  __shared__ cx<T> lds[RB * SS];
  __shared__ cx<T> tws[2 * M];  // twM[0..M), twN[0..M): read from LDS by every row
  const int t = threadIdx.x % P, r = threadIdx.x / P;
  int f, plane;
  unsigned y;
  bool valid;
  if (xorder) {  // XCD order, first-written planes first; the grid has 8 groups gpp blocks
    const unsigned gpp = rows / RB, xi = blockIdx.x >> 3;
    const int gq = (int)(xi / gpp);
    f = A.of(gq);
    plane = (int)(blockIdx.x & 7u) + 8 * (gq - A.first[f]);
    if (plane >= A.s[f].np) return;  // uniform over the block
    y = (xi % gpp) * RB + r;
    valid = true;
  } else {
    const unsigned grow = blockIdx.x * RB + r;
    valid = grow < total;
    const unsigned pl = valid ? grow / rows : 0;
    y = valid ? grow - pl * rows : 0;
    const int pg = __builtin_amdgcn_readfirstlane((int)pl);
    f = A.of(pg);
    plane = pg - A.first[f];
  }
  const C2rArg<T, TO> &S = A.s[f];
  const int nplanes = S.np;
  cx<T> *sc = lds + r * SS;
  const cx<T> *src = S.in + (long)plane * in_plane + y * in_pitch;
  for (int i = threadIdx.x; i < 2 * M; i += row_block<T>()) tws[i] = i < M ? twM[i] : twN[i - M];
  __shared__ T ikxs[IKX ? M + 1 : 1];  // the multipliers, in the transform's type
  if constexpr (IKX)
    for (int i = threadIdx.x; i <= M; i += row_block<T>()) ikxs[i] = (T)ikx[i];
  auto ld = [&](int k) -> cx<T> {
    cx<T> x = (valid && k < ncols_in) ? src[k] : mk<T>(0, 0);
    if (k == 0 || k == M) x.y = 0;
    return x;
  };
  __syncthreads();  // the twiddles
  cx<T> v[Q];
  if constexpr (IKX) {  // i kx X[k]: the kx = 0 and kx = M entries of the table are zero
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int k = t + P * q;
      const T sa = ikxs[k], sb = ikxs[M - k];
      const cx<T> ra = ld(k), rb = ld(M - k);
      v[q] = merge_c2r<false>(mk<T>(-ra.y * sa, ra.x * sa), mk<T>(-rb.y * sb, rb.x * sb), tws[M + k]);
    }
  } else {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int k = t + P * q;
      v[q] = merge_c2r<false>(ld(k), ld(M - k), tws[M + k]);
    }
  }
  F::stage1(v, t, sc, tws);
  slot_sync<P>();
  const long od = (long)plane * out_plane + y * out_pitch;
  TO *dst = S.out + od;
  const bool top = plane == nplanes - 1;
  const bool mid = plane >= 1 && plane <= nplanes - 2;
  const bool isw = DIV && S.w;
  // neighbour levels, clamped: uv k + 1 and k, w k and k - 1
  const TO *tzr = DIV ? S.tz + od : nullptr;
  const long up = isw || top ? 0 : out_plane, dn = isw && mid ? out_plane : 0;
#pragma unroll
  for (int j = 0; j < F::G; ++j) {
    cx<T> a[P];
    if (F::stage2(j, t, sc, a) && valid) {
      if constexpr (DIV) {
        // tz first: the compiler, which cannot tell it from the output, would wait for each
        // value's loads between two stores
        TO z[P][2];
#pragma unroll
        for (int k1 = 0; k1 < P; ++k1)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int x = 2 * (t + P * j + Q * k1) + h;
            z[k1][h] = tzr[x + up] - tzr[x - dn];
          }
#pragma unroll
        for (int k1 = 0; k1 < P; ++k1)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const TO v = h ? (TO)a[k1].y : (TO)a[k1].x, r = fmadd(cst, z[k1][h], v);
            dst[2 * (t + P * j + Q * k1) + h] = isw ? (mid ? r : v) : (top ? (TO)LP_BOGUS : r);
          }
      } else {
#pragma unroll
        for (int k1 = 0; k1 < P; ++k1) {
          const int n = t + P * j + Q * k1;
          dst[2 * n] = (TO)a[k1].x;
          dst[2 * n + 1] = (TO)a[k1].y;
        }
      }
    }
  }
  if (valid) {
    const TO pad = (DIV && !isw && top) ? (TO)LP_BOGUS : (TO)0;
    for (long n = 2 * M + t; n < out_pitch; n += P) dst[n] = pad;
  }
}

// ---------------------------------------------------------------------------------
// col_op: per kx column, forward DFT along y, spectral map, inverse DFT along y.
// A block owns TX adjacent columns (one 128-byte segment per y) of one plane; 16 lanes
// per column.  The spectrum between the transforms stays in registers in the
// "D16" layout: lane t holds entries t + 16*m, which is also what the padding,
// truncation and multiplier maps need, so they are lane-local.
// ---------------------------------------------------------------------------------
struct ColSlot {
  void *ptr;
  double scale;  // factor on the padded / truncated spectrum (padmode 1, 2)
  int pitch;     // complex elements between y rows of this output
  int plane;     // complex elements between planes of this output
  int mult;
  int ncols;     // columns stored (kx < ncols)
};
struct ColArg {
  const void *in;
  const double *dc;
  int np, nout;
  ColSlot outs[3];
};
static constexpr int kColLanes = 16;
template <typename T> __host__ __device__ constexpr int col_tx() { return 128 / (int)sizeof(cx<T>); }
// LDS stride of a column slot.  The 16 lanes of a quarter wavefront are 16 (8 in binary64)
// different columns at the same row offset, so an odd stride puts them on different banks.
__host__ __device__ constexpr int col_slot_stride(int n) { return n | 1; }

// forward DFT of length NY along a column held in the D16 layout (sp[m] = x[t + 16 m]),
// result in the same layout; sc is the column's LDS slot (block-wide barriers)
template <typename T, int NY>
__device__ __forceinline__ void col_forward(cx<T> (&sp)[NY / kColLanes], int t, cx<T> *sc,
                                            const cx<T> *__restrict__ twI) {
  constexpr int PL = kColLanes;
  using FI = Fft4<T, NY, PL, -1>;
  constexpr int QI = FI::Q;
  FI::stage1(sp, t, sc, twI);
  __syncthreads();
  if constexpr (QI == PL) {  // stage 2 already yields the D16 layout
    cx<T> a[PL];
    FI::stage2(0, t, sc, a);
#pragma unroll
    for (int k1 = 0; k1 < PL; ++k1) sp[k1] = a[k1];
    __syncthreads();
  } else {  // regroup through LDS in natural order
    cx<T> a[FI::G][PL];
    bool ok[FI::G];
#pragma unroll
    for (int j = 0; j < FI::G; ++j) ok[j] = FI::stage2(j, t, sc, a[j]);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < FI::G; ++j)
      if (ok[j]) {
#pragma unroll
        for (int k1 = 0; k1 < PL; ++k1) sc[t + PL * j + QI * k1] = a[j][k1];
      }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < QI; ++m) sp[m] = sc[t + PL * m];
    __syncthreads();
  }
}

// TX columns per block (16 for binary32, 8 for binary64: one 128-byte run per y); TX = 1
// serves a single trailing column.  Block column c handles kx = col0 + blockIdx.x*TX + c.
template <typename T, int NYI, int NYO, int N, int TX = col_tx<T>()>
__global__ __launch_bounds__(TX * kColLanes) void k_col_op(
    Sets<ColArg, N> Pr, int ngroups, long in_pitch, long in_plane, int ncols, int fwd, int inv, const double *__restrict__ kxt, const double *__restrict__ kyt,
    const double *__restrict__ G1, const double *__restrict__ G2, int lh_s, int ny_s,
    const cx<T> *__restrict__ twI, const cx<T> *__restrict__ twO, int col0) {
  constexpr int PL = kColLanes;
  using FI = Fft4<T, NYI, PL, -1>;
  using FO = Fft4<T, NYO, PL, +1>;
  constexpr int QI = FI::Q, QO = FO::Q;
  constexpr int PM = NYI == NYO ? 0 : (NYO > NYI ? 1 : 2);  // same grid / pad / truncate
  constexpr int DQ = (NYI > NYO ? NYI - NYO : NYO - NYI) / PL;
  constexpr int NS = FI::SCR > FO::SCR ? (FI::SCR > NYI ? FI::SCR : NYI) : (FO::SCR > NYI ? FO::SCR : NYI);
  constexpr int SS = col_slot_stride(NS);
  // binary32: the twiddles are read from LDS (staged once per workgroup), which also
  // lowers the register count; binary64 keeps the slots' LDS to itself and reads the tables
  constexpr bool TWL = sizeof(T) == 4;
  __shared__ cx<T> lds[TX * SS + (TWL ? NYI + NYO : 0)];
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  int plane = blockIdx.y, cg = blockIdx.x, f;
  if constexpr (xcd_order<T>()) {  // last-written planes first; the grid has gx x 8 groups blocks
    const int gx = gridDim.x;
    const long lin = blockIdx.x + (long)gx * blockIdx.y;
    const int gq = ngroups - 1 - (int)((lin >> 3) / gx);
    f = Pr.of(gq);
    plane = (int)(lin & 7) + 8 * (gq - Pr.first[f]);
    if (plane >= Pr.s[f].np) return;  // uniform over the block
    cg = (int)((lin >> 3) % gx);
  } else {
    f = Pr.of(plane);
    plane -= Pr.first[f];
  }
  const int kx = col0 + cg * TX + c;
  const bool cv = kx < ncols;
  cx<T> *sc = lds + c * SS;
  if constexpr (TWL) {
    cx<T> *tl = lds + TX * SS;
    for (int i = threadIdx.x; i < NYI + NYO; i += TX * kColLanes) tl[i] = i < NYI ? twI[i] : twO[i - NYI];
    twI = tl;
    twO = tl + NYI;
    __syncthreads();
  }
  // invalid columns load column ncols-1 and discard it (no divergent loads)
  const cx<T> *src = reinterpret_cast<const cx<T> *>(Pr.s[f].in) + (long)plane * in_plane + (cv ? kx : ncols - 1) +
                     (long)t * in_pitch;
  const long istep = (long)PL * in_pitch;
  cx<T> sp[QI];  // D16: sp[m] = spectrum[t + 16 m]
#pragma unroll
  for (int m = 0; m < QI; ++m) {
    const cx<T> x = src[m * istep];
    sp[m] = cv ? x : mk<T>(0, 0);
  }
  if constexpr (PM == 1) {
    if (Pr.s[f].dc && kx == 0) {
      const double dc = Pr.s[f].dc[plane];
#pragma unroll
      for (int m = 0; m < QI; ++m) sp[m].x = (T)((double)sp[m].x + dc);
    }
  }
  if (fwd) col_forward<T, NYI>(sp, t, sc, twI);
  const int nout = Pr.s[f].nout;
  const ColSlot *outs = Pr.s[f].outs;
  for (int jo = 0; jo < nout; ++jo) {
    const int mult = outs[jo].mult;
    // one multiplier table per output: i*kx, i*ky (imaginary) or a filter (real)
    const double *mt = mult == M_IKX ? kxt : mult == M_IKY ? kyt : mult == M_G1 ? G1 : G2;
    const bool imag = mult == M_IKX || mult == M_IKY;
    const bool keep = cv && kx != lh_s - 1;
    const int tp = lh_s;  // row length of the multiplier tables
    const double *mrow = mt + (long)t * tp + (cv ? kx : 0);
    cx<T> v[QO];
    if constexpr (PM == 0) {
      // the multipliers of all q are loaded together (block-uniform branch)
      T fq[QO];
      if (mult != M_ONE) {
#pragma unroll
        for (int q = 0; q < QO; ++q) fq[q] = (T)mrow[(long)q * PL * tp];
      }
#pragma unroll
      for (int q = 0; q < QO; ++q) {
        const int yo = t + PL * q;
        cx<T> x = sp[q];
        if (mult != M_ONE) x = mk<T>((imag ? -x.y : x.x) * fq[q], (imag ? x.x : x.y) * fq[q]);
        v[q] = (!keep || yo == ny_s / 2) ? mk<T>(0, 0) : x;
      }
    }
    if constexpr (PM != 0) {
      const T osc = (T)outs[jo].scale;
      const bool scaled = outs[jo].scale != 1.0;
#pragma unroll
      for (int q = 0; q < QO; ++q) {
        const int yo = t + PL * q;
        cx<T> x = mk<T>(0, 0);
        if constexpr (PM == 1) {  // padd.f90: ny -> ny2, middle rows zero
          if (q < QI && yo < NYI / 2) x = sp[q < QI ? q : 0];
          else if (q >= DQ && yo >= NYO - NYI / 2 + 1) x = sp[q >= DQ ? q - DQ : 0];
        } else {  // unpadd.f90: ny2 -> ny, Nyquist row zero
          if (yo < NYO / 2) x = sp[q];
          else if (yo > NYO / 2) x = sp[q + DQ];
        }
        v[q] = scaled ? mk<T>(x.x * osc, x.y * osc) : x;
      }
    }
    // addresses are formed from per-output values so that they are not hoisted out of
    // the output loop (which would keep 16 64-bit addresses live)
    const long pitch = outs[jo].pitch;
    const bool st = cv && kx < outs[jo].ncols;
    cx<T> *dst = reinterpret_cast<cx<T> *>(outs[jo].ptr) + (long)plane * outs[jo].plane + kx;
    if (inv) {
      FO::stage1(v, t, sc, twO);
      __syncthreads();
#pragma unroll
      for (int j = 0; j < FO::G; ++j) {
        cx<T> a[PL];
        if (FO::stage2(j, t, sc, a) && st) {
          cx<T> *d = dst + (long)(t + PL * j) * pitch;
          const long ostep = (long)QO * pitch;
#pragma unroll
          for (int k1 = 0; k1 < PL; ++k1) d[k1 * ostep] = a[k1];
        }
      }
      __syncthreads();
    } else if (st) {
      cx<T> *d = dst + (long)t * pitch;
      const long ostep = (long)PL * pitch;
#pragma unroll
      for (int q = 0; q < QO; ++q) d[q * ostep] = v[q];
    }
  }
}

// ---------------------------------------------------------------------------------
// col_div: the x- and y-derivative terms of divstress_uv.f90 / divstress_w.f90 summed in
// spectral space.  Per kx column: forward y DFTs of the x-spectra A and B, then
// i kx A + i ky B with the Nyquist row and column zeroed (the ddx / ddy multipliers),
// inverse y DFT into out.
// ---------------------------------------------------------------------------------
struct DivSets {
  DivSet s[kMaxSets];
};
template <typename T, int NY>
__global__ __launch_bounds__(col_tx<T>() * kColLanes) void k_col_div(
    DivSets D, int nplanes, long pitch, long plane_el, int ncols, const double *__restrict__ kxt, const double *__restrict__ kyt, int lh_s, int ny_s,
    const cx<T> *__restrict__ tw) {
  constexpr int TX = col_tx<T>();
  constexpr int PL = kColLanes;
  using FO = Fft4<T, NY, PL, +1>;
  constexpr int Q = NY / PL;
  constexpr int SS = col_slot_stride(FO::SCR > NY ? FO::SCR : NY);
  constexpr bool TWL = (TX * SS + NY) * sizeof(cx<T>) <= 40960;  // as in k_col_op
  __shared__ cx<T> lds[TX * SS + (TWL ? NY : 0)];
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const int kx = blockIdx.x * TX + c;
  const bool cv = kx < ncols;
  const int f = blockIdx.y / nplanes;
  const long plane = blockIdx.y % nplanes;
  const cx<T> *A = reinterpret_cast<const cx<T> *>(D.s[f].A), *B = reinterpret_cast<const cx<T> *>(D.s[f].B);
  cx<T> *out = reinterpret_cast<cx<T> *>(D.s[f].out);
  cx<T> *sc = lds + c * SS;
  if constexpr (TWL) {
    cx<T> *tl = lds + TX * SS;
    for (int i = threadIdx.x; i < NY; i += TX * kColLanes) tl[i] = tw[i];
    tw = tl;
    __syncthreads();
  }
  const long off = plane * plane_el + (cv ? kx : ncols - 1) + (long)t * pitch;
  const long istep = (long)PL * pitch;
  cx<T> sa[Q], sb[Q];  // D16
#pragma unroll
  for (int m = 0; m < Q; ++m) {
    sa[m] = A[off + m * istep];
    sb[m] = B[off + m * istep];
  }
  col_forward<T, NY>(sa, t, sc, tw);
  col_forward<T, NY>(sb, t, sc, tw);
  const bool keep = cv && kx != lh_s - 1;
  const long mo = (long)t * lh_s + (cv ? kx : 0);
  T fx[Q], fy[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    fx[q] = (T)kxt[mo + (long)q * PL * lh_s];
    fy[q] = (T)kyt[mo + (long)q * PL * lh_s];
  }
  cx<T> v[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int yo = t + PL * q;
    const cx<T> a = sa[q], b = sb[q];
    const cx<T> x = mk<T>(fmadd(-a.y, fx[q], -b.y * fy[q]), fmadd(a.x, fx[q], b.x * fy[q]));
    v[q] = (!keep || yo == ny_s / 2) ? mk<T>(0, 0) : x;
  }
  FO::stage1(v, t, sc, tw);
  __syncthreads();
  cx<T> *dst = out + plane * plane_el + kx;
#pragma unroll
  for (int j = 0; j < FO::G; ++j) {
    cx<T> a[PL];
    if (FO::stage2(j, t, sc, a) && cv) {
      cx<T> *d = dst + (long)(t + PL * j) * pitch;
      const long ostep = (long)Q * pitch;
#pragma unroll
      for (int k1 = 0; k1 < PL; ++k1) d[k1 * ostep] = a[k1];
    }
  }
}

template <typename T, int NY>
static hipError_t launch_col_div(const DivSet *sets, int n, int nplanes, long pitch, long plane, int ncols,
                                 const SpecTables &tab, hipStream_t s, Dt dt) {
  const void *tw = tw_ptr(NY, dt);
  if (!tw || n < 1 || n > kMaxSets || ncols < 1 || ncols > tab.lh || pitch < ncols || tab.ny != NY)
    return hipErrorInvalidValue;
  constexpr int TX = col_tx<T>();
  DivSets D{};
  for (int f = 0; f < n; ++f) D.s[f] = sets[f];
  dim3 grid((unsigned)((ncols + TX - 1) / TX), (unsigned)(n * nplanes));
  hipLaunchKernelGGL((k_col_div<T, NY>), grid, dim3(TX * kColLanes), 0, s, D, nplanes, pitch, plane, ncols, tab.kx,
                     tab.ky, tab.lh, tab.ny, (const cx<T> *)tw);
  return hipGetLastError();
}

hipError_t col_div(Dt dt, int ny, const DivSet *sets, int n, int nplanes, long pitch, long plane, int ncols,
                   const SpecTables &tab, hipStream_t s) {
#define CASE(n_)                                                                                \
  case n_:                                                                                      \
    return dt == F64 ? launch_col_div<double, n_>(sets, n, nplanes, pitch, plane, ncols, tab, s, dt) \
                     : launch_col_div<float, n_>(sets, n, nplanes, pitch, plane, ncols, tab, s, dt);
  switch (ny) {
    CASE(32) CASE(48) CASE(64) CASE(96) CASE(128) CASE(144) CASE(192) CASE(256)
    default: return hipErrorInvalidValue;
  }
#undef CASE
}

// ---------------------------------------------------------------------------------
// dispatch
// ---------------------------------------------------------------------------------
#define LP_ROW_LENGTHS(X) X(16) X(24) X(32) X(48) X(64) X(72) X(96) X(128) X(144) X(192)
#define LP_SMALL_ROW_LENGTHS(X) X(16) X(32) X(48) X(64) X(96) X(128)

bool fft_len_supported(int n) {
  switch (n) {
    case 32: case 48: case 64: case 96: case 128: case 144: case 192: case 256:
    case 288: case 384: return true;
    default: return false;
  }
}

template <typename T, int M, int N, bool VORT, typename TI>
static hipError_t launch_r2c_n(const R2cSet *sets, int n, long in_pitch, long in_plane, int rows, long out_pitch,
                             long out_plane, int ncols_out, hipStream_t s, Dt dt) {
  const void *twM = tw_ptr(M, dt), *twN = tw_ptr(2 * M, dt);
  constexpr int P = row_lanes(M), RPB = kR2cBlock / P;
  if (!twM || !twN || n < 1 || n > N || rows < 1 || rows % (64 / P) != 0) return hipErrorInvalidValue;
  Sets<R2cArg<T, TI>, N> A{};
  long planes = 0;
  for (int f = 0; f < N; ++f) {
    A.first[f] = INT_MAX;
    if (f >= n) continue;
    const R2cSet &x = sets[f];
    if (x.nplanes < 1 || (VORT && (!x.b || x.comp < 0 || x.comp > 2 || x.nplanes < 2))) return hipErrorInvalidValue;
    A.first[f] = (int)planes;
    A.s[f] = R2cArg<T, TI>{(const TI *)x.in, (cx<T> *)x.out, (TI)x.scale,
                           VORT ? (x.comp == 1 ? 1 : 0) | (x.comp < 2 ? 2 : 0) : (x.shift ? 1 : 0), (const T *)x.b,
                           x.shift_out};
    planes += x.nplanes;
  }
  const long total = (long)rows * planes;
  if (total > INT_MAX) return hipErrorInvalidValue;
  dim3 grid(r2c_grid((total + RPB - 1) / RPB, r2c_persistent<T>()));
  hipLaunchKernelGGL((k_row_r2c<T, M, N, VORT, TI>), grid, dim3(kR2cBlock), 0, s, A, in_pitch, in_plane,
                     (unsigned)rows, (unsigned)total, out_pitch, out_plane, ncols_out, (const cx<T> *)twM,
                     (const cx<T> *)twN);
  return hipGetLastError();
}

template <typename T, int M, bool VORT = false, typename TI = T>
static hipError_t launch_r2c(const R2cSet *sets, int n, long in_pitch, long in_plane, int rows, long out_pitch,
                             long out_plane, int ncols_out, hipStream_t s, Dt dt) {
  return n == 1 ? launch_r2c_n<T, M, 1, VORT, TI>(sets, n, in_pitch, in_plane, rows, out_pitch, out_plane, ncols_out,
                                                  s, dt)
                : launch_r2c_n<T, M, kMaxSets, VORT, TI>(sets, n, in_pitch, in_plane, rows, out_pitch, out_plane,
                                                         ncols_out, s, dt);
}

hipError_t row_r2c(Dt dt, Dt din, int M, const R2cSet *sets, int n, long in_pitch, long in_plane, int rows,
                   long out_pitch, long out_plane, int ncols_out, hipStream_t s) {
  if (n < 1 || (dt == F64 && din == F32)) return hipErrorInvalidValue;
  const bool vort = sets[0].comp >= 0;
  for (int f = 0; f < n; ++f)
    if ((sets[f].comp >= 0) != vort || (sets[f].shift && !(dt == F32 && din == F64))) return hipErrorInvalidValue;
  if (vort) {
    if (din != dt) return hipErrorInvalidValue;
#define CASE(m)                                                                                                    \
  case m:                                                                                                          \
    return dt == F64 ? launch_r2c<double, m, true>(sets, n, in_pitch, in_plane, rows, out_pitch, out_plane,        \
                                                   ncols_out, s, dt)                                               \
                     : launch_r2c<float, m, true>(sets, n, in_pitch, in_plane, rows, out_pitch, out_plane,         \
                                                  ncols_out, s, dt);
    switch (M) {
      LP_SMALL_ROW_LENGTHS(CASE)
      default: return hipErrorInvalidValue;
    }
#undef CASE
  }
#define CASE(m)                                                                                                    \
  case m:                                                                                                          \
    if (dt == F64)                                                                                                 \
      return launch_r2c<double, m>(sets, n, in_pitch, in_plane, rows, out_pitch, out_plane, ncols_out, s, dt);     \
    if (din == F32)                                                                                                \
      return launch_r2c<float, m>(sets, n, in_pitch, in_plane, rows, out_pitch, out_plane, ncols_out, s, dt);      \
    return launch_r2c<float, m, false, double>(sets, n, in_pitch, in_plane, rows, out_pitch, out_plane, ncols_out, \
                                               s, dt);
  switch (M) {
    LP_ROW_LENGTHS(CASE)
    default: return hipErrorInvalidValue;
  }
#undef CASE
}

template <typename T, typename TO, int M, int N, bool DIV>
static hipError_t launch_c2r_n(const C2rSet *sets, int n, long in_pitch, long in_plane, int ncols_in, int rows,
                             long out_pitch, long out_plane, hipStream_t s, Dt dt, const double *ikx, double cst) {
  const void *twM = tw_ptr(M, dt), *twN = tw_ptr(2 * M, dt);
  constexpr int P = row_lanes(M), RPB = row_block<T>() / P;
  if (!twM || !twN || n < 1 || n > N || rows < 1 || rows % (64 / P) != 0) return hipErrorInvalidValue;
  const int xorder = xcd_order<T>() && rows % RPB == 0 ? 1 : 0;
  Sets<C2rArg<T, TO>, N> A{};
  long planes = 0, groups = 0;
  for (int f = 0; f < N; ++f) {
    A.first[f] = INT_MAX;
    if (f >= n) continue;
    const C2rSet &x = sets[f];
    if (x.nplanes < 1 || (DIV && (!x.tz || x.nplanes < 2))) return hipErrorInvalidValue;
    A.first[f] = (int)(xorder ? groups : planes);
    A.s[f] = C2rArg<T, TO>{(const cx<T> *)x.in, (TO *)x.out, x.nplanes, x.div == 2 ? 1 : 0, (const TO *)x.tz};
    planes += x.nplanes;
    groups += xcd_planes(x.nplanes, 0);
  }
  const long total = (long)rows * planes;
  if (total > INT_MAX) return hipErrorInvalidValue;
  dim3 grid((unsigned)(xorder ? 8L * groups * (rows / RPB) : (total + RPB - 1) / RPB));
  // the x derivative is its own kernel: the plain transform then holds no multiplier
  // registers
  if (ikx) {
    if constexpr (DIV) return hipErrorInvalidValue;  // no caller asks for both
    else
      hipLaunchKernelGGL((k_row_c2r<T, TO, M, N, DIV, true>), grid, dim3(row_block<T>()), 0, s, A, in_pitch, in_plane,
                         ncols_in, (unsigned)rows, (unsigned)total, out_pitch, out_plane, (const cx<T> *)twM,
                         (const cx<T> *)twN, (TO)cst, ikx, xorder);
  } else
    hipLaunchKernelGGL((k_row_c2r<T, TO, M, N, DIV, false>), grid, dim3(row_block<T>()), 0, s, A, in_pitch, in_plane,
                       ncols_in, (unsigned)rows, (unsigned)total, out_pitch, out_plane, (const cx<T> *)twM,
                       (const cx<T> *)twN, (TO)cst, nullptr, xorder);
  return hipGetLastError();
}

template <typename T, typename TO, int M, bool DIV = false>
static hipError_t launch_c2r(const C2rSet *sets, int n, long in_pitch, long in_plane, int ncols_in, int rows,
                             long out_pitch, long out_plane, hipStream_t s, Dt dt, const double *ikx, double cst) {
  return n == 1 ? launch_c2r_n<T, TO, M, 1, DIV>(sets, n, in_pitch, in_plane, ncols_in, rows, out_pitch, out_plane, s,
                                                 dt, ikx, cst)
                : launch_c2r_n<T, TO, M, kMaxSets, DIV>(sets, n, in_pitch, in_plane, ncols_in, rows, out_pitch,
                                                        out_plane, s, dt, ikx, cst);
}

hipError_t row_c2r(Dt dtc, Dt dto, int M, const C2rSet *sets, int n, long in_pitch, long in_plane, int ncols_in,
                   int rows, long out_pitch, long out_plane, hipStream_t s, const double *ikx, double cst) {
  if (n < 1 || (dtc == F32 && dto == F64)) return hipErrorInvalidValue;
  const bool div = sets[0].div != 0;
  for (int f = 0; f < n; ++f)
    if ((sets[f].div != 0) != div) return hipErrorInvalidValue;
  if (div) {
    if (dtc != dto || ikx || out_pitch < 2 * M) return hipErrorInvalidValue;
#define CASE(m)                                                                                                   \
  case m:                                                                                                         \
    return dtc == F64 ? launch_c2r<double, double, m, true>(sets, n, in_pitch, in_plane, ncols_in, rows,          \
                                                            out_pitch, out_plane, s, dtc, nullptr, cst)           \
                      : launch_c2r<float, float, m, true>(sets, n, in_pitch, in_plane, ncols_in, rows, out_pitch, \
                                                          out_plane, s, dtc, nullptr, cst);
    switch (M) {
      LP_SMALL_ROW_LENGTHS(CASE)
      default: return hipErrorInvalidValue;
    }
#undef CASE
  }
#define CASE(m)                                                                                                     \
  case m:                                                                                                           \
    if (dtc == F64 && dto == F64)                                                                                   \
      return launch_c2r<double, double, m>(sets, n, in_pitch, in_plane, ncols_in, rows, out_pitch, out_plane, s,    \
                                           dtc, ikx, cst);                                                          \
    if (dtc == F64 && dto == F32)                                                                                   \
      return launch_c2r<double, float, m>(sets, n, in_pitch, in_plane, ncols_in, rows, out_pitch, out_plane, s,     \
                                          dtc, ikx, cst);                                                           \
    return launch_c2r<float, float, m>(sets, n, in_pitch, in_plane, ncols_in, rows, out_pitch, out_plane, s, dtc,   \
                                       ikx, cst);
  switch (M) {
    LP_ROW_LENGTHS(CASE)
    default: return hipErrorInvalidValue;
  }
#undef CASE
}

// Planes of a column launch: they lie along y, where the device takes 65536 blocks.  Lists of
// more (the test filters' 21 fields from 3121 levels on) are launched one set and this many
// planes at a time, whole groups of eight.
constexpr int kMaxPlanes = 65528;

// col0 > 0: the columns col0..ncols-1 only (same grid, one column per block)
template <typename T, int NYI, int NYO, int N>
static hipError_t launch_col_n(int padmode, int fwd, int inv, const ColSet *sets, int n, long in_pitch, long in_plane,
                               int ncols, long out_pitch, long out_plane, const SpecTables &tab, hipStream_t s,
                               Dt dt, int col0, LaunchEv ev) {
  const void *twI = tw_ptr(NYI, dt), *twO = tw_ptr(NYO, dt);
  if (!twI || !twO || n < 1 || n > N || col0 < 0 || col0 >= ncols) return hipErrorInvalidValue;
  // the map is fixed by the lengths: same grid (0), padd (1), unpadd (2)
  if (padmode != (NYI == NYO ? 0 : (NYO > NYI ? 1 : 2))) return hipErrorInvalidValue;
  constexpr int TX = col_tx<T>();
  Sets<ColArg, N> P{};
  long planes = 0, groups = 0;
  for (int f = 0; f < N; ++f) {
    P.first[f] = INT_MAX;
    if (f >= n) continue;
    const ColSet &x = sets[f];
    if (x.nplanes < 1 || x.nout < 1 || x.nout > 3 || (x.dc && padmode != 1)) return hipErrorInvalidValue;
    P.first[f] = (int)(xcd_order<T>() ? groups : planes);
    ColArg &A = P.s[f];
    A.in = x.in;
    A.dc = x.dc;
    A.np = x.nplanes;
    A.nout = x.nout;
    for (int j = 0; j < x.nout; ++j) {
      const ColOut &o = x.outs[j];
      if (padmode == 0 && o.scale != 1.0) return hipErrorInvalidValue;
      const long pl = o.plane ? o.plane : out_plane;
      if (pl > INT_MAX) return hipErrorInvalidValue;
      A.outs[j] = ColSlot{o.ptr, o.scale, (int)(o.pitch ? o.pitch : out_pitch), (int)pl, o.mult,
                          o.ncols ? o.ncols : ncols};
    }
    planes += x.nplanes;
    groups += xcd_planes(x.nplanes, 0);
  }
  const unsigned gy = (unsigned)(xcd_order<T>() ? 8 * groups : planes);
  if (col0 > 0) {
    if constexpr (NYI == NYO) {
      hipExtLaunchKernelGGL((k_col_op<T, NYI, NYO, N, 1>), dim3((unsigned)(ncols - col0), gy), dim3(kColLanes), 0, s,
                            ev.start, ev.stop, 0, P, (int)groups, in_pitch, in_plane, ncols, fwd, inv, tab.kx, tab.ky, tab.G1,
                            tab.G2, tab.lh, tab.ny, (const cx<T> *)twI, (const cx<T> *)twO, col0);
      return hipGetLastError();
    } else {
      return hipErrorInvalidValue;
    }
  }
  hipExtLaunchKernelGGL((k_col_op<T, NYI, NYO, N>), dim3((unsigned)((ncols + TX - 1) / TX), gy), dim3(TX * kColLanes), 0,
                        s, ev.start, ev.stop, 0, P, (int)groups, in_pitch, in_plane, ncols, fwd, inv, tab.kx, tab.ky, tab.G1,
                        tab.G2, tab.lh, tab.ny, (const cx<T> *)twI, (const cx<T> *)twO, 0);
  return hipGetLastError();
}

template <typename T, int NYI, int NYO>
static hipError_t launch_col(int padmode, int fwd, int inv, const ColSet *sets, int n, long in_pitch, long in_plane,
                             int ncols, long out_pitch, long out_plane, const SpecTables &tab, hipStream_t s, Dt dt,
                             int col0 = 0, LaunchEv ev = {}) {
  long gy = 0;
  for (int f = 0; f < n; ++f) gy += xcd_order<T>() ? 8L * xcd_planes(sets[f].nplanes, 0) : sets[f].nplanes;
  if (gy > kMaxPlanes) {
    for (int f = 0; f < n; ++f) {
      const int np = sets[f].nplanes;
      int p0 = 0;
      do {
        ColSet x = sets[f];
        x.in = (const cx<T> *)x.in + p0 * in_plane;
        x.nplanes = np - p0 < kMaxPlanes ? np - p0 : kMaxPlanes;
        if (x.dc) x.dc += p0;
        for (int j = 0; j < x.nout && j < 3; ++j)
          x.outs[j].ptr = (cx<T> *)x.outs[j].ptr + p0 * (x.outs[j].plane ? x.outs[j].plane : out_plane);
        const bool last = f == n - 1 && np - p0 <= kMaxPlanes;
        const hipError_t e = launch_col_n<T, NYI, NYO, 1>(
            padmode, fwd, inv, &x, 1, in_pitch, in_plane, ncols, out_pitch, out_plane, tab, s, dt, col0,
            LaunchEv{f == 0 && p0 == 0 ? ev.start : nullptr, last ? ev.stop : nullptr});
        if (e != hipSuccess) return e;
        p0 += kMaxPlanes;
      } while (p0 < np);
    }
    return hipSuccess;
  }
  return n == 1 ? launch_col_n<T, NYI, NYO, 1>(padmode, fwd, inv, sets, n, in_pitch, in_plane, ncols, out_pitch,
                                               out_plane, tab, s, dt, col0, ev)
                : launch_col_n<T, NYI, NYO, kMaxSets>(padmode, fwd, inv, sets, n, in_pitch, in_plane, ncols,
                                                      out_pitch, out_plane, tab, s, dt, col0, ev);
}

hipError_t col_op_tail(Dt dt, int ny, const ColSet &set, long in_pitch, long in_plane, int col0, int ncols,
                       long out_pitch, long out_plane, const SpecTables &tab, hipStream_t s, LaunchEv ev) {
#define CASE(n)                                                                                                  \
  case n:                                                                                                        \
    return dt == F64 ? launch_col<double, n, n>(0, 1, 1, &set, 1, in_pitch, in_plane, ncols, out_pitch,          \
                                                out_plane, tab, s, dt, col0, ev)                                 \
                     : launch_col<float, n, n>(0, 1, 1, &set, 1, in_pitch, in_plane, ncols, out_pitch,           \
                                               out_plane, tab, s, dt, col0, ev);
  switch (ny) {
    CASE(32) CASE(48) CASE(64) CASE(96) CASE(128) CASE(144) CASE(192) CASE(256) CASE(288) CASE(384)
    default: return hipErrorInvalidValue;
  }
#undef CASE
}

hipError_t col_op(Dt dt, int nyi, int nyo, int padmode, int fwd, int inv, const ColSet *sets, int n, long in_pitch,
                  long in_plane, int ncols, long out_pitch, long out_plane, const SpecTables &tab, hipStream_t s,
                  LaunchEv ev) {
#define PAIR(a, b)                                                                                            \
  if (nyi == a && nyo == b)                                                                                   \
    return dt == F64 ? launch_col<double, a, b>(padmode, fwd, inv, sets, n, in_pitch, in_plane, ncols,        \
                                                out_pitch, out_plane, tab, s, dt, 0, ev)                      \
                     : launch_col<float, a, b>(padmode, fwd, inv, sets, n, in_pitch, in_plane, ncols,         \
                                               out_pitch, out_plane, tab, s, dt, 0, ev);
  PAIR(32, 32) PAIR(48, 48) PAIR(64, 64) PAIR(96, 96) PAIR(128, 128) PAIR(144, 144) PAIR(192, 192) PAIR(256, 256)
  PAIR(288, 288) PAIR(384, 384)
  PAIR(32, 48) PAIR(48, 32) PAIR(64, 96) PAIR(96, 64) PAIR(96, 144) PAIR(144, 96)
  PAIR(128, 192) PAIR(192, 128) PAIR(192, 288) PAIR(288, 192) PAIR(256, 384) PAIR(384, 256)
#undef PAIR
  return hipErrorInvalidValue;
}

}  // namespace lp
