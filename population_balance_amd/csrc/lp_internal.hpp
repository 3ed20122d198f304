// lp_internal.hpp -- host-side interface between the C ABI layer (lp_api.hip) and the
// kernel launchers (lp_fft.hip, lp_physics.hip).  Not part of the public ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace lp {

enum Dt { F32 = 0, F64 = 1 };

// twiddle tables exp(-2 pi i j / N), j < N, in both precisions
struct Twiddle {
  int n;
  const void *d;  // double2[n]
  const void *f;  // float2[n]
};
const void *tw_ptr(int n, Dt dt);  // device pointer; aborts the launch (nullptr) if missing

// multiplier applied per spectral output of a column operation
enum Mult { M_ONE = 0, M_IKX = 1, M_IKY = 2, M_G1 = 3, M_G2 = 4 };

struct SpecTables {
  const double *kx, *ky, *G1, *G2;  // (lh, ny) of the small grid
  int lh, ny;                        // small-grid sizes
};

// Every pass takes a list of fields (sets): the same pass over several volumes in one launch.
// Small grids are bound by launches (a pass of 33 planes of 32 x 32 takes 3.4 us, the shortest
// kernel 2.0), and three fields fill the chip better than one.  A set's planes follow those of
// the sets before it.
constexpr int kMaxSets = 9;

// Row pass: real rows of length 2M (scaled by `scale`) -> complex half spectra (M+1 values,
// only the first ncols_out written).
//  shift (binary64 rows into a binary32 transform): each plane enters less its first value,
//  stored in shift_out[plane] when shift_out is given; only the plane's kx = ky = 0 mode
//  moves, by that value.
//  comp >= 0: the rows are a vorticity component formed from two derivative volumes (0:
//  w_y - v_z from in = dwdy, b = dvdz; 1: u_z - w_x from in = dwdx, b = dudz; 2: v_x - u_y
//  from in = dvdx, b = dudy), the derivatives of w averaged onto the uvp node on plane 0;
//  all sets of a launch or none.
struct R2cSet {
  const void *in;
  void *out;
  int nplanes;
  double scale;
  bool shift = false;
  double *shift_out = nullptr;
  const void *b = nullptr;
  int comp = -1;
};
// din: the type of the rows (dt, or F64 into an F32 transform)
hipError_t row_r2c(Dt dt, Dt din, int M, const R2cSet *sets, int n, long in_pitch, long in_plane, int rows,
                   long out_pitch, long out_plane, int ncols_out, hipStream_t s);

// Row pass: complex half spectra (ncols_in columns present, rest zero) -> real rows
// of length 2M; columns [2M, out_pitch) set to zero.  Compute type dtc, store type dto (dtc, or
// F32 from F64).
//  div 1 / 2 (dtc == dto; all sets of a launch or none): the z-derivative term of divstress
//  from tz (the layout of out): 1 (divstress_uv) adds cst (tz(k+1) - tz(k)) and writes BOGUS on
//  the top level; 2 (divstress_w) adds cst (tz(k) - tz(k-1)) on levels 1..nplanes-2.
struct C2rSet {
  const void *in;
  void *out;
  int nplanes;
  const void *tz = nullptr;
  int div = 0;
};
// ikx (optional, M+1 values, zero at kx = 0 and kx = M): the spectra are multiplied by
// i*ikx[kx] first, so the rows are the x-derivative of what they would be without it.
hipError_t row_c2r(Dt dtc, Dt dto, int M, const C2rSet *sets, int n, long in_pitch, long in_plane, int ncols_in,
                   int rows, long out_pitch, long out_plane, hipStream_t s, const double *ikx = nullptr,
                   double cst = 0.0);

struct ColOut {
  void *ptr;
  int mult;
  long pitch = 0;  // overrides of the call's out_pitch / out_plane / ncols (0: keep)
  long plane = 0;
  int ncols = 0;
  double scale = 1.0;  // padmode 1 and 2 only: factor on the output spectrum
};
// dc (padmode 1): dc[plane] is added to the real part of the input's kx = 0 column at every y,
// in binary64 (the inverse of row_r2c's shift on a spectrum that keeps the row means there)
struct ColSet {
  const void *in;
  int nplanes;
  int nout;
  ColOut outs[3];
  const double *dc = nullptr;
};

// Timing events taken by the dispatch of a launch itself (hipExtLaunchKernel): start at
// the first wave, stop at the end of the kernel, with no marker packet in the stream.
// Either may be null.
struct LaunchEv {
  hipEvent_t start = nullptr, stop = nullptr;
};

// Column pass over ncols kx-columns of the sets' spectra:
//  fwd: forward complex DFT of length nyi along y;
//  map: padmode 0 (same grid, Nyquist row/column killed, multiplier applied),
//       1 (zero-pad ny -> ny2 as padd.f90), 2 (truncate ny2 -> ny as unpadd.f90);
//  inv: inverse DFT of length nyo.
// An output may be the input's own buffer.
hipError_t col_op(Dt dt, int nyi, int nyo, int padmode, int fwd, int inv, const ColSet *sets, int n, long in_pitch,
                  long in_plane, int ncols, long out_pitch, long out_plane, const SpecTables &tab, hipStream_t s,
                  LaunchEv ev = {});

// col_op (same grid, forward + inverse) on the columns col0..ncols-1 only, one column per
// block: the few columns past the last full group of a block-wide launch.
hipError_t col_op_tail(Dt dt, int ny, const ColSet &set, long in_pitch, long in_plane, int col0, int ncols,
                       long out_pitch, long out_plane, const SpecTables &tab, hipStream_t s, LaunchEv ev = {});

// Column pass of the divergence terms: out = inverse_y( i kx fwd_y(A) + i ky fwd_y(B) )
// with the Nyquist row and column zeroed; A, B, out share pitch / plane; ny == tab.ny.
// out may be a buffer of A or B that no other set reads.
struct DivSet {
  const void *A, *B;
  void *out;
};
hipError_t col_div(Dt dt, int ny, const DivSet *sets, int n, int nplanes, long pitch, long plane, int ncols,
                   const SpecTables &tab, hipStream_t s);

bool fft_len_supported(int n);

// record the message that lp_last_error() returns; returns code
int set_error(int code, const char *fmt, ...);

}  // namespace lp
