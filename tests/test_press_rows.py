"""Where the pressure solves look for a row: the split of a row's place into a wavefront's
64-bit address and a lane's 32-bit offset (csrc/lp_press.hpp), evaluated on the host for
every segment and row of small volumes and of volumes past 4 GiB, against 64-bit arithmetic."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "population_balance_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include "lp_press.hpp"
#include <cstdio>
#include <cstdlib>
using namespace lp;

// element `row` of a volume of `rows` planes of ps values, addressed from row0
static void check(const char *what, int row, int row0, int rows, unsigned ps, unsigned o, unsigned bytes) {
  const long long want = ((long long)row * ps + o) * bytes;
  const long long got = (long long)row_base(row0, ps) * bytes + row_off(row, row0, ps, o, bytes);
  if (got != want || row < 0 || row >= rows || row0 < 0 || row0 >= rows) {
    std::printf("%s: row %d from %d of %d: %lld, not %lld\n", what, row, row0, rows, got, want);
    std::exit(1);
  }
}

int main(int argc, char **argv) {
  const int nx = std::atoi(argv[1]), ny = std::atoi(argv[2]), nz = std::atoi(argv[3]);
  const unsigned pitch = (nx / 2 + 1 + 15) / 16 * 16, ps = pitch * ny;
  const bool serial = std::atoi(argv[4]);  // the binary64 solve's split, else the scan's
  const int n = nz + 1, S = serial ? press_segs64(n, ps / kPsModes) : press_segs(n), W = 64 / kPsModes;
  const int per = (n + S - 1) / S, Lr = serial ? serial_rows(n, S) : per < kPsRows ? per : kPsRows;
  const int rounds = serial ? serial_rounds(n, S) : press_rounds(n) ? (n + S * Lr - 1) / (S * Lr) : 1;
  if ((long)rounds * S * Lr < n || Lr > kPsRows) return std::printf("rows left out\n"), 1;
  const unsigned at[2] = {0, ps - 1};
  auto low = [](int a, int b) { return a < b ? a : b; };
  for (int rd = 0; rd < rounds; ++rd)
    for (int s = 0; s < S; ++s) {
      const int j0 = (rd * S + s) * Lr, jw = (rd * S + s / W * W) * Lr;
      for (int q = 0; q <= Lr; ++q)
        for (unsigned o : at) {
          const int j = j0 + q;
          check("H binary32", press_plane(j, nz), press_plane(jw, nz), nz - 1, ps, o, 8);
          check("H binary64", press_plane(j, nz), press_plane(jw, nz), nz - 1, ps, o, 16);
          if (q == Lr) continue;
          check("bet", low(j, nz), low(jw, nz), n, ps, o, 8);
          check("adjoint of p", low(j, nz - 1), low(jw, nz - 1), nz, ps, o, 16);
          if (j <= nz) check("p_hat", j, jw, n, ps, o, 16);
        }
    }
  std::printf("ok %.2f GiB\n", (double)n * ps * 16 / (1u << 30));
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("press_rows")
    src, exe = d / "press_rows.hip", d / "press_rows"
    src.write_text(PROGRAM)
    cmd = [HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return str(exe)


@pytest.mark.parametrize("serial", [0, 1])
@pytest.mark.parametrize("nx,ny,nz", [(32, 32, 4), (64, 32, 71), (64, 32, 72), (64, 64, 143), (96, 64, 288),
                                      (128, 64, 144), (128, 128, 289), (256, 256, 257), (256, 256, 7281),
                                      (256, 256, 9000), (128, 128, 27000), (32, 32, 270000)])
def test_row_addresses(program, nx, ny, nz, serial):
    r = subprocess.run([program, str(nx), str(ny), str(nz), str(serial)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
