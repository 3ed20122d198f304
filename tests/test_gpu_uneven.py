"""GPU parity at uneven grids (nx != ny, the lengths 96 and 192 with their 144- and
288-point rows of the 3/2 grid) against the binary64 oracle, tolerance 1e-12 relative L2."""
import numpy as np
import pytest

from conftest import rel_l2
from population_balance_amd import abi

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("nx,ny,nz", [(96, 32, 7), (192, 64, 5)])
def test_dealias_uneven(nx, ny, nz):
    """more rows than one block of the row passes takes, and a last block that is not full"""
    from oracle import Oracle
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(nx, ny, nz)
    o, lg = Oracle(cfg), Lesgo(cfg)
    g = cfg.grid
    print(f"\n[case] dealias {nx}x{ny}x{nz}", flush=True)
    u = np.random.default_rng(11).standard_normal((g.nz, g.ny, g.ld))
    big = np.zeros((g.nz, g.ny2, g.ld_big))
    lg.dealias1(u, big)
    ref = o.dealias1(u)
    assert rel_l2(big, ref, g.nx2) < TOL
    out = np.zeros_like(u)
    lg.dealias2(out, ref.copy())
    assert rel_l2(out, o.dealias2(ref), g.nx) < TOL
    lg.close()
    o.close()
