"""Grids of few points per level and thousands of levels, against the binary64 oracle: more
planes than a grid of blocks has along y, and spectra so large that the spectral passes take
two fields or one at a time, as they do at 256x256x257."""
import numpy as np
import pytest

from conftest import rel_l2
from population_balance_amd import abi

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _tall(nx, ny, nz, **kw):
    return abi.make_config(nx, ny, nz, L_z=(nz - 1) / 32.0, **kw)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_padd_planes(prec):
    """padd and unpadd of more than 65535 planes: copies, so equal to the oracle's, on the
    first planes and across the 65528th and 65536th"""
    import torch
    from oracle import Oracle
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(32, 32, 5, precision=abi.LP_MIXED if prec == "mixed" else abi.LP_FP64)
    g = cfg.grid
    o, lg = Oracle(abi.copy_config(cfg, precision=abi.LP_FP64)), Lesgo(cfg)
    n = 65536 + 9
    print(f"\n[case] padd of {n} planes {prec}", flush=True)
    ct = torch.complex64 if prec == "mixed" else torch.complex128
    u = torch.randn((n, g.ny, g.lh), dtype=ct, device="cuda", generator=torch.Generator("cuda").manual_seed(5))
    big = torch.zeros((n, g.ny2, g.lh_big), dtype=ct, device="cuda")
    cc = torch.zeros_like(u)
    lg.padd(big, u)
    lg.unpadd(cc, big)
    lg.sync()
    for s in (slice(0, 3), slice(65525, n)):
        ref = o.padd(u[s].cpu().numpy().astype(np.complex128))
        assert np.array_equal(big[s].cpu().numpy(), ref)
        assert np.array_equal(cc[s].cpu().numpy(), o.unpadd(ref))
    lg.close()
    o.close()


@pytest.mark.parametrize("nz", [3121])
def test_steps_tall(nz):
    """binary64 steps with the dynamic model, whose test filters take 21 nz planes; bounds as in
    test_lag_level_runs (the averages are rounded to REAL(4), and RHS holds their result)"""
    from harness import load_gpu, load_oracle, seeded_state
    from oracle import Oracle
    from population_balance_amd.lesgo import Lesgo
    cfg = _tall(32, 32, nz, cs_count=1)
    o, lg = Oracle(cfg), Lesgo(cfg)
    print(f"\n[case] steps 32x32x{nz}", flush=True)
    st = seeded_state(cfg)
    load_oracle(o, st)
    load_gpu(lg, st)
    for _ in range(2):
        o.step(1)
        lg.step(1)
    for n, top in [(n, nz - 1) for n in ("u", "v", "w", "RHSx", "RHSy", "RHSz")] \
            + [(n, nz) for n in ("p", "Cs_opt2", "F_LM", "F_QN")]:
        err = rel_l2(lg.download(n)[:top], o.field(n)[:top], cfg.grid.nx)
        print(f"  {n}: {err:.2e}", end="")
        assert err < (1e-6 if n[0] in "CF" else 1e-11 if n[0] == "R" else TOL), (n, err)
    print()
    lg.close()
    o.close()
