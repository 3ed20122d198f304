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


@pytest.mark.parametrize("nz,model", [(2100, 5), (3121, 5), (3121, 4)])
def test_steps_tall(nz, model):
    """binary64 steps, two fields a launch (2100 levels) and one (3121); the test filters of model
    5 take 21 nz planes.  Bounds as in test_lag_level_runs (the averages are rounded to REAL(4),
    and RHS holds their result)"""
    from harness import load_gpu, load_oracle, seeded_state
    from oracle import Oracle
    from population_balance_amd.lesgo import Lesgo
    cfg = _tall(32, 32, nz, cs_count=1, model=model)
    o, lg = Oracle(cfg), Lesgo(cfg)
    print(f"\n[case] steps 32x32x{nz} model {model}", flush=True)
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


@pytest.mark.parametrize("nz", [4200, 6200])
def test_steps_tall_theta_mixed(nz):
    """binary32 steps with theta, two fields a launch and one, at the bound of
    test_steps_with_theta_mixed"""
    from test_gpu_theta import _cfg, _load, _pair, _theta_state
    cfg = _cfg(nz=nz, L_z=(nz - 1) / 32.0, wt_s=0.1, dTdz_top=0.01, precision=abi.LP_MIXED)
    g = cfg.grid
    o, lg = _pair(cfg)
    st = _theta_state(cfg)
    for n in ("RHS_T", "Nu_t", "ustar"):
        st.pop(n)
    _load(o, lg, st)
    print(f"\n[case] steps with theta mixed 32x32x{nz}", flush=True)
    o.step(2)
    lg.step(2)
    errs = {n: rel_l2(lg.download(n), o.field(n), g.nx) for n in ("u", "v", "w")}
    th0 = st["theta"]
    errs["theta change"] = rel_l2(lg.download("theta") - th0, o.field("theta") - th0, g.nx)
    print({k: f"{v:.2e}" for k, v in errs.items()})
    assert max(errs.values()) < 1e-5, errs
    lg.close()
    o.close()


@pytest.mark.parametrize("nz", [2100, 3121])
def test_adjoint_tall(nz):
    """the adjoint step, two fields a launch and one, at the bound of test_adjoint_row_segments"""
    import ctypes as C
    import torch
    from harness import random_fields
    from oracle import Oracle
    from population_balance_amd import ic
    from population_balance_amd.lesgo import Lesgo
    cfg = _tall(32, 32, nz)
    g = cfg.grid
    print(f"\n[case] adjoint 32x32x{nz}", flush=True)
    vel = dict(zip(("u", "v", "w"), ic.turbulent_ic(g, seed=4)))
    n = random_fields(cfg, ["u", "v", "w", "RHSx", "RHSy", "RHSz", "Nu_t", "ustar"], seed=5)
    ub0 = np.stack([n["u"], n["v"], n["w"]])
    rb0 = np.stack([n["RHSx"], n["RHSy"], n["RHSz"]])
    rb0[:, -1] = 0.0
    nut = 1e-3 * (1.0 + 0.1 * np.clip(n["Nu_t"], -3, 3))
    ust = 1.0 + 0.1 * np.clip(n["ustar"], -3, 3)
    o, lg = Oracle(cfg), Lesgo(cfg)
    for name, a in vel.items():
        o.set_field(name, a)
        lg.upload(name, a)
    o.set_time(3)
    lg.set_time(3)
    dp = C.POINTER(C.c_double)
    o.L.or_step_adjoint.argtypes = [C.c_void_p, dp, dp, dp, dp]
    p = lambda a: a.ctypes.data_as(dp)  # noqa: E731
    ub_o, rb_o = ub0.copy(), rb0.copy()
    assert o.L.or_step_adjoint(o.h, p(nut), p(ust), p(ub_o), p(rb_o)) == 0
    ub, rb, tn, tu = (torch.from_numpy(a).to("cuda") for a in (ub0, rb0, nut, ust))
    lg.step_adjoint(tn, tu, ub, rb)
    for q in range(3):
        eu = rel_l2(ub[q].cpu().numpy(), ub_o[q], g.nx)
        er = rel_l2(rb[q].cpu().numpy()[:nz - 1], rb_o[q][:nz - 1], g.nx)
        print(f"  {eu:.2e} {er:.2e}", end="")
        assert eu < TOL and er < TOL, (q, eu, er)
    print()
    lg.close()
    o.close()


def test_context_memory():
    """a context whose passes take one field a launch keeps no spectra for more: at 32x32x20000,
    binary64, model 1, no more than the 911.3 bytes a point that contexts took when every pass
    took one field"""
    import torch
    from population_balance_amd.lesgo import Lesgo
    Lesgo(abi.make_config(32, 32, 4)).close()
    cfg = _tall(32, 32, 20000, model=1)
    print("\n[case] memory of a 32x32x20000 context", flush=True)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    lg = Lesgo(cfg)
    used = free - torch.cuda.mem_get_info()[0]
    lg.close()
    print(f"  {used / (32 * 32 * 20000):.1f} bytes a point")
    assert used <= 911.3 * 32 * 32 * 20000
