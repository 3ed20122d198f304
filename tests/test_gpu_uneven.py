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


@pytest.mark.parametrize("nz", [4, 9, 71, 72, 143, 144, 287, 288, 320])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_pressure_row_segments(nz, prec):
    """the pressure solve at both sides of each number of segments per block (72, 144 and
    288 rows: nz + 1), with a last segment that is short or empty, and over several rounds;
    two solves, the second from other fields.  FP64 against the oracle at 1e-12; mixed at
    5e-6 (binary32 transforms of fields of order 1 without a mean flow: 6e-8 per operation
    over the 2 log2(64 32) additions of a plane's transform)."""
    from harness import random_fields
    from oracle import Oracle
    from population_balance_amd import ic
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(64, 32, nz, precision=abi.LP_MIXED if prec == "mixed" else abi.LP_FP64)
    g = cfg.grid
    o, lg = Oracle(abi.copy_config(cfg, precision=abi.LP_FP64)), Lesgo(cfg)
    print(f"\n[case] pressure segments nz={nz} {prec}", flush=True)
    for seed in (22, 23):
        u, v, w = ic.turbulent_ic(g, seed=seed, log_law=False)
        n = random_fields(cfg, ["u", "v", "w", "divtz"], seed=seed)
        for name, a in (("u", u + 0.1 * n["u"]), ("v", v + 0.1 * n["v"]), ("w", w + 0.1 * n["w"]),
                        ("divtz", n["divtz"])):
            o.set_field(name, a)
            lg.upload(name, a)
        o.call("press_stag_array")
        lg.press_stag_array()
        for name, top in (("p", nz), ("dpdx", nz - 1), ("dpdy", nz - 1)):
            err = rel_l2(lg.download(name)[:top], o.field(name)[:top], g.nx)
            print(f"  {name}: {err:.2e}", end="")
            assert err < (TOL if prec == "fp64" else 5e-6), (name, err)
        print()
    lg.close()
    o.close()


@pytest.mark.parametrize("nz", [9, 72, 144, 290])
def test_adjoint_row_segments(nz):
    """the transposed pressure solve inside the adjoint step, against the oracle's adjoint
    at 1e-12, over one and several rounds of segments"""
    import ctypes as C
    import torch
    from harness import random_fields
    from oracle import Oracle
    from population_balance_amd import ic
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(32, 32, nz)
    g = cfg.grid
    print(f"\n[case] adjoint segments nz={nz}", flush=True)
    vel = dict(zip(("u", "v", "w"), ic.turbulent_ic(g, seed=4)))
    n = random_fields(cfg, ["u", "v", "w", "RHSx", "RHSy", "RHSz", "Nu_t", "ustar"], seed=5)
    ub0 = np.stack([n["u"], n["v"], n["w"]])
    rb0 = np.stack([n["RHSx"], n["RHSy"], n["RHSz"]])
    rb0[:, -1] = 0.0
    nut = 1e-3 * (1.0 + 0.1 * np.clip(n["Nu_t"], -3, 3))
    ust = 1.0 + 0.1 * np.clip(n["ustar"], -3, 3)
    o, lg = Oracle(cfg), Lesgo(cfg)
    dp = C.POINTER(C.c_double)
    o.L.or_step_adjoint.argtypes = [C.c_void_p, dp, dp, dp, dp]
    p = lambda a: a.ctypes.data_as(dp)  # noqa: E731
    for name, a in vel.items():
        o.set_field(name, a)
        lg.upload(name, a)
    o.set_time(3)
    lg.set_time(3)
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


@pytest.mark.parametrize("nx,ny,nz,kw", [(96, 32, 10, {}), (64, 96, 9, {"lbc_mom": abi.LP_LBC_STRESS_FREE}),
                                         (32, 192, 13, {"model": 4})])
def test_steps_uneven(nx, ny, nz, kw):
    """whole binary64 steps with the passes over several fields in one launch, at level
    counts that leave the last group of eight planes of each field part full"""
    from harness import load_gpu, load_oracle, seeded_state
    from oracle import Oracle
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(nx, ny, nz, **kw)
    o, lg = Oracle(cfg), Lesgo(cfg)
    print(f"\n[case] steps uneven {nx}x{ny}x{nz} {kw}", flush=True)
    st = seeded_state(cfg)
    load_oracle(o, st)
    load_gpu(lg, st)
    for _ in range(3):
        o.step(1)
        lg.step(1)
    for n, top in [(n, nz - 1) for n in ("u", "v", "w", "RHSx", "RHSy", "RHSz")] + [("p", nz)]:
        err = rel_l2(lg.download(n)[:top], o.field(n)[:top], nx)
        print(f"  {n}: {err:.2e}", end="")
        assert err < TOL, (n, err)
    print()
    lg.close()
    o.close()


@pytest.mark.parametrize("nx,ny,nz", [(32, 32, 4), (32, 32, 5), (96, 32, 7), (128, 64, 65)])
def test_lag_level_runs(nx, ny, nz):
    """the Lagrangian relaxation in level runs of 1, 2, 3 and 4 (the 128-point test of fifty
    steps takes runs of 8): three binary64 steps, each with a new coefficient.  RHS at 1e-11
    and the coefficient at 1e-6: its averages are rounded to REAL(4) (6e-8 where a last bit
    of binary64 flips one), the SGS part is some 1e-2 of RHS and a flip one of 4000 points."""
    from harness import load_gpu, load_oracle, seeded_state
    from oracle import Oracle
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(nx, ny, nz, cs_count=1)
    o, lg = Oracle(cfg), Lesgo(cfg)
    print(f"\n[case] lag runs {nx}x{ny}x{nz}", flush=True)
    st = seeded_state(cfg)
    load_oracle(o, st)
    load_gpu(lg, st)
    for _ in range(3):
        o.step(1)
        lg.step(1)
    for n, top in [(n, nz - 1) for n in ("u", "v", "w", "RHSx", "RHSy", "RHSz")] \
            + [(n, nz) for n in ("Cs_opt2", "F_LM", "F_QN")]:
        err = rel_l2(lg.download(n)[:top], o.field(n)[:top], nx)
        print(f"  {n}: {err:.2e}", end="")
        assert err < (1e-6 if n[0] in "CF" else 1e-11 if n[0] == "R" else TOL), (n, err)
    print()
    lg.close()
    o.close()


@pytest.mark.parametrize("nx,ny,nz,nb,bc,kw", [
    (96, 32, 4, 2, (0, 1), dict(inertia=False)),       # 32-point tiles, two bins, runs of 1 and 2 levels
    (32, 64, 5, 5, (1, 0), {}),                        # a full group
    (64, 32, 20, 7, (2, 1), {}),                       # a group and a remainder, ghosts by sign along x
    (64, 96, 9, 11, (1, 2), dict(settling=False)),
    (192, 64, 34, 4, (0, 0), dict(inertia=False)),     # runs of 4 levels
    (128, 128, 130, 3, (1, 1), dict(sfc_flux=-0.5)),   # runs of 16
])
def test_droplet_transport_tiles(nx, ny, nz, nb, bc, kw):
    """the droplet right-hand side over its tiles, bin groups and level runs: one
    pollen_all_in_one2 with the previous RHS kept outside the cells, against the oracle at
    1e-12 (binary64, terms of the same order summed in the oracle's order up to contraction)"""
    from oracle import Oracle
    from population_balance_amd import droplets
    from population_balance_amd.lesgo import Lesgo
    from test_gpu_droplets import _load, _routine_state
    cfg = abi.make_config(nx, ny, nz)
    ds = droplets.DropletSet(nb)
    ds.fill(cfg, pbe=False, bc=bc, **kw)
    print(f"\n[case] droplet tiles {nx}x{ny}x{nz} bins {nb} bc {bc} {kw}", flush=True)
    o, lg = Oracle(cfg), Lesgo(cfg)
    st = _routine_state(cfg, ds)
    st["RHS_PCon"] = st["RHS_PCon"] + 1e-3
    _load(o, lg, st, jt_total=2)
    for c in (o, lg):
        c.set_time(2, 2)
    o.call("pollen_all_in_one2")
    lg.pollen_all_in_one2()
    for n in ("RHS_PCon", "PCon"):
        a, b = lg.download(n), o.field(n)
        err = rel_l2(a, b, nx)
        print(f"  {n}: {err:.2e}", end="")
        assert err < TOL, (n, err)
        for q in range(nb):
            e = rel_l2(a[q], b[q], nx)
            assert e < TOL, (n, q, e)
    print()
    assert np.array_equal(lg.download("RHS_PCon")[..., nx:], st["RHS_PCon"][..., nx:])
    assert np.array_equal(lg.download("RHS_PCon")[:, -1], st["RHS_PCon"][:, -1])
    lg.close()
    o.close()


@pytest.mark.parametrize("nx,ny,nz,nb,bc", [(96, 32, 7, 5, (1, 0)),    # a part-filled block, one bin per run
                                            (32, 64, 6, 2, (2, 1)),
                                            (128, 64, 20, 7, (0, 2)),  # runs of several bins
                                            (192, 96, 16, 3, (1, 1))])  # one run
def test_droplet_adjoint_runs(nx, ny, nz, nb, bc):
    """the transposed droplet transport over its blocks and runs of bins against the oracle;
    1e-11, and 1e-10 for the concentration's adjoint, as the adjoint's tests at 32x32x9 (its
    diffusion terms cancel to a few parts in 1e4 of themselves)"""
    import ctypes as C
    import torch
    from harness import random_fields
    from oracle import Oracle
    from population_balance_amd import droplets, ic
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(nx, ny, nz)
    ds = droplets.DropletSet(nb)
    ds.fill(cfg, bc=bc, inertia=False)
    g = cfg.grid
    print(f"\n[case] droplet adjoint runs {nx}x{ny}x{nz} bins {nb} bc {bc}", flush=True)
    rng = np.random.default_rng(6)
    shc = abi.field_shape(g, "PCon", nb)

    def phys(a):
        a[..., nx:] = 0.0
        return np.ascontiguousarray(a)
    n = random_fields(cfg, ["u", "v", "w", "RHSx", "RHSy", "RHSz", "Nu_t", "ustar"], seed=5)
    ub0, rb0 = np.stack([phys(n[q]) for q in ("u", "v", "w")]), np.stack([phys(n[q]) for q in ("RHSx", "RHSy", "RHSz")])
    cb0, rcb0 = phys(rng.standard_normal(shc)), phys(rng.standard_normal(shc))
    rb0[:, -1] = 0.0
    rcb0[:, -1] = 0.0
    nut = phys(1e-3 * (1.0 + 0.1 * np.clip(n["Nu_t"], -3, 3)))
    ust = 1.0 + 0.1 * np.clip(n["ustar"], -3, 3)
    st = dict(zip(("u", "v", "w"), ic.turbulent_ic(g, seed=4)))
    st["PCon"] = phys(droplets.initial_concentration(cfg, ds) * (1.0 + 0.3 * rng.random(shc)))
    o, lg = Oracle(cfg), Lesgo(cfg)
    for c, put in ((o, o.set_field), (lg, lg.upload)):
        for name, a in st.items():
            put(name, a)
        c.set_time(3, 3)
    dp = C.POINTER(C.c_double)
    o.L.or_step_adjoint2.argtypes = [C.c_void_p] + [dp] * 6
    p = lambda a: a.ctypes.data_as(dp)  # noqa: E731
    ref = [a.copy() for a in (ub0, rb0, cb0, rcb0)]
    assert o.L.or_step_adjoint2(o.h, p(nut), p(ust), *(p(a) for a in ref)) == 0
    dev = [torch.from_numpy(a).to("cuda") for a in (ub0, rb0, cb0, rcb0)]
    lg.step_adjoint(torch.from_numpy(nut).to("cuda"), torch.from_numpy(ust).to("cuda"), *dev)
    out = [a.cpu().numpy() for a in dev]
    for name, a, b, tol in zip(("u", "RHS", "PCon", "RHS_PCon"), out, ref, (1e-11, 1e-11, 1e-10, 1e-11)):
        top = nz - 1 if name == "RHS" else nz
        err = rel_l2(a[:, :top], b[:, :top], nx)
        print(f"  {name}: {err:.2e}", end="")
        assert err < tol, (name, err)
    print()
    assert not out[2][..., nx:].any()
    lg.close()
    o.close()


@pytest.mark.parametrize("nx,ny,nz", [(96, 32, 7), (192, 64, 5)])
def test_dealias_uneven_mixed(nx, ny, nz):
    """the binary32 rows of 72, 96, 144 and 192 points, at the bound that the binary32 filt_da,
    which takes as many passes, has"""
    from oracle import Oracle
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(nx, ny, nz, precision=abi.LP_MIXED)
    o, lg = Oracle(abi.copy_config(cfg, precision=abi.LP_FP64)), Lesgo(cfg)
    g = cfg.grid
    print(f"\n[case] dealias mixed {nx}x{ny}x{nz}", flush=True)
    u = np.random.default_rng(11).standard_normal((g.nz, g.ny, g.ld)).astype(np.float32)
    big = np.zeros((g.nz, g.ny2, g.ld_big), np.float32)
    lg.dealias1(u, big)
    ref = o.dealias1(u.astype(np.float64))
    e1 = rel_l2(big, ref, g.nx2)
    big = ref.astype(np.float32)
    out = np.zeros_like(u)
    lg.dealias2(out, big.copy())
    e2 = rel_l2(out, o.dealias2(big.astype(np.float64)), g.nx)
    print(f"  {e1:.2e} {e2:.2e}")
    assert e1 < 1e-6 and e2 < 1e-6, (e1, e2)
    lg.close()
    o.close()


@pytest.mark.parametrize("ny,nz", [(32, 7), (64, 9)])
def test_steps_192(ny, nz):
    """whole binary64 steps with 144-point convection rows; bounds as in test_lag_level_runs"""
    from harness import load_gpu, load_oracle, seeded_state
    from oracle import Oracle
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(192, ny, nz)
    o, lg = Oracle(cfg), Lesgo(cfg)
    print(f"\n[case] steps 192x{ny}x{nz}", flush=True)
    st = seeded_state(cfg)
    load_oracle(o, st)
    load_gpu(lg, st)
    for _ in range(3):
        o.step(1)
        lg.step(1)
    for n, top in [(n, nz - 1) for n in ("u", "v", "w", "RHSx", "RHSy", "RHSz")] + [("p", nz)]:
        err = rel_l2(lg.download(n)[:top], o.field(n)[:top], 192)
        print(f"  {n}: {err:.2e}", end="")
        assert err < (1e-11 if n[0] == "R" else TOL), (n, err)
    print()
    lg.close()
    o.close()


@pytest.mark.parametrize("nx,ny,nz", [(96, 32, 17), (192, 32, 9), (96, 192, 8)])
def test_steps_theta_uneven_mixed(nx, ny, nz):
    """binary32 steps with theta over the 72- and 144-point rows (convection, the padding of
    velocities and theta), at the bound of test_steps_with_theta_mixed"""
    from test_gpu_theta import _load, _pair, _theta_state
    cfg = abi.make_config(nx, ny, nz, precision=abi.LP_MIXED, L_z=1.5)
    abi.set_scalar_defaults(cfg.scal, s_flag=1)
    cfg.scal.wt_s, cfg.scal.dTdz_top = 0.1, 0.01
    o, lg = _pair(cfg)
    st = _theta_state(cfg)
    for n in ("RHS_T", "Nu_t", "ustar"):
        st.pop(n)
    _load(o, lg, st)
    print(f"\n[case] steps with theta mixed {nx}x{ny}x{nz}", flush=True)
    o.step(2)
    lg.step(2)
    errs = {n: rel_l2(lg.download(n), o.field(n), nx) for n in ("u", "v", "w")}
    th0 = st["theta"]
    errs["theta change"] = rel_l2(lg.download("theta") - th0, o.field("theta") - th0, nx)
    print({k: f"{v:.2e}" for k, v in errs.items()})
    assert max(errs.values()) < 1e-5, errs
    lg.close()
    o.close()


@pytest.mark.parametrize("nz", [143, 144, 287, 288, 500])
def test_pressure_rounds(nz):
    """the binary64 pressure solve where a block's segments go in rounds of equal length (128 x 64
    points: 320 blocks): one round, two, and more, at 1e-12 of the oracle"""
    from harness import random_fields
    from oracle import Oracle
    from population_balance_amd import ic
    from population_balance_amd.lesgo import Lesgo
    cfg = abi.make_config(128, 64, nz)
    g = cfg.grid
    o, lg = Oracle(cfg), Lesgo(cfg)
    print(f"\n[case] pressure rounds nz={nz}", flush=True)
    u, v, w = ic.turbulent_ic(g, seed=24, log_law=False)
    n = random_fields(cfg, ["u", "v", "w", "divtz"], seed=24)
    for name, a in (("u", u + 0.1 * n["u"]), ("v", v + 0.1 * n["v"]), ("w", w + 0.1 * n["w"]), ("divtz", n["divtz"])):
        o.set_field(name, a)
        lg.upload(name, a)
    o.call("press_stag_array")
    lg.press_stag_array()
    for name, top in (("p", nz), ("dpdx", nz - 1), ("dpdy", nz - 1)):
        err = rel_l2(lg.download(name)[:top], o.field(name)[:top], g.nx)
        print(f"  {name}: {err:.2e}", end="")
        assert err < TOL, (name, err)
    print()
    lg.close()
    o.close()


@pytest.mark.parametrize("nx,ny,nz,nb,bc,kw", [
    (32, 32, 70, 3, (2, 2), {}),      # 69 runs of one level split over the XCDs, the last XCD's part empty
    (32, 32, 140, 7, (0, 1), {}),     # two groups, runs of 2
    (96, 192, 9, 6, (1, 0), {}),      # 72 tiles, an XCD's consecutive
    (64, 64, 65, 2, (0, 0), {}),      # 16 tiles in the order of the blocks
])
def test_droplet_transport_split(nx, ny, nz, nb, bc, kw):
    """the droplet right-hand side in each order of tiles and runs, as test_droplet_transport_tiles"""
    test_droplet_transport_tiles(nx, ny, nz, nb, bc, kw)
