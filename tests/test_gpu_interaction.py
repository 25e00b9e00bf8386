"""Force interaction on the GPU vs the oracle (reference rows a12-a17, a25).

Parity metric: norm-wise relative error max|x_gpu - x_oracle| / max|x_oracle|
(per component set) with the oracle in the reference's FP32 semantics; each
result is also stated against the FP64 yardstick (FP64 pair arithmetic on
FP64 positions). Tolerances are written in the tests.
"""
import ctypes as C

import numpy as np
import pytest

from dualsphysics_amd import _native as N
from dualsphysics_amd import case as casemod
from tests.helpers import Dev, divdata, perturbed_case, rel_err, to_cte, per_particle_rel

pytestmark = pytest.mark.gpu

TOL_FP32 = 1e-5      # GPU vs FP32 oracle, norm-wise relative
TOL_PP = 1e-4        # GPU vs FP32 oracle, per particle (floor 1e-3 RMS)


def _prepared(c):
    from oracle.oracle import OracleSim
    o = OracleSim(c)
    d = o.download()
    dcell, poscell, cte = o.arrays()
    celldiv, be = o.celldiv()
    return o, d, dcell, poscell, cte, celldiv, be


def _run_both(c, tvisco, tddt, visco, viscob, lib, ctx, with_tau=False, kernel=N.FORCES_TILE):
    import oracle.oracle as orc
    assert lib.dsph_ctx_set_option(ctx, N.OPT_FORCES_KERNEL, kernel) == 0
    o, d, dcell, poscell, cte, celldiv, be = _prepared(c)
    st = o.stats()
    n, npb, npbok = st["np"], st["npb"], st["npbok"]
    rng = np.random.default_rng(2)
    tau = (rng.standard_normal((n, 6)) * 1e-3).astype(np.float32) if with_tau else None
    # GPU
    bc = Dev(lib, ctx, be)
    dv = divdata(celldiv, bc, cte)
    acte = to_cte(cte)
    assert lib.dsph_set_constants(ctx, C.byref(acte)) == 0
    gd = {k: Dev(lib, ctx, a) for k, a in (("dcell", dcell), ("poscell", poscell),
                                          ("velrho", d["velrho"]), ("code", d["code"]))}
    ace = Dev.zeros(lib, ctx, (n, 3), np.float32)
    ar = Dev.zeros(lib, ctx, n, np.float32)
    vdt = Dev.zeros(lib, ctx, n, np.float32)
    strain = Dev.zeros(lib, ctx, (n, 6), np.float32)
    taud = Dev(lib, ctx, tau) if with_tau else None
    t = N.DsphInterParms()
    t.tkernel, t.tvisco, t.tdensity = N.KERNEL_WENDLAND, tvisco, tddt
    t.viscob, t.viscof = viscob, visco
    t.np, t.npb, t.npbok = n, npb, npbok
    t.divdata = dv
    t.d_dcell, t.d_poscell, t.d_velrho, t.d_code = (gd["dcell"].ptr, gd["poscell"].ptr,
                                                     gd["velrho"].ptr, gd["code"].ptr)
    t.d_spstaurho2 = taud.ptr if with_tau else None
    t.d_viscdt, t.d_ar, t.d_ace, t.d_sps2strain = vdt.ptr, ar.ptr, ace.ptr, strain.ptr
    rc = lib.dsph_interaction_forces(ctx, C.byref(t))
    assert rc == 0, lib.dsph_last_error(ctx)
    g = {"ace": ace.get(), "ar": ar.get(), "viscdt": vdt.get(), "strain": strain.get()}
    # Oracle FP32 (GPU semantics) and FP64 yardstick.
    olib = orc.load()
    odiv = orc.OrcDiv(1, int(dv.ncx), int(dv.ncy), int(dv.ncz), int(dv.ncw), int(dv.cellfluid),
                      int(dv.cellzerox), int(dv.cellzeroy), int(dv.cellzeroz),
                      be.ctypes.data)
    res = {}
    for prec, sem in ((0, orc.SEM_GPU), (1, orc.SEM_F64)):
        oa = np.zeros((n, 3), np.float32)
        oar = np.zeros(n, np.float32)
        ov = np.zeros(n, np.float32)
        os_ = np.zeros((n, 6), np.float32)
        olib.orc_interaction(prec, sem, tvisco, tddt, viscob, visco, C.byref(cte), C.byref(odiv),
                             n, npb, npbok, dcell.ctypes.data, poscell.ctypes.data,
                             np.ascontiguousarray(d["pos"]).ctypes.data, d["velrho"].ctypes.data,
                             tau.ctypes.data if with_tau else None, oa.ctypes.data,
                             oar.ctypes.data, ov.ctypes.data, os_.ctypes.data, None)
        res[prec] = {"ace": oa, "ar": oar, "viscdt": ov, "strain": os_}
    return g, res, npb


CASES = [
    ("hydrostatic_art_ddt2full", False, 1, 3, 0.01, 0.01),
    ("perturbed_art_ddt2full", True, 1, 3, 0.01, 0.01),
    ("perturbed_art_ddt2", True, 1, 2, 0.01, 0.01),
    ("perturbed_art_ddt1", True, 1, 1, 0.01, 0.01),
    ("perturbed_art_noddt", True, 1, 0, 0.05, 0.02),
    ("perturbed_laminar", True, 3, 3, 1e-3, 1e-3),
    ("perturbed_laminarsps", True, 2, 3, 1e-3, 1e-3),
]


@pytest.mark.parametrize("kernel", [N.FORCES_TILE, N.FORCES_ROWS], ids=["staged", "rows"])
@pytest.mark.parametrize("name,pert,tvisco,tddt,visco,viscob", CASES, ids=[x[0] for x in CASES])
def test_interaction_parity(lib, ctx, name, pert, tvisco, tddt, visco, viscob, kernel):
    c = casemod.dam_break(dp=0.02)
    if pert:
        c = perturbed_case(c)
    g, res, npb = _run_both(c, tvisco, tddt, visco, viscob, lib, ctx, with_tau=(tvisco == 2),
                            kernel=kernel)
    o32, o64 = res[0], res[1]
    fl = slice(npb, None)
    e_ace = rel_err(g["ace"][fl], o32["ace"][fl])
    e_ar = rel_err(g["ar"], o32["ar"])
    e_vdt = rel_err(g["viscdt"], o32["viscdt"])
    e64_gpu = rel_err(g["ace"][fl], o64["ace"][fl])
    e64_orc = rel_err(o32["ace"][fl], o64["ace"][fl])
    e64_ar_gpu = rel_err(g["ar"], o64["ar"])
    e64_ar_orc = rel_err(o32["ar"], o64["ar"])
    print(f"{name}: gpu-vs-fp32 ace {e_ace:.2e} ar {e_ar:.2e} viscdt {e_vdt:.2e} | "
          f"vs-fp64 ace gpu {e64_gpu:.2e} oracle32 {e64_orc:.2e} ar gpu {e64_ar_gpu:.2e} "
          f"oracle32 {e64_ar_orc:.2e}")
    assert e_ace < TOL_FP32
    # In the hydrostatic state ar is pure rounding noise around 0 (norm-wise
    # relative error is then meaningless): there the GPU must stay inside the
    # FP32 noise band of the oracle itself.
    assert e_ar < max(TOL_FP32, 3 * e64_ar_orc if not pert else 0.0)
    assert e_vdt < TOL_FP32
    # GPU FP32 is as close to FP64 as the FP32 oracle is (within 2x + 1e-6).
    assert e64_gpu < 2 * e64_orc + 1e-6
    if pert:
        assert e64_ar_gpu < 2 * e64_ar_orc + 1e-6
    pp = per_particle_rel(g["ace"][fl], o32["ace"][fl])
    assert np.max(pp) < TOL_PP, np.max(pp)
    if tvisco == 2:
        assert rel_err(g["strain"][fl], o32["strain"][fl]) < TOL_FP32


def _shuffled(c, m=None, seed=5):
    """The first m fluid particles (all by default) moved by up to 0.15 dp,
    with random velocities, in random order; floating particles with random
    velocities."""
    import dataclasses
    c = perturbed_case(c, seed=seed)
    rng = np.random.default_rng(seed)
    nb, m = c.nbound, c.nfluid if m is None else m
    pos = c.pos[:nb + m].copy()
    d = rng.uniform(-0.15 * c.dp, 0.15 * c.dp, (m, 3))
    if c.data2d:
        d[:, 1] = 0
    pos[nb:] = (pos[nb:] + d)[rng.permutation(m)]
    c.velrho[nb - c.nfloat:nb, :3] = 0.3 * rng.standard_normal((c.nfloat, 3))
    return dataclasses.replace(c, idp=c.idp[:nb + m], pos=pos, velrho=c.velrho[:nb + m], nfluid=m)


_P = casemod.Parameters
FORMS = [("n%d" % m, lambda m=m: _shuffled(casemod.dam_break(dp=0.03), m))
         for m in (1, 15, 16, 17, 65)] + [
    ("ddt1", lambda: _shuffled(casemod.dam_break(dp=0.02, params=_P(tdensity=N.DDT_DDT)))),
    ("ddt2", lambda: _shuffled(casemod.dam_break(dp=0.02, params=_P(tdensity=N.DDT_DDT2)))),
    ("laminar_half_cells", lambda: _shuffled(casemod.dam_break(
        dp=0.02, params=_P(tvisco=N.VISCO_LAMINAR, visco=1e-4, cellmode=2)))),
    ("sps_mdbc", lambda: _shuffled(casemod.dam_break(dp=0.02, params=_P(
        tboundary=N.BC_MDBC, tvisco=N.VISCO_LAMINARSPS, visco=1e-6)))),
    ("mdbc2", lambda: _shuffled(casemod.dam_break(dp=0.02, params=_P(
        tboundary=N.BC_MDBC, slipmode=N.SLIP_NOSLIP, tvisco=N.VISCO_LAMINAR, visco=1e-4)))),
    ("floating", lambda: casemod.dam_break_floating(dp=0.03)),
    ("sparse", lambda: _sparse(casemod.dam_break_2d(dp=0.0025), 400)),
    # Above the team kernel's sizes (180k, 140k, 100k fluid particles in 3-D with
    # artificial, laminar, SPS viscosity; three quarters in 2-D): the tile kernel.
    ("tile_2d", lambda: _shuffled(casemod.dam_break_2d(dp=0.0008))),
    ("tile_half_cells", lambda: _shuffled(casemod.dam_break(
        dp=0.0072, params=_P(tvisco=N.VISCO_LAMINAR, visco=1e-4, cellmode=2)))),
] + [("tile_n%d" % (m % 64), lambda m=m: _shuffled(casemod.dam_break_2d(dp=0.0008), m))
     for m in (135040, 135041, 135055, 135057, 135103)]


def _sparse(c, m):
    """m fluid particles spread over the column (about one in four cells), so
    the particles of a wave span many cells of a row."""
    import dataclasses
    nb = c.nbound
    pick = nb + np.sort(np.random.default_rng(4).choice(c.nfluid, m, replace=False))
    return _shuffled(dataclasses.replace(
        c, idp=c.idp[:nb + m], pos=np.concatenate([c.pos[:nb], c.pos[pick]]),
        velrho=np.concatenate([c.velrho[:nb], c.velrho[pick]]), nfluid=m))


@pytest.mark.parametrize("make", [f for _, f in FORMS], ids=[n for n, _ in FORMS])
def test_fluid_kernel_forms_equal_bitwise(make):
    """The form that the size and options choose (teams of lanes or the tile
    kernel) and the rows kernel add the same terms in the same order: identical
    bits, also around the 16 particles of a wave and for particles in no
    order."""
    from dualsphysics_amd.sim import SphGpuSingle
    out = []
    for k in (N.FORCES_TILE, N.FORCES_ROWS):   # a run of its own each: SPS keeps tau
        s = SphGpuSingle(make())
        try:
            assert s.lib.dsph_ctx_set_option(s.lib.dsph_sim_ctx(s._h), N.OPT_FORCES_KERNEL, k) == 0
            s.run(2, sync_dt=True)
            out.append(s.forces())
        finally:
            s.close()
    for a, b in zip(*out):
        assert np.abs(b).max() > 0
        np.testing.assert_array_equal(a, b)


def _staged_and_rows(lib, ctx, c, tvisco, tddt, mdbc2=False, floating=False, poscell=None):
    """(outputs of the kernels chosen by size and options, of the rows kernels,
    boundary particles, sorted codes) for one interaction of case c: random tau,
    with ``mdbc2`` random boundary modes and tangential velocities, with
    ``floating`` two bodies, one lighter and one heavier than 1.2 fluid
    particles. ``poscell``: changes a copy of the PosCell array in place."""
    o, d, dcell, ps, cte, celldiv, be = _prepared(c)
    st = o.stats()
    n, npb, npbok = st["np"], st["npb"], st["npbok"]
    rng = np.random.default_rng(2)
    code, ps = d["code"].copy(), ps.copy()
    if poscell:
        poscell(ps, npb)
    f32 = np.float32
    dev = {"dcell": dcell, "poscell": ps, "velrho": d["velrho"],
           "spstaurho2": (rng.standard_normal((n, 6)) * 1e-3).astype(f32)}
    if mdbc2:
        dev["boundmode"] = rng.integers(0, 3, n).astype(np.uint8)
        dev["tangenvel"] = (rng.standard_normal((n, 3)) * 0.3).astype(f32)
    if floating:
        ft = (code & 0x1800) == 0x1000
        assert ft.any()
        code[ft] = (code[ft] & 0xf800) | rng.integers(0, 2, ft.sum()).astype(code.dtype)
        dev["ftomassp"] = np.array([1.1 * c.massfluid, 1.3 * c.massfluid], f32)
    dev["code"] = code
    dev = {k: Dev(lib, ctx, a) for k, a in dev.items()}
    bc = Dev(lib, ctx, be)
    acte = to_cte(cte, tboundary=N.BC_MDBC if mdbc2 else N.BC_DBC)
    assert lib.dsph_set_constants(ctx, C.byref(acte)) == 0
    outs = []
    for kernel in (N.FORCES_TILE, N.FORCES_ROWS):
        out = {k: Dev.zeros(lib, ctx, s, f32) for k, s in (
            ("ace", (n, 3)), ("ar", n), ("viscdt", n), ("sps2strain", (n, 6)))}
        t = N.DsphInterParms()
        t.tkernel, t.tvisco, t.tdensity = N.KERNEL_WENDLAND, tvisco, tddt
        t.viscob, t.viscof = 0.01, 0.02
        t.np, t.npb, t.npbok = n, npb, npbok
        t.divdata = divdata(celldiv, bc, cte)
        for k, a in (*dev.items(), *out.items()):
            setattr(t, "d_" + k, a.ptr)
        assert lib.dsph_ctx_set_option(ctx, N.OPT_FORCES_KERNEL, kernel) == 0
        rc = lib.dsph_interaction_forces(ctx, C.byref(t))
        assert lib.dsph_ctx_set_option(ctx, N.OPT_FORCES_KERNEL, N.FORCES_TILE) == 0
        assert rc == 0, lib.dsph_last_error(ctx)
        outs.append({k: a.get() for k, a in out.items()})
    return (*outs, npb, code)


def _strange_positions(ps, npb):
    """Positions that are not finite, huge, or (finite) far outside the map in
    about one of 50 particles, among them first ones of a wave."""
    rng = np.random.default_rng(6)
    for i0, i1 in ((0, npb), (npb, len(ps))):
        pick = np.concatenate([rng.integers(i0, i1, (i1 - i0) // 50),
                               i0 + 64 * rng.integers(0, (i1 - i0) // 64, (i1 - i0) // 500 + 5)])
        for kind, i in enumerate(np.array_split(pick, 5)):
            if kind < 4:
                ps[i, rng.integers(0, 3, len(i))] = (np.inf, -np.inf, np.nan, 1e20)[kind]
            else:
                ps[i, 3] = (ps[i, 3].view(np.uint32) + np.uint32(300 << 19)).view(np.float32)


@pytest.mark.parametrize("make", [lambda: casemod.dam_break(dp=0.02),
                                  lambda: casemod.dam_break_2d(dp=0.0008)], ids=["team", "tile"])
def test_strange_positions_leave_the_other_particles_alone(lib, ctx, make):
    """A position that is not finite or far from its cell has no neighbours but
    itself may be first of a wave: the sums of all particles are those
    of the kernels in which each particle walks its own cells."""
    a, b, npb, _ = _staged_and_rows(lib, ctx, perturbed_case(make()), N.VISCO_ARTIFICIAL,
                                    N.DDT_DDT2FULL, poscell=_strange_positions)
    assert np.isfinite(b["ace"]).all()
    assert np.count_nonzero(b["ace"][npb:].any(1)) > 0.9 * (len(b["ace"]) - npb)
    for k in a:
        np.testing.assert_array_equal(a[k].view(np.uint32), b[k].view(np.uint32), err_msg=k)


_ART, _LAM, _SPS = N.VISCO_ARTIFICIAL, N.VISCO_LAMINAR, N.VISCO_LAMINARSPS
_FLOAT = lambda: _shuffled(casemod.dam_break_floating(dp=0.02))  # noqa: E731  teams
_SMALL = lambda: _shuffled(casemod.dam_break(dp=0.02))  # noqa: E731  teams
_LARGE = lambda: _shuffled(casemod.dam_break(dp=0.0072))   # noqa: E731  215k fluid particles: tile
OPTIONS = [
    ("floating_ddt1", _FLOAT, _ART, N.DDT_DDT, {"floating": True}),
    ("floating_laminar_ddt2", _FLOAT, _LAM, N.DDT_DDT2, {"floating": True}),
    ("floating_sps_ddt2full", _FLOAT, _SPS, N.DDT_DDT2FULL, {"floating": True}),
    ("floating_sps_ddt1", _FLOAT, _SPS, N.DDT_DDT, {"floating": True}),
    ("team_mdbc2_ddt1", _SMALL, _ART, N.DDT_DDT, {"mdbc2": True}),
    ("team_mdbc2_laminar_ddt2", _SMALL, _LAM, N.DDT_DDT2, {"mdbc2": True}),
    ("team_mdbc2_sps_ddt2full", _SMALL, _SPS, N.DDT_DDT2FULL, {"mdbc2": True}),
    ("team_noddt", _SMALL, _ART, N.DDT_NONE, {}),
    ("tile_ddt1", _LARGE, _ART, N.DDT_DDT, {}),
    ("tile_ddt2", _LARGE, _ART, N.DDT_DDT2, {}),
    ("tile_noddt", _LARGE, _LAM, N.DDT_NONE, {}),
    ("tile_sps", _LARGE, _SPS, N.DDT_DDT2FULL, {}),
    ("tile_mdbc2_ddt1", _LARGE, _ART, N.DDT_DDT, {"mdbc2": True}),
    ("tile_mdbc2_laminar", _LARGE, _LAM, N.DDT_DDT2FULL, {"mdbc2": True}),
    ("tile_mdbc2_sps_ddt2", _LARGE, _SPS, N.DDT_DDT2, {"mdbc2": True}),
]


@pytest.mark.parametrize("make,tvisco,tddt,options", [x[1:] for x in OPTIONS],
                         ids=[x[0] for x in OPTIONS])
def test_options_equal_bitwise(lib, ctx, make, tvisco, tddt, options):
    """The rules of floating bodies (one lighter, one heavier than 1.2 fluid
    particles), of mDBC2 boundaries and of the density diffusion terms in the team and tile
    kernels: bits of the rows kernel, strain included."""
    a, b, npb, code = _staged_and_rows(lib, ctx, make(), tvisco, tddt, **options)
    assert np.abs(b["ace"][npb:]).max() > 0 and np.abs(b["ar"][npb:]).max() > 0
    if tvisco == _SPS:
        assert np.abs(b["sps2strain"][npb:]).max() > 0
    for k in a:
        np.testing.assert_array_equal(a[k].view(np.uint32), b[k].view(np.uint32), err_msg=k)


@pytest.mark.parametrize("dp", [0.01, 0.0072], ids=["team", "tile"])
def test_tile_kernel_equals_rows_kernel_bitwise(lib, ctx, dp):
    """The staged kernels (80k fluid particles: teams, 215k: tile) and the rows
    kernel sum the same pairs in the same order: identical bits."""
    c = perturbed_case(casemod.dam_break(dp=dp), seed=3)
    gq, _, npb = _run_both(c, 1, 3, 0.01, 0.01, lib, ctx, kernel=N.FORCES_TILE)
    gr, _, _ = _run_both(c, 1, 3, 0.01, 0.01, lib, ctx, kernel=N.FORCES_ROWS)
    lib.dsph_ctx_set_option(ctx, N.OPT_FORCES_KERNEL, N.FORCES_TILE)
    for k in ("ace", "ar", "viscdt"):
        np.testing.assert_array_equal(gq[k].view(np.uint32), gr[k].view(np.uint32))


def test_pips_counts_exact(lib, ctx):
    import oracle.oracle as orc
    c = perturbed_case(casemod.dam_break(dp=0.02))
    o, d, dcell, poscell, cte, celldiv, be = _prepared(c)
    st = o.stats()
    bc = Dev(lib, ctx, be)
    dv = divdata(celldiv, bc, cte)
    res = (C.c_uint64 * 4)()
    rc = lib.dsph_pips_count_sync(ctx, st["npbok"], 0, st["np"] - st["npb"], st["npb"],
                                  C.byref(dv), Dev(lib, ctx, dcell).ptr, Dev(lib, ctx, poscell).ptr,
                                  res)
    assert rc == 0
    assert list(res) == o.pips()


def test_sps_tau(lib, ctx):
    import oracle.oracle as orc
    n, npb = 5000, 1000
    rng = np.random.default_rng(9)
    s2 = (rng.standard_normal((n, 6)) * 10).astype(np.float32)
    vr = np.ones((n, 4), np.float32)
    vr[:, 3] = (1000 + rng.standard_normal(n)).astype(np.float32)
    tau = Dev.zeros(lib, ctx, (n, 6), np.float32)
    smag, blin = 1.9e-6, 2.2e-7
    rc = lib.dsph_sps_tau(ctx, n, npb, smag, blin, Dev(lib, ctx, vr).ptr, Dev(lib, ctx, s2).ptr,
                          tau.ptr)
    assert rc == 0
    ot = np.zeros((n, 6), np.float32)
    orc.load().orc_sps_tau(n, npb, smag, blin, vr.ctypes.data, s2.ctypes.data, ot.ctypes.data)
    assert rel_err(tau.get()[npb:], ot[npb:]) < 1e-6


def test_boundary_kernel_forms_equal_bitwise(lib, ctx):
    """The boundary interaction with staged neighbours (form 1, and 0, the
    default) and its one-lane-per-particle form (2) give the same bits
    (DSPH_OPT_BOUND_KERNEL)."""
    c = perturbed_case(casemod.dam_break(dp=0.01), seed=4)
    o, d, dcell, poscell, cte, celldiv, be = _prepared(c)
    st = o.stats()
    n, npb, npbok = st["np"], st["npb"], st["npbok"]
    bc = Dev(lib, ctx, be)
    dv = divdata(celldiv, bc, cte)
    assert lib.dsph_set_constants(ctx, C.byref(to_cte(cte))) == 0
    gd = {k: Dev(lib, ctx, a) for k, a in (("dcell", dcell), ("poscell", poscell),
                                          ("velrho", d["velrho"]), ("code", d["code"]))}
    outs = []
    try:
        for form, reps in ((N.BOUND_TILE, 1), (N.BOUND_ROWS, 1), (N.BOUND_AUTO, 1)):
            assert lib.dsph_ctx_set_option(ctx, N.OPT_BOUND_KERNEL, form) == 0
            for _ in range(reps):
                ace = Dev.zeros(lib, ctx, (n, 3), np.float32)
                ar = Dev.zeros(lib, ctx, n, np.float32)
                vdt = Dev.zeros(lib, ctx, n, np.float32)
                t = N.DsphInterParms()
                t.tkernel, t.tvisco, t.tdensity = N.KERNEL_WENDLAND, 1, 3
                t.viscob = t.viscof = 0.01
                t.np, t.npb, t.npbok = n, npb, npbok
                t.divdata = dv
                t.d_dcell, t.d_poscell = gd["dcell"].ptr, gd["poscell"].ptr
                t.d_velrho, t.d_code = gd["velrho"].ptr, gd["code"].ptr
                t.d_viscdt, t.d_ar, t.d_ace = vdt.ptr, ar.ptr, ace.ptr
                assert lib.dsph_interaction_forces(ctx, C.byref(t)) == 0, lib.dsph_last_error(ctx)
                outs.append((ar.get(), vdt.get()))
    finally:
        lib.dsph_ctx_set_option(ctx, N.OPT_BOUND_KERNEL, N.BOUND_AUTO)
    assert np.abs(outs[0][0][:npbok]).max() > 0
    for a, v in outs[1:]:
        np.testing.assert_array_equal(a.view(np.uint32), outs[0][0].view(np.uint32))
        np.testing.assert_array_equal(v.view(np.uint32), outs[0][1].view(np.uint32))
    assert lib.dsph_ctx_set_option(ctx, N.OPT_BOUND_KERNEL, 3) != 0
