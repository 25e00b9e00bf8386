"""The calls whose speed is measured, with their inputs, work and FP64 values.

Four kinds of pass, each through entry points that a user's program calls:

- ``steps``: a simulation advanced by a few time steps and its particles read
  back (``SphGpuSingle.run`` and ``download``), the program of every plain
  run between two outputs;
- ``forces``: one force interaction over a program's own device arrays (the C
  ABI's ``dsph_interaction_forces``), what the reference's host code calls;
- ``ensemble``: uneven cases advanced together and read back (``Ensemble``);
- ``infer`` and ``train``: the learned closure's network (``dsph_mlp_*``).

``listed()`` names the cases; ``draw()`` gives more of the same ranges.
"""
from __future__ import annotations

import ctypes as C
import dataclasses
import math

import numpy as np
import torch

from dualsphysics_amd import _native as N
from dualsphysics_amd import case as casemod
from dualsphysics_amd.closure import FLOP_FORWARD, FLOP_GRAD, Mlp, init_params
from dualsphysics_amd.ensemble import Ensemble, dam_break_ensemble
from dualsphysics_amd.sim import SphGpuSingle

DEV = "cuda:0"
# Options of the simulated scenes (Parameters fields), as their tests and
# benchmarks set them.
OPTIONS = {
    "artificial": {},
    "laminar_verlet": {"tstep": 1, "tvisco": N.VISCO_LAMINAR, "visco": 1e-4, "tdensity": N.DDT_DDT2},
    "mdbc_sps": {"tboundary": N.BC_MDBC, "tvisco": N.VISCO_LAMINARSPS, "visco": 1e-6},
    "mdbc2_noslip": {"tboundary": N.BC_MDBC, "slipmode": N.SLIP_NOSLIP,
                     "tvisco": N.VISCO_LAMINAR, "visco": 1e-4},
    "shifting": {"shifting": N.SHIFT_FULL, "shifttfs": 2.75},
    "ddt1": {"tdensity": N.DDT_DDT},
    "half_cells": {"cellmode": 2},
}


def listed():
    return [
        # The smallest runs: a 2-D section in seconds, where launches and
        # host round trips are the time.
        dict(name="steps_2d_2k", kind="steps", scene="dam2d", dp=0.01, opt="artificial", steps=40),
        # A coarse 3-D run (26k particles), the size of quick studies and of
        # the learned closure's coarse runs.
        dict(name="steps_3d_26k", kind="steps", scene="dam3d", dp=0.02, opt="artificial", steps=20),
        # The plain 3-D dam break (141k particles).
        dict(name="steps_3d_141k", kind="steps", scene="dam3d", dp=0.01, opt="artificial", steps=20),
        # The large dam break of the benchmark (6.08M particles).
        dict(name="steps_3d_6m", kind="steps", scene="dam3d", dp=0.0025, opt="artificial", steps=20),
        # The large 2-D dam break (3.0M particles, 36 neighbours each).
        dict(name="steps_2d_3m", kind="steps", scene="dam2d", dp=0.0002, opt="artificial", steps=20),
        # The wave flume: piston, mDBC walls, Laminar+SPS (1.2M particles).
        dict(name="steps_flume_sps", kind="steps", scene="flume", dp=0.02, opt="mdbc_sps", steps=10),
        # mDBC2 no-slip walls with laminar viscosity, an odd spacing.
        dict(name="steps_mdbc2", kind="steps", scene="dam3d", dp=0.0087, opt="mdbc2_noslip", steps=10),
        # A floating box, moved by the rigid-body update of each half step.
        dict(name="steps_floating", kind="steps", scene="floating", dp=0.0113, opt="artificial", steps=10),
        # One interaction of a developed flow in a program's own arrays.
        dict(name="forces_1m6", kind="forces", dp=0.004, visco="artificial"),
        # Uneven dam breaks in one ensemble (1.3M particles).
        dict(name="ensemble_20", kind="ensemble", n=20, steps=24),
        # The closure network in a coarse run, and one training step of it.
        dict(name="infer_1m", kind="infer", n=1000003),
        dict(name="train_4096", kind="train", n=4096),
    ]


def draw(rng):
    """One more case: sizes log-uniform over the listed ranges."""
    def log_uniform(a, b):
        return math.exp(rng.uniform(math.log(a), math.log(b)))
    kind = rng.choice(["steps"] * 6 + ["forces"] * 2 + ["ensemble", "infer", "train"])
    if kind == "steps":
        scene = rng.choice(["dam2d", "dam3d", "dam3d", "flume", "floating", "channel"])
        lo, hi = {"dam2d": (0.0002, 0.01), "dam3d": (0.0025, 0.02), "flume": (0.02, 0.04),
                  "floating": (0.008, 0.02), "channel": (0.008, 0.02)}[scene]
        opts = {"flume": ["mdbc_sps", "artificial"], "channel": ["artificial", "laminar_verlet"],
                "floating": ["artificial", "laminar_verlet"]}.get(scene, list(OPTIONS))
        return dict(kind=kind, scene=scene, dp=round(log_uniform(lo, hi), 6),
                    opt=rng.choice(opts), steps=rng.choice([5, 10, 20]))
    if kind == "forces":
        return dict(kind=kind, dp=round(log_uniform(0.004, 0.03), 6),
                    visco=rng.choice(["artificial", "laminar", "sps"]))
    if kind == "ensemble":
        return dict(kind=kind, n=rng.randrange(3, 21), steps=rng.choice([3, 12, 24]))
    if kind == "infer":
        return dict(kind=kind, n=int(log_uniform(1e3, 4e6)))
    return dict(kind=kind, n=int(log_uniform(256, 2e5)))


# ------------------------------------------------------------------ simulations
def _scene(case, seed):
    par = casemod.Parameters(**OPTIONS[case["opt"]])
    dp, seed = case["dp"], seed & 0xffffffff
    if case["scene"] == "dam2d":
        return casemod.dam_break_2d(dp=dp, seed=seed, params=par)
    if case["scene"] == "dam3d":
        return casemod.dam_break(dp=dp, seed=seed, params=par)
    if case["scene"] == "flume":
        return casemod.flume(dp=dp, length=12.0, width=1.0, height=1.2, depth=0.6, ampl=0.1,
                             period=1.6, seed=seed, params=par)
    if case["scene"] == "floating":
        return casemod.dam_break_floating(dp=dp, seed=seed, params=par)
    par = dataclasses.replace(par, periodic=1)
    return casemod.periodic_channel(dp=dp, seed=seed, params=par)


def _particles(case):
    """(particles, fluid particles, neighbours of a fluid particle)."""
    dp = case["dp"]
    if case.get("scene") == "dam2d":
        nf, nb = 0.4 * 0.3 / dp ** 2, 2 * (1.6 + 0.8) / dp
        return nf + nb, nf, math.pi * (2.4 * math.sqrt(2)) ** 2
    ng = 4 / 3 * math.pi * (2.4 * math.sqrt(3)) ** 3
    if case.get("scene") == "flume":
        nf, nb = 12 * 0.6 / dp ** 3, 2 * (12 + 2 * 12 * 1.2 + 2 * 1.2) / dp ** 2
    elif case.get("scene") == "channel":
        nf, nb = 0.4 * 0.2 * 0.15 / dp ** 3, 4 * 0.4 * 0.2 / dp ** 2
    else:
        nf, nb = 0.4 * 0.67 * 0.3 / dp ** 3, 2 * (1.6 * 0.67 + 2 * 0.4 * (1.6 + 0.67)) / dp ** 2
    return nf + nb, nf, ng


# ------------------------------------------------------------------ forces
def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _call(lib, ctx, rc):
    if rc:
        raise RuntimeError(lib.dsph_last_error(ctx).decode())


class _Forces:
    """Device arrays, neighbour list and parameters of one interaction: a dam
    break whose fluid moves (smooth velocities of about 1 m/s with noise,
    densities within a percent of hydrostatic, particles off the lattice)."""

    def __init__(self, case, seed):
        rng = np.random.default_rng(seed)
        c = casemod.dam_break(dp=case["dp"], seed=seed & 0xffffffff)
        nb, n, f32 = c.nbound, c.np, np.float32
        dp, h = c.dp, float(f32(c.h))
        pos = torch.from_numpy(c.pos).to(DEV)
        vr = torch.from_numpy(c.velrho).to(DEV)
        g = torch.Generator(device=DEV).manual_seed(seed & 0x7fffffff)
        rand = lambda *s: torch.rand(*s, device=DEV, generator=g)  # noqa: E731
        pos[nb:] += (rand(n - nb, 3).double() - 0.5) * (0.2 * dp)
        k = torch.from_numpy(rng.uniform(5, 20, (3, 3))).to(DEV)
        vr[nb:, :3] = (torch.sin(pos[nb:] @ k).float() + 0.05 * (rand(n - nb, 3) - 0.5))
        vr[nb:, 3] *= 1 + 0.01 * (rand(n - nb) - 0.5)
        # Constants (the reference's rules, as the simulations set them).
        ks = f32(h * 2.0)
        t = N.DsphCte()
        t.massb, t.massf, t.kernelh = c.massbound, c.massfluid, h
        t.kernelsize2, t.poscellsize = f32(ks * ks), ks
        t.awen, t.bwenh = 0.41778 / h ** 3, -2.08891 / h ** 5
        cteb, gamma, rho0 = float(f32(c.b)), float(f32(c.gamma)), float(f32(c.rhop0))
        t.cs0, t.eta2 = math.sqrt(gamma * cteb / rho0), (h * 0.1) ** 2
        t.ddtkh, t.ddtgz = f32(ks * f32(0.1)), rho0 * 9.81 / cteb
        t.scell = t.kernelsize = ks
        t.dp, t.cteb, t.gamma, t.rhopzero, t.ovrhopzero = dp, cteb, gamma, rho0, f32(1) / f32(rho0)
        t.movlimit, t.tboundary = f32(ks * f32(0.9)), N.BC_DBC
        mn, mx = np.array(c.maprealposmin), np.array(c.maprealposmax)
        nc = [int(v) for v in np.ceil((mx - mn) / float(ks))]
        bits = [max(2, (v + 1).bit_length()) for v in nc]
        for i in range(31 - sum(bits)):   # all 31 bits are used, x first
            bits[i % 3] += 1
        sx, sy, sz = bits
        t.cellcode = ((sx + 1) << 25 | sy << 20 | sz << 15 | (sy + sz) << 10 | (sx + 1 + sz) << 5 |
                      (sx + 1 + sy))
        for a, v in zip("xyz", mn):
            setattr(t, f"domposmin{a}", v)
            setattr(t, f"maprealposmin{a}", v)
        for a, v in zip("xyz", mx - mn):
            setattr(t, f"maprealsize{a}", v)
        self.cte = t
        # Neighbour list over the whole map.
        cell = ((pos - torch.from_numpy(mn).to(DEV)) / float(ks)).to(torch.int32)
        dcell = (cell[:, 0] << (sy + sz)) | (cell[:, 1] << sz) | cell[:, 2]
        code = torch.zeros(n, dtype=torch.int16, device=DEV)
        code[nb:] = 0x1800
        idp = torch.arange(n, dtype=torch.int32, device=DEV)
        xy, z = pos[:, :2].contiguous(), pos[:, 2].contiguous()
        nct = nc[0] * nc[1] * nc[2]
        lib = self.lib = N.load()
        self.ctx = C.c_void_p()
        if lib.dsph_ctx_create(0, C.byref(self.ctx)):
            raise RuntimeError("no context")
        _call(lib, self.ctx, lib.dsph_ctx_reserve(self.ctx, n, 2 * nct + 5))
        _call(lib, self.ctx, lib.dsph_set_constants(self.ctx, C.byref(t)))
        i32 = dict(dtype=torch.int32, device=DEV)
        keys, order = torch.empty(n, **i32), torch.empty(n, **i32)
        self.begin = torch.zeros(2 * nct + 5, 2, **i32)
        self.vr, self.dcell, self.code = torch.empty_like(vr), torch.empty_like(dcell), torch.empty_like(code)
        self.ps = torch.empty_like(vr)
        outs = [torch.empty_like(idp), self.code, self.dcell, torch.empty_like(xy), torch.empty_like(z), self.vr]
        torch.cuda.synchronize()
        u3 = lambda v: (C.c_uint32 * 3)(*v)  # noqa: E731
        _call(lib, self.ctx, lib.dsph_presort_full(self.ctx, n, t.cellcode, _ptr(dcell), _ptr(code),
                                                   u3([0, 0, 0]), u3(nc), _ptr(keys), _ptr(order)))
        _call(lib, self.ctx, lib.dsph_sort_by_cell(self.ctx, _ptr(keys), _ptr(order), n, 2 * nct + 5))
        _call(lib, self.ctx, lib.dsph_begin_end_cell(self.ctx, 1, n, nb, 2 * nct + 5, nct + 1,
                                                     _ptr(keys), _ptr(self.begin)))
        _call(lib, self.ctx, lib.dsph_sort_data_basic_poscell(
            self.ctx, n, 0, _ptr(order), _ptr(idp), _ptr(code), _ptr(dcell), _ptr(xy), _ptr(z),
            _ptr(vr), *[_ptr(o) for o in outs], (C.c_double * 3)(*mn), ks, _ptr(self.ps)))
        _call(lib, self.ctx, lib.dsph_synchronize(self.ctx))
        self.n, self.nb, self.nc, self.visco = n, nb, nc, case["visco"]
        zero = lambda *s: torch.zeros(*s, device=DEV)  # noqa: E731
        self.viscdt, self.ar, self.ace = zero(n), zero(n), zero(n, 3)
        p = N.DsphInterParms()
        p.tkernel, p.tdensity = N.KERNEL_WENDLAND, N.DDT_DDT2FULL
        p.tvisco = {"artificial": N.VISCO_ARTIFICIAL, "laminar": N.VISCO_LAMINAR,
                    "sps": N.VISCO_LAMINARSPS}[self.visco]
        p.viscob = p.viscof = 0.01 if self.visco == "artificial" else 1e-4
        p.np, p.npb, p.npbok = n, nb, nb
        d = p.divdata
        d.scelldiv, d.ncx, d.ncy, d.ncz = 1, *nc
        d.ncw, d.cellfluid, d.d_beginendcell = nc[0] * nc[1], nct + 1, self.begin.data_ptr()
        d.scell, d.domcellcode, d.kernelsize2, d.poscellsize = t.scell, t.cellcode, t.kernelsize2, ks
        d.domposminx, d.domposminy, d.domposminz = mn
        p.d_dcell, p.d_poscell, p.d_velrho = self.dcell.data_ptr(), self.ps.data_ptr(), self.vr.data_ptr()
        p.d_code = self.code.data_ptr()
        p.d_viscdt, p.d_ar, p.d_ace = self.viscdt.data_ptr(), self.ar.data_ptr(), self.ace.data_ptr()
        self.tau = self.strain = None
        if self.visco == "sps":
            self.tau, self.strain = 1e-6 * (rand(n, 6) - 0.5), zero(n, 6)
            self.tau[:nb] = 0
            p.d_spstaurho2, p.d_sps2strain = self.tau.data_ptr(), self.strain.data_ptr()
        self.p = p

    def run(self):
        lib, ctx = self.lib, self.ctx
        outs = [self.ace, self.ar, self.viscdt] + ([self.strain] if self.strain is not None else [])
        for o in outs:
            _call(lib, ctx, lib.dsph_memset_async(ctx, _ptr(o), 0, 4 * o.numel()))
        _call(lib, ctx, lib.dsph_interaction_forces(ctx, C.byref(self.p)))
        return outs

    def exact(self):
        """The interaction in FP64 (pairs within 2h, the formulas of
        JSphGpu_ker.cu:450-777): per block of particles, the candidates of
        their 27 cells and the sums over the real pairs."""
        t, nb, n = self.cte, self.nb, self.n
        w = self.ps[:, 3].contiguous().view(torch.int32)
        pcell = torch.stack([(w >> 19) & 0x1fff, (w >> 9) & 0x3ff, w & 0x1ff], 1)
        vr = self.vr.double()
        q = self.ps[:, :3].double()
        rho = vr[:, 3]
        press = t.cteb * ((rho * t.ovrhopzero) ** t.gamma - 1)
        ncx, ncy, ncz = self.nc
        cell = pcell.long()   # PosCell cells are the search cells (full cells, origin of the map)
        begin = self.begin.long()
        out = {k: torch.zeros(n, m, dtype=torch.float64, device=DEV)
               for k, m in (("ace", 3), ("ar", 1), ("visc", 1), ("strain", 6))}
        vis = self.p.viscof

        def rows(p1, bound2):
            base = 0 if bound2 else ncx * ncy * ncz + 1
            x0 = (cell[p1, 0] - 1).clamp(min=0)
            x1 = (cell[p1, 0] + 1).clamp(max=ncx - 1)
            for dz in (-1, 0, 1):
                for dy in (-1, 0, 1):
                    y, z = cell[p1, 1] + dy, cell[p1, 2] + dz
                    ok = (y >= 0) & (y < ncy) & (z >= 0) & (z < ncz)
                    row = base + (z.clamp(0, ncz - 1) * ncy + y.clamp(0, ncy - 1)) * ncx
                    for dx in (0, 1, 2):
                        cx = x0 + dx
                        b = begin[row + cx.clamp(max=ncx - 1)]
                        cnt = torch.where(ok & (cx <= x1), b[:, 1] - b[:, 0], 0)
                        yield b[:, 0], cnt

        def pairs(p1, bound2):
            for b0, cnt in rows(p1, bound2):
                tot = int(cnt.sum())
                if not tot:
                    continue
                i = torch.repeat_interleave(torch.arange(len(p1), device=DEV), cnt)
                j = torch.arange(tot, device=DEV) - (cnt.cumsum(0) - cnt)[i] + b0[i]
                a = p1[i]
                dr = q[a] - q[j] + float(t.poscellsize) * (pcell[a] - pcell[j]).double()
                rr2 = (dr * dr).sum(1)
                keep = (rr2 <= t.kernelsize2) & (rr2 >= 1e-18)
                yield a[keep], j[keep], dr[keep], rr2[keep]

        for bound1 in (False, True):
            lo, hi = (0, nb) if bound1 else (nb, n)
            for s in range(lo, hi, 100000):
                p1 = torch.arange(s, min(s + 100000, hi), device=DEV)
                for bound2 in ((False,) if bound1 else (False, True)):
                    for a, j, dr, rr2 in pairs(p1, bound2):
                        m2 = t.massb if bound2 else t.massf
                        fac = t.bwenh * (1 - 0.5 * rr2.sqrt() / t.kernelh) ** 3
                        fr = fac[:, None] * dr
                        dv = vr[a, :3] - vr[j, :3]
                        out["ar"].index_add_(0, a, (m2 * (dv * fr).sum(1) * rho[a] / rho[j])[:, None])
                        dot = (dr * dv).sum(1)
                        inv = 1 / (rr2 + t.eta2)
                        out["visc"].index_reduce_(0, a, (dot * inv)[:, None], "amax")
                        if bound1:
                            continue
                        acc = -m2 * ((press[a] + press[j]) / (rho[a] * rho[j]))[:, None] * fr
                        dot3 = (dr * fr).sum(1)
                        if not bound2:
                            drho = t.rhopzero * (1 + t.ddtgz * dr[:, 2]) ** (1 / t.gamma) - t.rhopzero
                            d = t.ddtkh * t.cs0 * (rho[j] - rho[a] - drho) * inv * dot3 * m2 / rho[j]
                            out["ar"].index_add_(0, a, -d[:, None])
                        if self.visco == "artificial":
                            amu = t.kernelh * dot * inv
                            pi = torch.where(dot < 0, -vis * t.cs0 * amu / ((rho[a] + rho[j]) * 0.5), 0.0) * m2
                            acc = acc - pi[:, None] * fr
                        else:
                            vt = m2 * 4 * vis / ((rr2 + t.eta2) * (rho[a] + rho[j])) * dot3
                            acc = acc + vt[:, None] * dv
                        if self.visco == "sps":
                            tau = self.tau[a].double() + (0 if bound2 else self.tau[j].double())
                            x, y, z = fr.unbind(1)
                            sx, sy, sz = (tau[:, [0, 1, 2]], tau[:, [1, 3, 4]], tau[:, [2, 4, 5]])
                            acc = acc + m2 * torch.stack([(r * fr).sum(1) for r in (sx, sy, sz)], 1)
                            u = dv * (-m2 / rho[j])[:, None]
                            out["strain"].index_add_(0, a, torch.stack(
                                [u[:, 0] * x, u[:, 0] * y + u[:, 1] * x, u[:, 0] * z + u[:, 2] * x,
                                 u[:, 1] * y, u[:, 1] * z + u[:, 2] * y, u[:, 2] * z], 1))
                        out["ace"].index_add_(0, a, acc)
        res = [out["ace"], out["ar"][:, 0], out["visc"][:, 0]]
        return res + ([out["strain"]] if self.strain is not None else [])

    def __del__(self):
        try:
            self.lib.dsph_ctx_destroy(self.ctx)
        except Exception:
            pass


# ------------------------------------------------------------------ network
class _Net:
    """The closure network with its device batch: features as a coarse run's
    interaction gives them (velocity gradients of tens per second, densities
    near 1000, one dp) and eddy viscosities of about 1e-5 m2/s."""

    def __init__(self, case, seed):
        n, rng = case["n"], np.random.default_rng(seed)
        g = torch.Generator(device=DEV).manual_seed(seed & 0x7fffffff)
        self.n = n
        self.feats = torch.empty(n, 11, device=DEV)
        self.feats[:, :9] = 30 * torch.randn(n, 9, device=DEV, generator=g)
        self.feats[:, 9] = 1000 + 5 * torch.randn(n, device=DEV, generator=g)
        self.feats[:, 10] = 0.02
        self.targets = 1e-5 * torch.rand(n, device=DEV, generator=g)
        self.mean = np.array([0] * 9 + [1000, 0.02], np.float32)
        self.scale = np.array([1 / 30] * 9 + [0.2, 0], np.float32)
        self.out_scale = 5e-6
        self.lib = N.load()
        self.ctx = C.c_void_p()
        if self.lib.dsph_ctx_create(0, C.byref(self.ctx)):
            raise RuntimeError("no context")
        self.params = init_params(int(rng.integers(1 << 30)))
        self.net = Mlp(self.lib, self.ctx, self.params, self.mean, self.scale, self.out_scale)
        np_ = self.net.nparam
        self.out = torch.empty(n, device=DEV)
        self.grad, self.loss = torch.empty(np_, device=DEV), torch.empty(1, device=DEV)
        self.scratch = torch.empty(1024 * (np_ + 1), device=DEV)
        torch.cuda.synchronize()

    def run(self, train):
        lib, ctx, m = self.lib, self.ctx, C.byref(self.net.m)
        if not train:
            _call(lib, ctx, lib.dsph_mlp_forward(ctx, m, self.n, _ptr(self.feats), _ptr(self.out)))
            return self.out
        _call(lib, ctx, lib.dsph_mlp_grad(ctx, m, self.n, _ptr(self.feats), _ptr(self.targets),
                                          _ptr(self.scratch), 4 * self.scratch.numel(),
                                          _ptr(self.grad), _ptr(self.loss)))
        return [self.grad, self.loss]

    def exact(self, train):
        p = torch.from_numpy(self.params).to(DEV).double().requires_grad_(True)
        w1, b1 = p[:1024].view(64, 16)[:, :11], p[1024:1088]
        w2, b2 = p[1088:5184].view(64, 64), p[5184:5248]
        w3, b3 = p[5248:5312], p[5312]
        x = (self.feats.double() - torch.from_numpy(self.mean).to(DEV)) * torch.from_numpy(self.scale).to(DEV)
        silu, softplus = torch.nn.functional.silu, torch.nn.functional.softplus
        y = softplus(silu(silu(x @ w1.T + b1) @ w2.T + b2) @ w3 + b3)
        if not train:
            return (self.out_scale * y).detach()
        loss = ((y - self.targets.double() / self.out_scale) ** 2).mean()
        loss.backward()
        return [p.grad, loss.detach().reshape(1)]

    def __del__(self):
        try:
            self.net.free()
            self.lib.dsph_ctx_destroy(self.ctx)
        except Exception:
            pass


# ------------------------------------------------------------------ the passes
def prepare(case, seed):
    kind = case["kind"]
    if kind == "steps":
        return kind, case, SphGpuSingle(_scene(case, seed))
    if kind == "forces":
        return kind, case, _Forces(case, seed)
    if kind == "ensemble":
        # The benchmark ensemble's own sizes, every particle shifted by up to
        # 1e-4 dp from the seed; far from their end times.
        rng, cases = np.random.default_rng(seed), []
        for c in dam_break_ensemble(case["n"]):
            off = rng.uniform(-1e-4 * c.dp, 1e-4 * c.dp, c.pos.shape)
            cases.append(dataclasses.replace(c, pos=c.pos + off))
        e = Ensemble(cases, 100.0)
        e.autotune(1)
        return kind, case, e
    return kind, case, _Net(case, seed)


def run(state):
    kind, case, s = state
    if kind == "steps":
        s.run(case["steps"])
        return s.download()
    if kind == "forces":
        return s.run()
    if kind == "ensemble":
        s.run(case["steps"])
        got = [s.download(i) for i in range(case["n"])]
        return [[d["idp"], d["pos"], d["velrho"]] for d in got]
    return s.run(kind == "train")


def work(case):
    """Bytes and FP32 operations of one pass. A time step reads and writes the
    state (id, code, cell, FP64 position, velocity and density: 50 bytes) in
    each of its half steps and does two interactions (Verlet: one of each), 79
    operations a pair."""
    kind = case["kind"]
    if kind == "infer":
        return {"bytes": 48.0 * case["n"], "flops": float(FLOP_FORWARD) * case["n"]}
    if kind == "train":
        return {"bytes": 48.0 * case["n"] + 2 * 21252, "flops": float(FLOP_GRAD) * case["n"]}
    if kind == "ensemble":
        npart, nf, ng = 64000.0 * case["n"], 33000.0 * case["n"], _particles({"dp": 1})[2]
        k = case["steps"] // 3 * 3
        return {"bytes": 200.0 * npart * k, "flops": 2 * 79 * nf * ng * k}
    npart, nf, ng = _particles(case)
    if kind == "forces":
        sps = case["visco"] == "sps"
        return {"bytes": 36.0 * npart + (20 + 48 * sps) * npart, "flops": (79 + 40 * sps) * nf * ng}
    inter = 1 if OPTIONS[case["opt"]].get("tstep") == 1 else 2
    return {"bytes": 100.0 * inter * npart * case["steps"], "flops": 79 * inter * nf * ng * case["steps"]}


def exact(case, seed):
    if case["kind"] in ("steps", "ensemble"):
        return None   # several steps of a whole solver
    s = prepare(case, seed)[2]
    return s.exact() if case["kind"] == "forces" else s.exact(case["kind"] == "train")
