"""The work a user has this framework do, as cases that can be timed and
checked one by one through the package's public entry points.

  listed()               the cases, each a dict of plain values
  draw(rng)              one more case of the same ranges
  prepare(case, seed)    what a flow solver holds before the call, on the GPU
  run(state)             one pass; returns its outputs
  work(case)             bytes and operations one pass cannot do without
  exact(case, seed)      run's outputs in 64 bits from plain torch

Kinds of a case:
  poisson          pp_solve_device from p = 0 (the pressure solve of a step)
  adjoint          pp_adjoint_device of a pressure-force objective
  momentum         pp_solve_ad_device / pp_solve_ad_cn2_device (u, v, w)
  correct_vel      pp_correct_vel_device
  update_pressure  pp_update_pressure_device
  divergence       pp_divergence_noalloc
  projection       divergence, solve, correct_vel and update_pressure in turn
  moving           geometry, pp_set_geometry and the solve of a moving body
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from flow_structure_interaction_fem_ibm_amd import pp

DEV = "cuda:0"
F8 = torch.float64
DT = 1e-3          # time step of the momentum and projection cases
NU = 1e-3          # viscosity of the momentum cases
SCHEMES = {"AB": pp.PP_ADAMS_BASHFORTH2, "CN1": pp.PP_CRANK_NICOLSON1, "CN2": pp.PP_CRANK_NICOLSON2}


def listed():
    return [
        # a laminar test case on a laptop-sized grid: launch latency decides
        dict(name="poisson_24", kind="poisson", nx=24, ny=24, nz=24, beta=1.5, bodies=1, fp64=False, tol=1e-8),
        # odd counts in every direction: nothing halves evenly on the finest level
        dict(name="poisson_65x49x41", kind="poisson", nx=65, ny=49, nz=41, beta=1.5, bodies=1, fp64=False, tol=1e-10),
        # the headline solve: 9.4 million cells, one ellipsoid, FP32 cycles
        dict(name="poisson_256", kind="poisson", nx=256, ny=192, nz=192, beta=2.0, bodies=0, fp64=False, tol=1e-8),
        # the same solve with FP64 cycles
        dict(name="poisson_256_fp64", kind="poisson", nx=256, ny=192, nz=192, beta=2.0, bodies=0, fp64=True, tol=1e-8),
        # the largest grid in use: 1e8 cells with 64 bodies
        dict(name="poisson_512", kind="poisson", nx=512, ny=512, nz=384, beta=1.5, bodies=64, fp64=False, tol=1e-8),
        # gradient of a body's pressure force with respect to the divergence
        dict(name="adjoint_256", kind="adjoint", nx=256, ny=192, nz=192, beta=2.0, bodies=0, tol=1e-8),
        # the implicit momentum step on the headline grid
        dict(name="momentum_256", kind="momentum", nx=256, ny=192, nz=192, beta=2.0, bodies=0, scheme="CN1"),
        # a smaller momentum step on a ragged grid, face velocities updated in the loop
        dict(name="momentum_cn2_130x98x82", kind="momentum", nx=130, ny=98, nz=82, beta=1.5, bodies=1, scheme="CN2"),
        # the two cheapest steps either side of the solve: one pass over the fields
        dict(name="correct_vel_256", kind="correct_vel", nx=256, ny=192, nz=192, beta=2.0, bodies=0),
        dict(name="divergence_256", kind="divergence", nx=256, ny=192, nz=192, beta=2.0, bodies=0),
        # a whole projection step on a small grid, fields resident
        dict(name="projection_128x96x96", kind="projection", nx=128, ny=96, nz=96, beta=2.0, bodies=1, tol=1e-8),
        # a step of a moving sphere: geometry on the GPU, set-up, solve
        dict(name="moving_384", kind="moving", nx=384, ny=256, nz=256, beta=2.0, bodies=1, tol=1e-10),
    ]


def draw(rng):
    """A case of the listed ranges: 24 to 512 cells along x, the other
    directions 0.6 to 1 times that, odd counts among them."""
    kind = rng.choice(["poisson", "poisson", "poisson", "adjoint", "momentum", "momentum", "correct_vel",
                       "update_pressure", "divergence", "projection", "moving"])
    top = {"poisson": 512, "adjoint": 320, "momentum": 320, "moving": 384}.get(kind, 448)
    nx = round(math.exp(rng.uniform(math.log(24.0), math.log(top))))
    ny, nz = (max(20, round(nx * rng.uniform(0.6, 1.0))) for _ in range(2))
    if rng.random() < 0.5:
        nx, ny, nz = (8 * ((n + 7) // 8) for n in (nx, ny, nz))
    nz = min(nz, int(9e7 / (nx * ny)))
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz, beta=rng.choice([0.0, 1.0, 1.5, 2.0] if nx >= 48 else [0.0, 1.0, 1.5]),
                bodies=1)
    if min(nx, ny, nz) >= 160 and kind != "moving":
        case["bodies"] = rng.choice([0, 1, 1, rng.randint(2, 24)])
    if kind == "poisson":
        case["fp64"] = nx <= 320 and rng.random() < 0.3
    if kind == "momentum":
        case["scheme"] = rng.choice(["AB", "CN1", "CN1", "CN2"])
    if kind in ("poisson", "adjoint", "projection", "moving"):
        case["tol"] = rng.choice([1e-8, 1e-8, 1e-10])
    return case


# ---------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------
def _grid(case):
    """Node coordinates: 4 long in x, equal mean spacing; x uniform unless
    there are many bodies, y and z clustered at the centre."""
    n = (case["nx"], case["ny"], case["nz"])
    b = case["beta"]
    return [pp.tanh_nodes(m, 4.0 * m / n[0], b if d or case["bodies"] > 1 else 0.0) for d, m in enumerate(n)]


def _bodies(case, nodes, shift=0.0):
    L = [float(a[-1]) for a in nodes]
    if case["bodies"] == 0:  # one prolate ellipsoid, rotated
        return [pp.Ellipsoid((0.375 * L[0], 0.5 * L[1], 0.5 * L[2]), (0.5, 0.25, 0.25), 20.0, 96)]
    if case["bodies"] == 1:  # a sphere at least 8 mean cells in radius where the box allows it
        r = min(0.2, max(0.075, 8.0 / min(case["nx"], case["ny"], case["nz"]))) * min(L)
        return [pp.Ellipsoid((0.45 * L[0] + shift, 0.5 * L[1], 0.5 * L[2]), (r, r, r), 0.0, 48)]
    rng = np.random.Generator(np.random.PCG64(5))
    h = max(float(np.diff(a).max()) for a in nodes)
    found = []
    for _ in range(20000):
        if len(found) == case["bodies"]:
            break
        r = rng.uniform(0.05, 0.15)
        if any(2 * (r + 4 * h) >= length for length in L):
            continue
        c = [rng.uniform(r + 4 * h, length - r - 4 * h) for length in L]
        if all(np.linalg.norm(np.subtract(c, q)) >= r + s + 3 * h for q, s in found):
            found.append((c, r))
    return [pp.Ellipsoid(tuple(c), (r, r, r), 0.0, 48) for c, r in found]


def _geometry(case):
    """Grid and geometry of a case (they do not depend on the seed)."""
    nodes = _grid(case)
    if case["kind"] == "moving":
        prev = pp.build_geometry(*nodes, _bodies(case, nodes, -2.5 / case["nx"]), mode=pp.PP_GEOM_TRIANGULATED, device=0)[0]
        ib, fr, gs, ex = pp.build_geometry(*nodes, _bodies(case, nodes), mode=pp.PP_GEOM_TRIANGULATED,
                                           iblank_prev=prev, device=0)
        ex["prev"] = prev
    else:
        ib, fr, gs, ex = pp.build_geometry(*nodes, _bodies(case, nodes), mode=pp.PP_GEOM_ANALYTIC)
    return nodes, ib, gs, ex


def _noise(gen, shape):
    return torch.randn(shape, generator=gen, dtype=F8, device=DEV)


def _inner(a):
    return a[1:-2, 1:-2, 1:-2]


def _centres(nodes):
    return [torch.from_numpy(0.5 * (a[1:] + a[:-1])).to(DEV) for a in nodes]


def _faces(nodes, shape, gen):
    """Face velocities N(0,1) under an envelope that vanishes on the outer
    boundary, in the reference layout (face i at index i)."""
    out = []
    sines = [[torch.sin(math.pi * torch.from_numpy(a).to(DEV) / a[-1]) for a in nodes],
             [torch.sin(math.pi * c / float(a[-1])) for c, a in zip(_centres(nodes), nodes)]]
    for d in range(3):
        f = torch.zeros(shape, dtype=F8, device=DEV)
        env = [sines[0 if q == d else 1][q] for q in range(3)]
        sub = f[1:1 + len(env[2]), 1:1 + len(env[1]), 1:1 + len(env[0])]
        sub.copy_(_noise(gen, sub.shape))
        sub *= env[2][:, None, None] * env[1][None, :, None] * env[0][None, None, :]
        out.append(f)
    return out


def _divergence(nodes, faces, fluid, dtinv):
    w = [torch.from_numpy(np.diff(a)).to(DEV) for a in nodes]
    u, v, s = faces
    d = ((u[1:-2, 1:-2, 2:-1] - _inner(u)) / w[0][None, None, :] + (v[1:-2, 2:-1, 1:-2] - _inner(v)) / w[1][None, :, None]
         + (s[2:-1, 1:-2, 1:-2] - _inner(s)) / w[2][:, None, None])
    out = torch.zeros_like(u)
    _inner(out).copy_(dtinv * d * fluid)
    return out


def _smooth(nodes, shape, gen, modes=4):
    """A smooth random field of amplitude 1: products of random cosines."""
    f = torch.ones(shape, dtype=F8, device=DEV)
    for d, a in enumerate(nodes):
        x = torch.linspace(0.0, 1.0, shape[2 - d], dtype=F8, device=DEV)
        c = torch.randn(modes, generator=gen, dtype=F8, device=DEV)
        s = sum(c[m] * torch.cos(math.pi * (m + 1) * x) for m in range(modes))
        f = f * (s / s.abs().max()).reshape([-1 if q == 2 - d else 1 for q in range(3)])
    return f


def _force_weights(nodes, ib):
    """w with sum(w * p) the x pressure force on the bodies."""
    w = torch.zeros(ib.shape, dtype=F8, device=DEV)
    dy, dz = (torch.from_numpy(np.diff(nodes[d])).to(DEV) for d in (1, 2))
    fl = _inner(ib) == 0
    up = (fl & (ib[1:-2, 1:-2, 2:-1] == 1)).to(F8)
    dn = (fl & (ib[1:-2, 1:-2, 0:-3] == 1)).to(F8)
    _inner(w).copy_(dz[:, None, None] * dy[None, :, None] * (up - dn))
    return w


def _inputs(case, seed, nodes, ib, gs):
    """The fields of a case, made on the GPU from the seed."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1000003 * (seed + 1))
    shape = ib.shape
    ibt = torch.from_numpy(ib).to(DEV)
    fluid = (_inner(ibt) == 0).to(F8)
    kind = case["kind"]
    if kind == "poisson":
        return dict(rhs=_divergence(nodes, _faces(nodes, shape, gen), fluid, 1.0))
    if kind == "moving":
        rhs = torch.zeros(shape, dtype=F8, device=DEV)
        _inner(rhs).copy_(_noise(gen, fluid.shape) * fluid)
        return dict(rhs=rhs, guess=_smooth(nodes, shape, gen) * _mask(shape))
    if kind == "adjoint":
        # the force objective plus a smooth observation of the field
        return dict(w=_force_weights(nodes, ibt) + 1e-3 * _smooth(nodes, shape, gen) * (1 - ibt.to(F8)) * _mask(shape))
    if kind == "divergence":
        return dict(faces=_faces(nodes, shape, gen))
    vel = [_smooth(nodes, shape, gen) + 0.1 * _noise(gen, shape) for _ in range(3)]
    bc = [_smooth(nodes, shape, gen) for _ in range(3)]
    if kind == "correct_vel":
        return dict(p=_smooth(nodes, shape, gen) + 0.01 * _noise(gen, shape), vel=vel, faces=_faces(nodes, shape, gen), bc=bc,
                    vbi=0.1 * _noise(gen, (gs.n, 3)))
    if kind == "update_pressure":
        return dict(p=_smooth(nodes, shape, gen), pprime=_smooth(nodes, shape, gen))
    if kind == "momentum":
        return dict(vel=vel, nl=[v + 0.1 * _noise(gen, shape) for v in vel], faces=_faces(nodes, shape, gen),
                    visc=torch.full(shape, NU, dtype=F8, device=DEV), p=_smooth(nodes, shape, gen), bc=bc,
                    vbi=0.1 * _noise(gen, (gs.n, 3)))
    return dict(vel=vel, faces=_faces(nodes, shape, gen), bc=bc, p=_smooth(nodes, shape, gen),
                vbi=0.1 * _noise(gen, (gs.n, 3)))


def _mask(shape):
    m = torch.zeros(shape, dtype=F8, device=DEV)
    _inner(m).fill_(1.0)
    return m


def prepare(case, seed):
    nodes, ib, gs, ex = _geometry(case)
    s = dict(case=case, nodes=nodes, **_inputs(case, seed, nodes, ib, gs))
    solver = pp.PressureSolver(*nodes)
    s["solver"] = solver
    kind = case["kind"]
    if kind == "moving":
        s["prev"], s["bodies"] = ex["prev"], _bodies(case, nodes)
    else:
        solver.set_geometry(ib, gs)
    if kind in ("poisson", "projection", "divergence"):
        s["sol"] = torch.zeros(ib.shape, dtype=F8, device=DEV)
        s["div"] = torch.zeros(ib.shape, dtype=F8, device=DEV)
    if kind == "moving":
        s["sol"] = torch.zeros(ib.shape, dtype=F8, device=DEV)
    if kind in ("correct_vel", "momentum", "projection"):
        solver.set_vel_ghosts(ex["coeffD"], 2.0, 1.0)
    if kind == "momentum":
        solver.set_solve_ad_device(DT, s["visc"], s["visc"], s["visc"], s["visc"])
    if kind in ("momentum", "projection"):
        s["out"] = [v.clone() for v in s["vel"]]
        s["fout"] = [f.clone() for f in s["faces"]]
    if kind == "adjoint":
        s["lam"] = torch.zeros(ib.shape, dtype=F8, device=DEV)
        s["dg"] = torch.zeros(gs.n, dtype=F8, device=DEV)
    torch.cuda.synchronize()
    return s


def run(s):
    case, solver = s["case"], s["solver"]
    kind = case["kind"]
    if kind == "poisson":
        s["sol"].zero_()
        solver.solve_device(s["sol"], s["rhs"], rel_tol=case["tol"],
                            precision=pp.PP_PREC_FP64 if case["fp64"] else pp.PP_PREC_MIXED)
        return s["sol"]
    if kind == "adjoint":
        solver.adjoint_device(s["w"], s["lam"], s["dg"], rel_tol=case["tol"])
        return s["lam"], s["dg"]
    if kind == "momentum":
        for a, b in zip(s["out"], s["vel"]):
            a.copy_(b)
        if case["scheme"] != "CN2":
            solver.solve_ad_device(SCHEMES[case["scheme"]], *s["out"], *s["nl"], *s["faces"], vel_bi=s["vbi"])
            return s["out"]
        for a, b in zip(s["fout"], s["faces"]):
            a.copy_(b)
        st = pp.ADStats()
        t = s["out"] + s["nl"] + s["fout"]
        rc = pp.lib().pp_solve_ad_cn2_device(solver.h, *[a.data_ptr() for a in t], 1, s["p"].data_ptr(),
                                             *[a.data_ptr() for a in s["bc"]], s["vbi"].data_ptr(), 1000, 1e-10,
                                             ctypes.byref(st))
        if rc not in (pp.PP_OK, pp.PP_NOT_CONVERGED):
            raise pp.PPError(rc, pp.lib().pp_last_error().decode())
        return s["out"], s["fout"]
    if kind == "correct_vel":
        solver.correct_vel_device(DT, s["p"], *s["vel"], *s["faces"], *s["bc"], vel_bi=s["vbi"])
        return s["vel"], s["faces"]
    if kind == "update_pressure":
        solver.update_pressure_device(1, s["pprime"], s["p"])
        return s["p"]
    if kind == "divergence":
        total = solver.divergence_noalloc(*s["faces"], s["div"], dtinv=1.0 / DT)
        return s["div"], total
    if kind == "projection":
        for a, b in zip(s["out"] + s["fout"], s["vel"] + s["faces"]):
            a.copy_(b)
        solver.divergence_noalloc(*s["fout"], s["div"], dtinv=1.0 / DT, want_sum=False)
        s["sol"].zero_()
        solver.solve_device(s["sol"], s["div"], rel_tol=case["tol"])
        solver.correct_vel_device(DT, s["sol"], *s["out"], *s["fout"], *s["bc"], vel_bi=s["vbi"])
        solver.update_pressure_device(1, s["sol"], s["p"])
        return s["sol"], s["out"], s["fout"], s["p"]
    ib, fresh, ghosts, _ = pp.build_geometry(*s["nodes"], s["bodies"], mode=pp.PP_GEOM_TRIANGULATED,
                                             iblank_prev=s["prev"], device=0)
    solver.set_geometry(ib, ghosts, fresh=fresh)
    s["sol"].copy_(s["guess"])
    solver.solve_device(s["sol"], s["rhs"], rel_tol=case["tol"])
    return s["sol"], ib


def work(case):
    """Fields read and written once (8 bytes a value), and the operations of
    one application of each operator the pass must apply."""
    cells = float(case["nx"] * case["ny"] * case["nz"])
    fields, flops = {"poisson": (2, 13), "adjoint": (2, 13), "momentum": (18, 3 * 15), "correct_vel": (16, 45),
                     "update_pressure": (3, 1), "divergence": (4, 10), "projection": (20, 70),
                     "moving": (3, 13)}[case["kind"]]
    return {"bytes": 8.0 * fields * cells, "flops": flops * cells}


# ---------------------------------------------------------------------
# the same results in 64 bits from plain torch
# ---------------------------------------------------------------------
# the 2x2x2 stencil of a ghost cell: offsets (i, j, k) in coefficient order
CORNERS = np.array([[0, 0, 0], [0, 1, 0], [1, 1, 0], [1, 0, 0], [0, 0, 1], [0, 1, 1], [1, 1, 1], [1, 0, 1]])


class _Discrete:
    """The discrete operators of a case on torch tensors."""

    def __init__(self, case):
        self.nodes, ib, self.gs, self.ex = _geometry(case)
        gs = self.gs
        self.ib = ib
        self.n = [len(a) - 1 for a in self.nodes]
        self.shape = ib.shape
        ibt = torch.from_numpy(ib).to(DEV)
        self.blank = _inner(ibt) == 1
        self.fluid = (~self.blank).to(F8)
        ey, ex = self.shape[1], self.shape[2]
        gid = gs.ig.astype(np.int64) + ex * (gs.jg.astype(np.int64) + ey * gs.kg)
        self.gid = torch.from_numpy(gid).to(DEV)
        ghost = np.zeros(ib.size, bool)
        ghost[gid] = True
        self.ghost = _inner(torch.from_numpy(ghost.reshape(self.shape)).to(DEV))
        own = np.zeros((gs.n, 8), bool)
        ids = np.zeros((2, gs.n, 8), np.int64)  # stencil offsets as they are, and kept off the outer layer
        for r, (a, b, c) in enumerate(CORNERS):
            raw = [gs.ic + a, gs.jc + b, gs.kc + c]
            own[:, r] = (raw[0] == gs.ig) & (raw[1] == gs.jg) & (raw[2] == gs.kg)
            for t in range(2):
                i, j, k = raw if t == 0 else [np.clip(x, 1, m) for x, m in zip(raw, self.n)]
                ids[t, :, r] = i.astype(np.int64) + ex * (j.astype(np.int64) + ey * k.astype(np.int64))
        solid = (ib.reshape(-1)[ids[1]] == 1) & ~ghost[ids[1]] & ~own
        self.solid_corners = int(solid.sum())
        self.stencil = torch.from_numpy(ids[1]).to(DEV)
        self.stencil_raw = torch.from_numpy(ids[0]).to(DEV)
        self.own = torch.from_numpy(own).to(DEV)
        self.cN = torch.from_numpy(np.where(own | solid, 0.0, gs.coeff)).to(DEV)
        self.cB = torch.from_numpy((gs.coeff * own).sum(1) + gs.probe).to(DEV)
        self.cD = torch.from_numpy(np.ascontiguousarray(self.ex["coeffD"])).to(DEV)
        # 1-D metrics with the mirrored outer nodes: widths, centre distances
        self.dx, self.dc, self.fx = [], [], []
        for a in self.nodes:
            x = np.concatenate([[-a[1]], a, [2.0 * a[-1] - a[-2]]])
            xc = np.concatenate([0.5 * (x[1:] + x[:-1]), [x[-1]]])
            m = len(a)
            dc = xc[1:m + 1] - xc[:m]                      # face q between cells q and q+1
            self.dx.append(torch.from_numpy(np.diff(a)).to(DEV))
            self.dc.append(torch.from_numpy(dc).to(DEV))
            self.fx.append(torch.from_numpy((a - xc[:m]) / dc).to(DEV))
        # face masks: 1 where a face is closed (outer boundary)
        self.vol = self._along(self.dx[0], 0) * self._along(self.dx[1], 1) * self._along(self.dx[2], 2)

    @staticmethod
    def _along(v, d):
        return v.reshape([-1 if q == 2 - d else 1 for q in range(3)])

    def shift(self, f, d, s):
        """Interior view of f moved by s along direction d."""
        sl = [slice(1, -2)] * 3
        sl[2 - d] = slice(1 + s, f.shape[2 - d] - 2 + s)
        return f[tuple(sl)]

    def closed(self, d):
        """(lower, upper) masks of the outer faces along direction d."""
        lo = torch.zeros(self.n[d], dtype=F8, device=DEV)
        hi = torch.zeros(self.n[d], dtype=F8, device=DEV)
        lo[0], hi[-1] = 1.0, 1.0
        return self._along(lo, d), self._along(hi, d)

    # -- pressure -------------------------------------------------------
    def extend(self, p, data=None):
        """Fluid values (interior array) to the full layout with solved ghost
        rows (data: the Neumann values at the body)."""
        full = torch.nn.functional.pad(p * self.fluid, (1, 2, 1, 2, 1, 2)).reshape(-1)
        if self.gs.n:
            base = full
            for sweep in range(200):
                g = (self.cN * full[self.stencil]).sum(1)
                if data is not None:
                    g = g + self.cB * data
                new = base.index_add(0, self.gid, g)
                # with a gradient every sweep counts: a fixed number of them
                done = sweep == 59 if new.requires_grad else bool(
                    (new - full).abs().max() <= 1e-17 * new.abs().max())
                full = new
                if done:
                    break
        return full.reshape(self.shape)

    def laplace(self, p, data=None):
        """A p on the fluid cells (closed outer faces)."""
        full = self.extend(p, data)
        c, out = _inner(full), 0.0
        for d in range(3):
            lo, hi = self.closed(d)
            cm = (1.0 - lo) * self._along(1.0 / (self.dc[d][:-1] * self.dx[d]), d)
            cp = (1.0 - hi) * self._along(1.0 / (self.dc[d][1:] * self.dx[d]), d)
            out = out + cm * (self.shift(full, d, -1) - c) + cp * (self.shift(full, d, 1) - c)
        return out * self.fluid

    def box_inverse(self):
        """Pseudo-inverse of the Laplacian of the box without bodies, by
        diagonalising the three 1-D operators."""
        basis, lam = [], []
        for d in range(3):
            w = self.dx[d]
            face = 1.0 / self.dc[d][1:-1]
            m = torch.zeros((self.n[d], self.n[d]), dtype=F8, device=DEV)
            i = torch.arange(self.n[d] - 1, device=DEV)
            off = face / torch.sqrt(w[:-1] * w[1:])
            m[i, i + 1], m[i + 1, i] = off, off
            m[i, i] -= face / w[:-1]
            m[i + 1, i + 1] -= face / w[1:]
            e, q = np.linalg.eigh(m.cpu().numpy())
            lam.append(torch.from_numpy(e).to(DEV))
            basis.append(torch.from_numpy(q).to(DEV))
        root = torch.sqrt(self.vol)
        total = self._along(lam[0], 0) + self._along(lam[1], 1) + self._along(lam[2], 2)
        zero = total.abs() < 1e-9 * total.abs().max() / max(self.n) ** 2
        scale = torch.where(zero, torch.zeros_like(total), 1.0 / torch.where(zero, torch.ones_like(total), total))

        def rotate(f, back):
            for d in range(3):
                q = basis[d] if not back else basis[d].t()
                f = torch.movedim(torch.movedim(f, 2 - d, 2).contiguous() @ q, 2, 2 - d)
            return f

        return lambda f: rotate(rotate(f * root, False) * scale, True) / root

    def bordered(self):
        """(K, to_p): K y = A p + c on fluid cells with p = to_p(y) and c the
        fluid mean of y, which is close to the identity."""
        inv = self.box_inverse()
        vf = self.vol * self.fluid
        total = vf.sum()
        to_p = lambda y: inv(y * self.fluid) * self.fluid  # noqa: E731
        return lambda y: self.laplace(to_p(y)) + self.fluid * ((vf * y).sum() / total), to_p

    def poisson(self, rhs):
        """The zero-mean solution in the full layout."""
        K, to_p = self.bordered()
        with torch.no_grad():
            p = to_p(_gmres(K, _inner(rhs) * self.fluid))
            vf = self.vol * self.fluid
            return self.outer(self.extend(p - (vf * p).sum() / vf.sum()))

    def outer(self, full):
        """Neumann copies into the outer layer, x then y then z."""
        for ax, m in ((2, self.n[0]), (1, self.n[1]), (0, self.n[2])):
            for to, frm in ((0, 1), (m + 1, m)):
                full.select(ax, to)[_planes(full, ax, self.n)] = full.select(ax, frm)[_planes(full, ax, self.n)]
        return full

    def adjoint(self, w):
        """d sum(w p) / d rhs of the zero-mean solve, and its ghost data part."""
        K, to_p = self.bordered()
        vf = self.vol * self.fluid

        def objective(y, data=None):
            p = to_p(y)
            return (self.extend(p - (vf * p).sum() / vf.sum(), data) * w).sum()

        def transpose(v):
            y = torch.zeros_like(v, requires_grad=True)
            return torch.autograd.grad((K(y) * v).sum(), y)[0]

        y = torch.zeros_like(vf, requires_grad=True)
        start = torch.autograd.grad(objective(y), y)[0]
        with torch.enable_grad():
            lam = _gmres(transpose, start) * self.fluid
            data = torch.zeros(self.gs.n, dtype=F8, device=DEV, requires_grad=True)
            still = torch.zeros_like(vf)
            dg, = torch.autograd.grad(objective(still, data) - (self.laplace(still, data) * lam).sum(), data)
        return torch.nn.functional.pad(lam, (1, 2, 1, 2, 1, 2)), dg

    # -- velocity -------------------------------------------------------
    def vel_ghosts(self, vel, vbi):
        """Velocity ghost rows: u_g = 2 u_b - sum c x (in place)."""
        if not self.gs.n:
            return
        flat = [v.reshape(-1) for v in vel]
        for _ in range(300):
            worst = 0.0
            for q in range(3):
                x = torch.where(self.own, vbi[:, q:q + 1], flat[q][self.stencil_raw])
                new = 2.0 * vbi[:, q] - (self.cD * x).sum(1)
                worst = max(worst, float((new - flat[q][self.gid]).abs().max()) / max(float(new.abs().max()), 1e-300))
                flat[q][self.gid] = new
            if worst < 1e-16:
                break

    def correct_vel(self, dt, p, vel, faces, bc, vbi):
        vel, faces = [v.clone() for v in vel], [f.clone() for f in faces]
        pc = _inner(p)
        solid = torch.nn.functional.pad((self.blank & ~self.ghost).to(F8), (1, 2, 1, 2, 1, 2))
        for d in range(3):
            lo, hi = self.closed(d)
            fx, dx, dc = self.fx[d], self._along(self.dx[d], d), self.dc[d]
            fe, fw = self._along(fx[1:], d), self._along(fx[:-1], d)
            pe = (fe * self.shift(p, d, 1) + (1 - fe) * pc) * (1 - hi) + pc * hi
            pw = (fw * pc + (1 - fw) * self.shift(p, d, -1)) * (1 - lo) + pc * lo
            _inner(vel[d]).sub_(dt * (pe - pw) / dx * self.fluid)
            west = (_inner(faces[d]) - dt * (pc - self.shift(p, d, -1)) * self._along(1 / dc[:-1], d)) * (1 - lo)
            west = (west + _inner(bc[d]) * lo) * (1 - torch.maximum(_inner(solid), self.shift(solid, d, -1)))
            last = (1 - _inner(solid)) * _inner(bc[d])
            _inner(faces[d]).copy_(west)
            sl = [slice(1, -2)] * 3
            sl[2 - d] = self.n[d] + 1
            faces[d][tuple(sl)] = last.select(2 - d, self.n[d] - 1)
        self.vel_ghosts(vel, vbi)
        return vel, faces

    def update_pressure(self, p, pprime):
        out = (p + pprime).reshape(-1)
        for _ in range(200):
            if not self.gs.n:
                break
            g = (self.cN * out[self.stencil]).sum(1)
            done = float((g - out[self.gid]).abs().max()) <= 1e-17 * float(g.abs().max())
            out[self.gid] = g
            if done:
                break
        return out.reshape(self.shape)

    def momentum(self, half_dt, dt, nu, vel, nl, faces, vbi):
        """Fixed point of the implicit momentum rows by point Jacobi."""
        vel = [v.clone() for v in vel]
        rows, diag = [], 1.0
        for d in range(3):
            lo, hi = self.closed(d)
            dx, dc, fx = self._along(self.dx[d], d), self.dc[d], self.fx[d]
            am = -0.5 * dt * nu * (self._along(1 / dc[:-1], d) * (1 - lo) + 2.0 * lo / dx) / dx
            ap = -0.5 * dt * nu * (self._along(1 / dc[1:], d) * (1 - hi) + 2.0 * hi / dx) / dx
            vm, vp = _inner(faces[d]), self.shift(faces[d], d, 1)
            fm, fp = self._along(fx[:-1], d), self._along(fx[1:], d)
            diag = diag - (am + ap) + half_dt * (vp * (1 - fp) * (1 - hi) - vm * fm * (1 - lo)) / dx
            rows.append(((am - half_dt * vm * (1 - fm) / dx) * (1 - lo), (ap + half_dt * vp * fp / dx) * (1 - hi)))
        keep = torch.where(self.ghost, torch.ones_like(self.fluid), torch.zeros_like(self.fluid))
        for _ in range(400):
            worst = 0.0
            for q in range(3):
                s = _inner(nl[q]).clone()
                for d in range(3):
                    s -= rows[d][0] * self.shift(vel[q], d, -1) + rows[d][1] * self.shift(vel[q], d, 1)
                new = s / diag * self.fluid + _inner(vel[q]) * keep
                worst = max(worst, float((new - _inner(vel[q])).abs().max()))
                _inner(vel[q]).copy_(new)
            self.vel_ghosts(vel, vbi)
            if worst < 1e-14:
                break
        return vel


def _planes(full, ax, n):
    """The entries 0..n+1 of the two directions a face of axis ax spans."""
    return tuple(slice(0, n[d] + 2) for d in (2, 1, 0) if 2 - d != ax)


def _gmres(K, b, tol=1e-13, steps=80):
    """Full GMRES with re-orthogonalisation on interior arrays."""
    beta = float(b.norm())
    if beta == 0.0:
        return torch.zeros_like(b)
    basis, H = [b / beta], np.zeros((steps + 1, steps))
    for j in range(steps):
        w = K(basis[j])
        for _ in range(2):
            for i, v in enumerate(basis):
                h = float((w * v).sum())
                H[i, j] += h
                w = w - h * v
        H[j + 1, j] = float(w.norm())
        rhs = np.zeros(j + 2)
        rhs[0] = beta
        y, *_ = np.linalg.lstsq(H[:j + 2, :j + 1], rhs, rcond=None)
        left = float(np.linalg.norm(H[:j + 2, :j + 1] @ y - rhs))
        if left <= tol * beta or H[j + 1, j] < 1e-14 * beta:
            break
        basis.append(w / H[j + 1, j])
    return sum(float(c) * v for c, v in zip(y, basis))


def exact(case, seed):
    kind = case["kind"]
    cells = case["nx"] * case["ny"] * case["nz"]
    if (kind == "adjoint" and cells > 1.2e7) or (kind == "momentum" and case["scheme"] == "CN2"):
        return None
    D = _Discrete(case)
    if D.solid_corners and kind in ("poisson", "adjoint", "projection", "moving"):
        return None  # the operator has no exact left null vector: the solve's mean is not defined by it
    s = _inputs(case, seed, D.nodes, D.ib, D.gs)
    if kind == "poisson":
        return D.poisson(s["rhs"])
    if kind == "adjoint":
        return D.adjoint(s["w"])
    if kind == "moving":
        return D.poisson(s["rhs"]), torch.from_numpy(D.ib).to(DEV)
    if kind == "divergence":
        d = _divergence(D.nodes, s["faces"], D.fluid, 1.0 / DT)
        return d, float((_inner(d) * D.vol).sum())
    if kind == "correct_vel":
        return D.correct_vel(DT, s["p"], s["vel"], s["faces"], s["bc"], s["vbi"])
    if kind == "update_pressure":
        return D.update_pressure(s["p"], s["pprime"])
    if kind == "momentum":
        return D.momentum(0.0 if case["scheme"] == "AB" else 0.5 * DT, DT, NU, s["vel"], s["nl"], s["faces"], s["vbi"])
    sol = D.poisson(_divergence(D.nodes, s["faces"], D.fluid, 1.0 / DT))
    vel, faces = D.correct_vel(DT, sol, s["vel"], s["faces"], s["bc"], s["vbi"])
    return sol, vel, faces, D.update_pressure(s["p"], sol)
