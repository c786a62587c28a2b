"""Performance cases of the MHD time step: what a program that uses this package has it do.

A pass is what such a program's loop does between two outputs: a number of RK3 steps from where the
state stands and a download of the whole state; or, for the reverse mode, upload, taped forward
steps and the backward pass that returns the gradient.  Every call goes through ``Solver``,
``Batch`` or ``Rollout``; host arrays are the package's ghost-inclusive float64 arrays.

``exact`` restates the step in plain torch FP64 (PPM / TVD minmod, HLL, upwind constrained
transport, SSP-RK3, ghost fill, CFL step) without this package's kernels, and takes gradients of it
by autograd.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch
import torch.utils.checkpoint

from cumpic_amd import ics
from cumpic_amd.autograd import Rollout, initial_velocity, magnetic_energy
from cumpic_amd.config import CARTESIAN, FP64, MIXED, PPMC, TVDMM, Config, uniform_faces
from cumpic_amd.cumc import Batch, Solver

RECON = {"ppm": PPMC, "tvd": TVDMM}
PRECISION = {"fp64": FP64, "mixed": MIXED}
BOUNDARY = {"periodic": (0,) * 6, "outflow": (1,) * 6}


def listed():
    return [
        # a 1D shock tube between two plots: 800 cells, the smallest grids, bound by latency and launches
        {"name": "riemann1d_800", "kind": "riemann1d", "nx": 800, "steps": 64},
        # a 2D problem on one GPU (the MHD rotor with outflow sides)
        {"name": "rotor2d_400", "kind": "rotor", "nx": 400, "steps": 32},
        # a 2D box of odd, uneven sides with the TVD limiter
        {"name": "box2d_333x190_tvd", "kind": "box", "nx": 333, "ny": 190, "nz": 1, "recon": "tvd",
         "precision": "fp64", "boundary": "periodic", "steps": 32},
        # a small 3D box, as in parameter scans and convergence series
        {"name": "box3d_48", "kind": "box", "nx": 48, "ny": 48, "nz": 48, "recon": "ppm", "precision": "fp64",
         "boundary": "periodic", "steps": 32},
        # a ragged 3D box with outflow sides and the TVD limiter
        {"name": "box3d_101x67x45_tvd", "kind": "box", "nx": 101, "ny": 67, "nz": 45, "recon": "tvd",
         "precision": "fp64", "boundary": "outflow", "steps": 32},
        # an ordinary production box in FP64
        {"name": "box3d_128", "kind": "box", "nx": 128, "ny": 128, "nz": 128, "recon": "ppm", "precision": "fp64",
         "boundary": "periodic", "steps": 64},
        # the largest: the benchmark's 256^3 box in FP64
        {"name": "box3d_256", "kind": "box", "nx": 256, "ny": 256, "nz": 256, "recon": "ppm", "precision": "fp64",
         "boundary": "periodic", "steps": 32},
        # a large box in the mixed form
        {"name": "box3d_192_mixed", "kind": "box", "nx": 192, "ny": 192, "nz": 192, "recon": "ppm",
         "precision": "mixed", "boundary": "periodic", "steps": 64},
        # the accretion torus on a cylindrical grid: curved geometry, sources, floors, inflow clamps
        {"name": "torus_128x64x128", "kind": "torus", "nx": 128, "ny": 64, "nz": 128, "precision": "fp64",
         "steps": 32},
        # many 2D boxes of uneven sizes advanced together (training data, ensembles)
        {"name": "batch48_forward", "kind": "batch", "boxes": 48, "smallest": 64, "largest": 256, "steps": 40},
        # the same in reverse mode: the gradient of an observable with respect to every box's initial state
        {"name": "batch12_adjoint", "kind": "batch_adjoint", "boxes": 12, "smallest": 64, "largest": 192,
         "steps": 12, "every": 4},
        # one 3D box inside a torch program: forward and backward through the autograd function
        {"name": "rollout_40x36x28", "kind": "rollout", "nx": 40, "ny": 36, "nz": 28, "steps": 8, "every": 4},
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["riemann1d", "rotor", "box2d", "box", "box", "box", "torus", "batch", "batch_adjoint", "rollout"])
    if kind == "riemann1d":
        return {"kind": kind, "nx": _log(rng, 200, 4000), "steps": rng.randint(32, 96)}
    if kind == "rotor":
        return {"kind": kind, "nx": _log(rng, 100, 900), "steps": rng.randint(16, 40)}
    if kind == "box2d":
        return {"kind": "box", "nx": _log(rng, 64, 1000), "ny": _log(rng, 64, 1000), "nz": 1,
                "recon": rng.choice(["ppm", "tvd"]), "precision": "fp64",
                "boundary": rng.choice(["periodic", "outflow"]), "steps": rng.randint(16, 40)}
    if kind == "box":
        return {"kind": kind, "nx": _log(rng, 24, 200), "ny": _log(rng, 24, 200), "nz": _log(rng, 24, 200),
                "recon": rng.choice(["ppm", "ppm", "tvd"]), "precision": rng.choice(["fp64", "fp64", "mixed"]),
                "boundary": rng.choice(["periodic", "outflow"]), "steps": rng.randint(24, 64)}
    if kind == "torus":
        return {"kind": kind, "nx": _log(rng, 48, 192), "ny": _log(rng, 16, 96), "nz": _log(rng, 48, 192),
                "precision": rng.choice(["fp64", "mixed"]), "steps": rng.randint(16, 40)}
    if kind == "batch":
        return {"kind": kind, "boxes": rng.randint(8, 48), "smallest": 64, "largest": rng.choice([128, 192, 256]),
                "steps": rng.randint(16, 40)}
    if kind == "batch_adjoint":
        return {"kind": kind, "boxes": rng.randint(4, 12), "smallest": 64, "largest": rng.choice([96, 128, 192]),
                "steps": rng.randint(6, 12), "every": 4}
    return {"kind": kind, "nx": _log(rng, 16, 56), "ny": _log(rng, 16, 56), "nz": _log(rng, 16, 56),
            "steps": rng.randint(6, 12), "every": 4}


# ---------------------------------------------------------------------------------------------
# initial states
# ---------------------------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _box(case, seed):
    """Periodic box of a few random modes: rho about 1, v of rms 0.2, p about 0.5, B = B_z + curl A on
    the staggered faces (divergence-free to round-off)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    cfg = Config(nx=nx, ny=ny, nz=nz, coordinate=CARTESIAN, boundary_flag=BOUNDARY[case["boundary"]],
                 recon=RECON[case["recon"]], cfl=0.3, precision=PRECISION[case["precision"]])
    rng, dev = random.Random(seed), _device()
    co = [torch.arange(n, device=dev, dtype=torch.float64) / n * (2.0 * math.pi) for n in (nz, ny, nx)]

    def field():
        f = torch.zeros((nz, ny, nx), device=dev, dtype=torch.float64)
        for _ in range(6):
            k = [rng.randint(-4, 4) if n > 1 else 0 for n in (nz, ny, nx)]
            if not any(k):
                k[2] = 1
            ph = k[0] * co[0][:, None, None] + k[1] * co[1][None, :, None] + k[2] * co[2][None, None, :]
            f += torch.cos(ph + rng.uniform(0.0, 2.0 * math.pi)) * (rng.gauss(0.0, 1.0) / math.sqrt(sum(q * q for q in k)))
        return f / f.square().mean().sqrt()

    v = [0.2 / math.sqrt(3.0) * field() for _ in range(3)]
    rho, p = torch.exp(0.1 * field()), 0.5 * torch.exp(0.1 * field())
    a = [field() for _ in range(3)]
    dm = lambda q, ax: q - torch.roll(q, 1, ax)  # noqa: E731
    b = [dm(a[2], 1) * ny - dm(a[1], 0) * nz, dm(a[0], 0) * nz - dm(a[2], 2) * nx, dm(a[1], 2) * nx - dm(a[0], 1) * ny]
    s = 0.2 / float(torch.sqrt(sum(q.square().mean() for q in b)))
    b = [q * s for q in b]
    b[2] = b[2] + 1.0
    inner = torch.stack([rho, *v, p, *b], dim=-1)
    for ax, n in enumerate((nz, ny, nx)):
        inner = inner.index_select(ax, (torch.arange(-3, n + 3, device=dev) % n))
    prim = inner.cpu().numpy()
    eps = (inner[..., 4] / inner[..., 0] / (cfg.ggas - 1.0)).cpu().numpy()
    return ics.Problem(cfg, uniform_faces(nx, 0.0, 1.0), uniform_faces(ny, 0.0, 1.0), uniform_faces(nz, 0.0, 1.0),
                       prim, eps)


def _problem(case, seed):
    kind = case["kind"]
    if kind == "riemann1d":
        return ics.riemann_1d(n=case["nx"], seed=seed)
    if kind == "rotor":
        return ics.randomize(ics.riemann_test(ics.MHD_ROTOR, n=case["nx"], cfl=0.4), seed=seed, amp=0.02)
    if kind == "torus":
        pr = ics.torus_cyn(nr=case["nx"], nphi=case["ny"], nzz=case["nz"], seed=seed, cfl=0.3)
        pr.cfg.precision = PRECISION[case["precision"]]
        return pr
    if kind == "rollout":
        return _box({**case, "recon": "ppm", "precision": "fp64", "boundary": "periodic"}, seed)
    return _box(case, seed)


def _batch_sizes(case):
    """Box sizes of a batch: uneven, drawn from the batch sizes of the package within the case's range."""
    sizes = [n for n in ics.BATCH_SIZES if case["smallest"] <= n <= case["largest"]]
    return random.Random(1000 * case["boxes"] + case["largest"]).choices(sizes, k=case["boxes"])


def _batch_problems(case, seed):
    return [ics.spectral_box(n=n, seed=100 * (seed % 1000000) + i, ndim=2) for i, n in enumerate(_batch_sizes(case))]


def _weights(probs, seed):
    """Random weights of the observable J = sum w . B_cell over the interior cells of each box."""
    out = []
    for i, p in enumerate(probs):
        w = np.zeros(p.cfg.shape + (3,))
        c = p.cfg
        inner = (slice(3, 3 + c.nz), slice(3, 3 + c.ny), slice(3, 3 + c.nx))
        w[inner] = np.random.default_rng((seed, i)).standard_normal(w[inner].shape)
        out.append(w)
    return out


# ---------------------------------------------------------------------------------------------
# what is measured
# ---------------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "steps": case["steps"]}
    if kind in ("batch", "batch_adjoint"):
        probs = _batch_problems(case, seed)
        boxes = [Solver.from_problem(p) for p in probs]
        st.update(probs=probs, boxes=boxes, batch=Batch(boxes))
        if kind == "batch":
            for s in boxes:
                s.initial_update()
        else:
            st.update(weights=_weights(probs, seed), every=case["every"])
        return st
    prob = _problem(case, seed)
    if kind == "rollout":
        s = Solver.from_problem(prob)
        v0 = initial_velocity(prob).to(_device()).requires_grad_(True)
        st.update(solver=s, prob=prob, v0=v0, every=case["every"])
        return st
    s = Solver.from_problem(prob)
    s.initial_update()
    st["solver"] = s
    return st


def run(state):
    kind, steps = state["kind"], state["steps"]
    if kind == "batch":
        dts = state["batch"].run(steps, graph_steps=8)
        return {"dts": dts, "prim": [s.download()["prim"] for s in state["boxes"]]}
    if kind == "batch_adjoint":
        for s, p in zip(state["boxes"], state["probs"]):
            s.upload(p.prim, p.eps)
        dts = state["batch"].tape_run(steps, every=state["every"])
        return {"dts": dts, "grad": state["batch"].tape_backward(state["weights"])}
    if kind == "rollout":
        v0 = state["v0"]
        prim, bcell = Rollout.apply(v0, state["solver"], state["prob"], steps, state["every"], None)
        (grad,) = torch.autograd.grad(magnetic_energy(bcell, state["prob"]), v0)
        return {"prim": prim.detach(), "bcell": bcell.detach(), "grad": grad}
    dts, _ = state["solver"].run(steps)
    return {"dts": dts, **state["solver"].download()}


def work(case):
    """State traffic of the RK3 steps (64 FP64 words per zone and step: stage 1 reads one state and
    writes one, stages 2 and 3 read two and write one) and about 6000 operations per zone and step
    (three faces and three stages; half of it per extra dimension in 1D and 2D is not taken off).
    The reverse mode needs the forward step, its derivative's operations (twice those) and the
    state and its adjoint read and written once more."""
    kind = case["kind"]
    if kind in ("batch", "batch_adjoint"):
        zones = sum(p * p for p in _batch_sizes(case))
    else:
        zones = case["nx"] * (case["nx"] if kind == "rotor" else case.get("ny", 1)) * case.get("nz", 1)
    zs = zones * case["steps"]
    f = 3 if kind in ("batch_adjoint", "rollout") else 1
    return {"bytes": 512.0 * f * zs, "flops": 6000.0 * f * zs}


# ---------------------------------------------------------------------------------------------
# the same results in plain torch FP64
# ---------------------------------------------------------------------------------------------
def _sqrt(x):
    pos = x > 0
    return torch.where(pos, torch.sqrt(torch.where(pos, x, torch.ones_like(x))), torch.zeros_like(x))


def _up(a, ax):  # a at index + 1 along axis 0 (x), 1 (y) or 2 (z)
    return torch.roll(a, -1, -1 - ax)


def _dn(a, ax):
    return torch.roll(a, 1, -1 - ax)


class _Exact:
    """Boxes of one shape, stacked along the first axis of every field [nbox, nz+6, ny+6, nx+6]."""

    def __init__(self, probs):
        c = probs[0].cfg
        self.c, self.dev = c, _device()
        self.n = (c.nx, c.ny, c.nz)
        faces = (probs[0].xf, probs[0].yf, probs[0].zf)
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev, dtype=torch.float64)  # noqa: E731
        view = [(1, 1, 1, -1), (1, 1, -1, 1), (1, -1, 1, 1)]
        self.D = [t(f[1:] - f[:-1]).view(view[a]) for a, f in enumerate(faces)]       # widths of cells -2..n+3
        self.C = [t(0.5 * (f[1:] + f[:-1])).view(view[a]) for a, f in enumerate(faces)]
        self.F = [t(f[1:]).view(view[a]) for a, f in enumerate(faces)]                # high face of each cell
        self.Fm = [t(f[:-1]).view(view[a]) for a, f in enumerate(faces)]
        self.cyl, self.torus = c.coordinate == 2, c.model == 1

    def inner(self, lo=1):
        return tuple(slice(lo + 2, n + 3) for n in (self.n[2], self.n[1], self.n[0]))

    # ghost fill, x then y then z (periodic and outflow sides), and the torus inflow clamps; a pass
    # covers the cells [0, n] of the axes that are still to come, and leaves the face field along
    # its own axis alone
    def ghost(self, P, eps, BC):
        P, BC = list(P), list(BC)
        for ax in range(3):
            n = self.n[ax]
            idx = torch.arange(-2, n + 4, device=self.dev)
            lo, hi = self.c.boundary_flag[2 * ax], self.c.boundary_flag[2 * ax + 1]
            src = torch.where(idx < 1, (idx - 1) % n + 1 if lo == 0 else torch.ones_like(idx),
                              torch.where(idx > n, (idx - 1) % n + 1 if hi == 0 else torch.full_like(idx, n), idx)) + 2
            rows = (Ellipsis,) + tuple(slice(2, self.n[a] + 3) if a > ax else slice(None) for a in (2, 1, 0))
            g = lambda a: _put(a, a.index_select(-1 - ax, src)[rows], rows)  # noqa: B023, E731
            for i in range(8):
                if i != 5 + ax:
                    P[i] = g(P[i])
            BC = [g(b) for b in BC]
            eps = g(eps)
        P[4] = P[0] * eps * (self.c.ggas - 1.0)
        if self.torus:
            x = torch.arange(-2, self.n[0] + 4, device=self.dev).view(1, 1, 1, -1)
            z = torch.arange(-2, self.n[2] + 4, device=self.dev).view(1, -1, 1, 1)
            P[1] = torch.where(x < 1, P[1].clamp(max=0.0), torch.where(x > self.n[0], P[1].clamp(min=0.0), P[1]))
            P[3] = torch.where(z < 1, P[3].clamp(max=0.0), torch.where(z > self.n[2], P[3].clamp(min=0.0), P[3]))
        return P, eps, BC

    def edges(self, q, ax):
        D = self.D[ax]
        dp, dm = _up(D, ax), _dn(D, ax)
        qp, qm = _up(q, ax), _dn(q, ax)
        if self.c.recon == TVDMM:
            a, b = 2.0 * (qp - q) / ((D + dp) / D), 2.0 * (q - qm) / ((D + dm) / D)
            s = torch.where(a * b > 0, torch.where(a.abs() < b.abs(), a, b), torch.zeros_like(a))
            return q - 0.5 * s, q + 0.5 * s
        delta = D / (dm + D + dp) * ((2.0 * dm + D) / (dp + D) * (qp - q) + (D + 2.0 * dp) / (dm + D) * (q - qm))
        lim = torch.minimum(delta.abs(), 2.0 * torch.minimum((q - qm).abs(), (qp - q).abs()))
        sl = torch.where((qp - q) * (q - qm) > 0, torch.sign(delta) * lim, torch.zeros_like(q))
        del delta, lim
        dpp = _up(dp, ax)
        z1, z = (dm + D) / (2.0 * D + dp), (dpp + dp) / (2.0 * dp + D)
        w = dm + D + dp + dpp
        vr = q + (D / (D + dp) + 2.0 * dp * D / (dp + D) * (z1 - z) / w) * (qp - q) - D * z1 / w * _up(sl, ax) + dp * z / w * sl
        vl = _dn(vr, ax)
        flat = (vr - q) * (q - vl) <= 0
        lo = torch.where((vr - vl) * (vl - 3.0 * q + 2.0 * vr) < 0, 3.0 * q - 2.0 * vr, vl)
        hi = torch.where((vr - lo) * (3.0 * q - 2.0 * vl - vr) < 0, 3.0 * q - 2.0 * vl, vr)
        return torch.where(flat, q, lo), torch.where(flat, q, hi)

    def side(self, q, bn):
        rho, vn, v1, v2, p, b1, b2 = q
        g = self.c.ggas
        vsq, bsq, vdb = vn * vn + v1 * v1 + v2 * v2, bn * bn + b1 * b1 + b2 * b2, vn * bn + v1 * b1 + v2 * b2
        E = p / (g - 1.0) + 0.5 * rho * vsq + 0.5 * bsq
        u = [rho, rho * vn, rho * v1, rho * v2, E, b1, b2]
        f = [rho * vn, rho * vn * vn + p + 0.5 * bsq - bn * bn, rho * vn * v1 - bn * b1, rho * vn * v2 - bn * b2,
             (E + p + 0.5 * bsq) * vn - bn * vdb, vn * b1 - v1 * bn, vn * b2 - v2 * bn]
        a2, c2 = g * p / rho, bsq / rho
        cf = _sqrt(0.5 * (a2 + c2 + _sqrt((a2 + c2) * (a2 + c2) - 4.0 * a2 * bn * bn / rho)))
        return u, f, cf

    # HLL fluxes on the high faces along ax; order rho, m_x, m_y, m_z, E, and the two transverse B
    def flux(self, P, BC, ax):
        n, t1, t2 = ax, (ax + 1) % 3, (ax + 2) % 3
        vl, vr = [], []
        for q in (P[0], P[1 + n], P[1 + t1], P[1 + t2], P[4], BC[t1], BC[t2]):
            m, p = self.edges(q, ax)
            vl.append(p)
            vr.append(_up(m, ax))
        uL, fL, cL = self.side(vl, P[5 + ax])
        uR, fR, cR = self.side(vr, P[5 + ax])
        sl, sr = _sqrt(vl[0]), _sqrt(vr[0])
        ub, cb = (sl * vl[1] + sr * vr[1]) / (sl + sr), (sl * cL + sr * cR) / (sl + sr)
        a, b = vl[1] - cL, ub - cb
        SL = torch.where(b < a, b, a)
        a, b = vr[1] + cR, ub + cb
        SR = torch.where(b > a, b, a)
        out = []
        for ul, ur, fl, fr in zip(uL, uR, fL, fR):
            h = (SR * fl - SL * fr + SL * SR * (ur - ul)) / (SR - SL)
            out.append(torch.where(SL >= 0, fl, torch.where(SR <= 0, fr, h)))
        r = [None] * 5
        r[0], r[1 + n], r[1 + t1], r[1 + t2], r[4] = out[:5]
        return r, {t1: out[5], t2: out[6]}

    def div(self, f, ax):
        m = _dn(f, ax)
        if self.cyl and ax == 0:
            return (f * self.F[0] - m * self.Fm[0]) / (self.C[0] * self.D[0])
        if self.cyl and ax == 1:
            return (f - m) / (self.C[0] * self.D[1])
        return (f - m) / self.D[ax]

    def sources(self, P, BC):
        rho, vx, vy, vz, p = P[:5]
        bx, by, bz = BC
        z = torch.zeros_like(rho)
        s = [z, z, z, z, z]
        if self.cyl:
            k = float(self.c.geom_source_repeat)
            s[1] = s[1] + k * (p + rho * vy * vy + 0.5 * (bx * bx + by * by + bz * bz) - by * by) / self.C[0]
            s[2] = s[2] - k * (rho * vx * vy - bx * by) / self.C[0]
        if self.torus:
            w = torch.where(rho - self.c.rho_floor >= 0, rho, z)
            R = torch.sqrt(self.C[0] ** 2 + self.C[2] ** 2)
            gx, gz = self.C[0] / R / (R - self.c.r_sh) ** 2, self.C[2] / R / (R - self.c.r_sh) ** 2
            s[1], s[3], s[4] = s[1] - w * gx, s[3] - w * gz, s[4] - w * (vx * gx + vz * gz)
        return s

    def rhs(self, P, BC):
        hydro, ct = self.sources(P, BC), [0.0, 0.0, 0.0]
        E = [0.0, 0.0, 0.0]
        v = P[1:4]
        for ax in range(3):
            f, fb = self.flux(P, BC, ax)
            hydro = [h - self.div(q, ax) for h, q in zip(hydro, f)]
            t1, t2 = (ax + 1) % 3, (ax + 2) % 3
            # E_t2 = -F(B_t1), E_t1 = F(B_t2), averaged to the corner
            E[t2] = E[t2] + 0.25 * (-fb[t1] - _up(fb[t1], t1))
            E[t1] = E[t1] + 0.25 * (fb[t2] + _up(fb[t2], t2))
        for ax in range(3):
            t1, t2 = (ax + 1) % 3, (ax + 2) % 3
            e = v[t2] * BC[t1] - v[t1] * BC[t2]
            s = e + _up(e, t1)
            E[ax] = 2.0 * E[ax] - 0.25 * (s + _up(s, t2))
        R = self.C[0] if self.cyl else 1.0
        d = lambda a, ax: a - _dn(a, ax)  # noqa: E731
        ct[0] = -(d(E[2], 1) / (self.D[1] * (self.F[0] if self.cyl else 1.0)) - d(E[1], 2) / self.D[2])
        ct[1] = -(d(E[0], 2) / self.D[2] - d(E[2], 0) / self.D[0])
        ey = E[1] * self.F[0] - _dn(E[1], 0) * self.Fm[0] if self.cyl else d(E[1], 0)
        ct[2] = -(ey / (R * self.D[0]) - d(E[0], 1) / (R * self.D[1]))
        return hydro, ct

    # the primitive state from the conserved one (face B in U[5:8]), with the floors and the ghosts
    def prims(self, U, P, BC, eps):
        inn = (Ellipsis,) + self.inner()
        put = lambda old, new, s=inn: _put(old, new[s], s)  # noqa: E731
        P = list(P)
        for ax in range(3):
            lo = [1, 1, 1]
            lo[ax] = 0
            s = (Ellipsis,) + tuple(slice(lo[a] + 2, self.n[a] + 3) for a in (2, 1, 0))
            P[5 + ax] = put(P[5 + ax], U[5 + ax], s)
        b = [0.5 * (P[5 + a] + _dn(P[5 + a], a)) for a in range(3)]
        rho = U[0]
        vel = [U[i] / rho for i in (1, 2, 3)]
        e = (U[4] - 0.5 * (b[0] ** 2 + b[1] ** 2 + b[2] ** 2)) / rho - 0.5 * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2)
        rho, e = self.floors(rho, e)
        for i, q in enumerate([rho, *vel]):
            P[i] = put(P[i], q)
        P, eps, BC = self.ghost(P, put(eps, e), [put(o, q) for o, q in zip(BC, b)])
        return P, BC, eps

    def floors(self, rho, e):
        if self.torus:
            return torch.where(rho < self.c.rho_floor, self.c.rho_floor, rho), torch.where(e < self.c.eps_floor, self.c.eps_floor, e)
        return rho, torch.where(e < 0, torch.zeros_like(e), e)

    def cons(self, P, BC, eps):
        rho, vx, vy, vz = P[:4]
        E = rho * (eps + 0.5 * (vx * vx + vy * vy + vz * vz)) + 0.5 * (BC[0] ** 2 + BC[1] ** 2 + BC[2] ** 2)
        return [rho, vx * rho, vy * rho, vz * rho, E, P[5], P[6], P[7]]

    def start(self, prim, eps):
        P = [prim[..., i] for i in range(8)]
        inn = (Ellipsis,) + self.inner()
        z = torch.zeros_like(eps)
        BC = [_put(z, (0.5 * (P[5 + a] + _dn(P[5 + a], a)))[inn], inn) for a in range(3)]
        rho, e = self.floors(P[0], eps)
        P[0], eps = _put(P[0], rho[inn], inn), _put(eps, e[inn], inn)
        P, eps, BC = self.ghost(P, eps, BC)
        return P, BC, eps

    def dt(self, P, BC):
        i = (Ellipsis,) + self.inner()
        rho, v, p, b = P[0][i], [q[i] for q in P[1:4]], P[4][i], [q[i] for q in BC]
        a2, b2 = self.c.ggas * p / rho, (b[0] ** 2 + b[1] ** 2 + b[2] ** 2) / rho
        lam = [v[k].abs() + torch.sqrt(0.5 * (a2 + b2 + torch.sqrt((a2 + b2) ** 2 - 4.0 * a2 * b[k] ** 2 / rho))) for k in range(3)]
        d = torch.minimum(torch.minimum(self.D[0], self.D[1] * (self.C[0] if self.cyl else 1.0)), self.D[2])
        d = d.expand((1,) + tuple(n + 6 for n in self.n[::-1]))[i]
        return (d * self.c.cfl / torch.maximum(torch.maximum(lam[0], lam[1]), lam[2])).amin((1, 2, 3), keepdim=True)

    def step(self, P, BC, eps, dt):
        U0 = self.cons(P, BC, eps)
        U = U0
        for a0, a1 in ((0.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0)):
            h, ct = self.rhs(P, BC)
            U = [a0 * u0 + a1 * (u + dt * r) if a0 else u + dt * r for u0, u, r in zip(U0, U, [*h, *ct])]
            P, BC, eps = self.prims(U, P, BC, eps)
            U = self.cons(P, BC, eps)
        return P, BC, eps

    def go(self, prim, eps, steps, grad=False):
        P, BC, eps = self.start(prim, eps)
        if self.n[2] == 1 and grad:
            # one periodic z cell: its two z faces are one face, and the steps' derivative goes to
            # the high one's entry
            low = (slice(None), slice(2, 3))
            P[7] = _put(P[7], P[7][:, 3:4], low)
        dts = []
        for _ in range(steps):
            with torch.no_grad():
                dt = self.dt(P, BC)
            dts.append(dt.reshape(-1))
            if grad:
                def f(*a, dt=dt):
                    p, b, e = self.step(a[:8], a[8:11], a[11], dt)
                    return (*p, *b, e)
                r = torch.utils.checkpoint.checkpoint(f, *P, *BC, eps, use_reentrant=False)
                P, BC, eps = list(r[:8]), list(r[8:11]), r[11]
            else:
                P, BC, eps = self.step(P, BC, eps, dt)
        return P, BC, eps, torch.stack(dts)

    def inputs(self, probs):
        t = lambda a: torch.as_tensor(np.stack(a), device=self.dev)  # noqa: E731
        return t([p.prim for p in probs]), t([p.eps for p in probs])


def _put(old, new, where):
    out = old.clone()
    out[where] = new
    return out


def exact(case, seed):
    kind, steps = case["kind"], case["steps"]
    if kind in ("batch", "batch_adjoint"):
        return _exact_batch(case, seed)
    prob = _problem(case, seed)
    x = _Exact([prob])
    prim, eps = x.inputs([prob])
    if kind == "rollout":
        c = prob.cfg
        v0 = initial_velocity(prob).to(x.dev).requires_grad_(True)
        inn = (slice(None),) + x.inner() + (slice(1, 4),)
        P, BC, _, _ = x.go(_put(prim, v0[None], inn), eps, steps, grad=True)
        s = (0,) + x.inner()
        p, b = torch.stack([q[s] for q in P], -1), torch.stack([q[s] for q in BC], -1)
        vol = 1.0 / (c.nx * c.ny * c.nz)
        (g,) = torch.autograd.grad(0.5 * (b * b).sum() * vol, v0)
        return {"prim": p.detach(), "bcell": b.detach(), "grad": g}
    with torch.no_grad():
        P, BC, e, dts = x.go(prim, eps, steps)
    return {"dts": dts[:, 0].cpu().numpy(), "prim": torch.stack([q[0] for q in P], -1).cpu().numpy(),
            "eps": e[0].cpu().numpy(), "bcell": torch.stack([q[0] for q in BC], -1).cpu().numpy()}


def _exact_batch(case, seed):
    probs = _batch_problems(case, seed)
    adj = case["kind"] == "batch_adjoint"
    w = _weights(probs, seed) if adj else None
    out, dts = [None] * len(probs), np.zeros((case["steps"], len(probs)))
    for n in sorted({p.cfg.nx for p in probs}):
        at = [i for i, p in enumerate(probs) if p.cfg.nx == n]
        x = _Exact([probs[i] for i in at])
        prim, eps = x.inputs([probs[i] for i in at])
        prim.requires_grad_(adj)
        with torch.set_grad_enabled(adj):
            P, BC, _, d = x.go(prim, eps, case["steps"], grad=adj)
            if adj:
                ww = torch.as_tensor(np.stack([w[i] for i in at]), device=x.dev)
                (res,) = torch.autograd.grad((torch.stack(BC, -1) * ww).sum(), prim)
            else:
                res = torch.stack(P, -1)
        dts[:, at] = d.detach().cpu().numpy()
        for k, i in enumerate(at):
            out[i] = res[k].cpu().numpy()
    return {"dts": dts, "grad" if adj else "prim": out}
