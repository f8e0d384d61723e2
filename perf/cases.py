"""The work that users of this framework have it do, through its public entry points.

Most cases are a run's inner loop as the Fortran driver and the Python API drive it: a simulation in hand (its start-up
steps behind it), then one save interval, that is some time steps with the forces of every step, and at its end the
fields of every level and the body state as a save writes them.  They go from the smallest coupled system to the
largest, with rigid, torsional and flexible bodies, on power-of-two grids and on ones with large prime factors, one
simulation at a time and many together.  Beside them stand the discrete adjoint (forward and reverse sweep together)
and the two forms in which a solver of the user's own takes the Schur operator: its action and its matrix.
"""
import math
import random

import numpy as np
import torch

from ib_parallel_amd import GpuBatch, GpuSim, decks
from ib_parallel_amd.abi import BodySpec, make_params

WARM = 3  # start-up steps before a state counts as in hand: the first step is an Euler step from rest


def listed():
    return [
        # a coupled system on the smallest grid in use: every launch and every wait shows
        dict(name="small_coupled", kind="small", m=32, n=24, levels=2, steps=10),
        # flow past a cylinder with the reference's default restart: GMRES(30), pressure on the save step
        dict(name="cylinder_gmres", kind="cylinder", m=200, n=200, levels=3, steps=20, pressure=True),
        # the same flow held fixed (precomputed solve), on a grid whose transforms have the prime factors 67 and 53
        dict(name="cylinder_fixed", kind="fixed", m=268, n=212, levels=4, steps=40),
        # a hinged plate, coupled to 1e-10
        dict(name="plate", kind="plate", m=400, n=400, levels=4, steps=10),
        # a flexible plate (beam elements) on a smaller uneven grid
        dict(name="beam", kind="beam", m=320, n=240, levels=3, steps=10),
        # airfoil with a hinged flap at full size: the largest single simulation
        dict(name="airfoil_flap", kind="airfoil_flap", m=1024, n=512, levels=5, airfoil=300, flap=100, steps=20),
        # a parameter study: uneven rigid ellipses advanced together
        dict(name="ellipse_batch", kind="ellipses", sims=16, steps=20),
        # three airfoil + flap systems advanced together (a stiffness study)
        dict(name="flap_batch", kind="flap_batch", sims=3, m=640, n=256, levels=3, airfoil=200, flap=60, steps=10),
        # gradients of drag and lift through 20 steps past a fixed cylinder
        dict(name="adjoint_cylinder", kind="adjoint_fixed", m=200, n=200, levels=3, steps=20),
        # gradients through coupled steps of the hinged plate, with its stiffness, pitch and point positions
        dict(name="adjoint_plate", kind="adjoint_plate", m=400, n=400, levels=3, steps=4),
        # one product with the Schur operator, never assembled
        dict(name="schur_product", kind="product", m=1024, n=512, levels=5),
        # the Schur matrix by columns
        dict(name="schur_matrix", kind="matrix", m=400, n=400, levels=4),
    ]


def draw(rng):
    def cells(lo, hi, by=4):
        return by * max(1, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / by))

    kind = rng.choice(["small", "cylinder", "fixed", "fixed", "plate", "beam", "airfoil_flap", "ellipses", "flap_batch",
                       "adjoint_fixed", "adjoint_plate", "product", "matrix"])
    if kind == "small":
        m = cells(24, 96)
        return dict(kind=kind, m=m, n=max(20, 4 * round(0.1875 * m)), levels=rng.randint(1, 3), steps=rng.randint(4, 12))
    if kind == "airfoil_flap":
        return dict(kind=kind, m=cells(640, 1000), n=cells(200, 512), levels=rng.randint(2, 5),
                    airfoil=rng.randint(120, 300), flap=rng.randint(30, 100), steps=rng.randint(6, 16))
    if kind == "ellipses":
        return dict(kind=kind, sims=rng.randint(3, 24), steps=rng.randint(8, 20), study=rng.randint(1, 10 ** 6))
    if kind == "flap_batch":
        return dict(kind=kind, sims=rng.randint(2, 3), m=cells(640, 800), n=cells(200, 320), levels=rng.randint(2, 3),
                    airfoil=rng.randint(120, 240), flap=rng.randint(30, 80), steps=rng.randint(4, 10))
    big = {"product": 1024, "matrix": 400, "adjoint_plate": 400, "plate": 400, "beam": 400}.get(kind, 400)
    m = cells(96, big, 8 if kind == "beam" else 4)
    n = cells(0.6 * m, min(1.1 * m, big))
    c = dict(kind=kind, m=m, n=n, levels=rng.randint(2, 5 if kind == "product" else 4))
    if kind not in ("product", "matrix"):
        c["steps"] = rng.randint(3, 4 if kind == "adjoint_plate" else 16)
    if kind == "cylinder":
        c["pressure"] = rng.random() < 0.5
    return c


# ------------------------------------------------------------------ decks
def _box(c, dt, re, tol, **kw):
    """A domain 4 long around the body, square cells, as the named decks have it."""
    m, n = c["m"], c["n"]
    return make_params(m, n, c["levels"], dt, re, 4.0, 1.0, 2.0 * n / m, fsi_tol=tol, atol=tol, rtol=tol, **kw)


def _circle(c, turn):
    npts = max(24, round(math.pi * c["m"] / 4.0))  # points one cell apart
    t = turn + 2.0 * np.pi * np.arange(npts) / npts
    return BodySpec(0.5 * np.cos(t), 0.5 * np.sin(t), fam=1)


def _deck(c, seed):
    """[(params, bodies), ...]: flow conditions and structural parameters vary with the seed."""
    r = random.Random(1000003 * int(seed) + 17)
    kind, dx = c["kind"], 4.0 / c.get("m", 400)
    re, pitch, stiff, turn = r.uniform(0.9, 1.1), r.uniform(8.0, 12.0), r.uniform(0.8, 1.2), r.uniform(0.01, 0.2)
    if kind == "small":
        p, bodies = decks.tiny_case(m=c["m"], n=c["n"], mgridlev=c["levels"], tol=1e-10, re=50.0 * re, gmres_restart=200,
                                    dt=0.32 / c["m"])
        bodies[1].ktheta *= stiff
        return [(p, bodies)]
    if kind in ("cylinder", "product", "matrix"):
        kw = dict(schur_mode=1) if kind == "product" else {}
        return [(_box(c, 0.2 * dx, 100.0 * re, 1e-8, **kw), [_circle(c, turn)])]
    if kind in ("fixed", "adjoint_fixed"):
        return [(_box(c, 0.2 * dx, 100.0 * re, 1e-10, num_stat=1), [_circle(c, turn)])]
    if kind in ("plate", "adjoint_plate"):
        body = decks.plate_body(c["m"] // 4 + 1, pitch_deg=pitch, k_theta=0.1 * stiff)
        return [(_box(c, 0.1 * dx, 200.0 * re, 1e-10, gmres_restart=250), [body])]
    if kind == "beam":
        body = decks.beam_body(c["m"] // 4 + 1, pitch_deg=pitch, k_b=0.1 * stiff)
        return [(_box(c, 0.1 * dx, 200.0 * re, 1e-10, gmres_restart=250), [body])]
    if kind in ("airfoil_flap", "flap_batch"):
        return [decks.airfoil_flap_case(m=c["m"], n=c["n"], mgridlev=c["levels"], n_airfoil=c["airfoil"], n_flap=c["flap"],
                                        re=1000.0 * re, k_theta=0.05 * stiff * (1.0 + 0.3 * k), flap_deg=pitch)
                for k in range(c.get("sims", 1))]
    if kind == "ellipses":
        cases = decks.ellipse_batch_cases(c["sims"], seed=c.get("study", 20240611))
        for p, _ in cases:  # the sizes are the study's, the flow conditions the seed's
            p.re *= re * r.uniform(0.97, 1.03)
        return cases
    raise ValueError(kind)


def prepare(case, seed):
    kind = case["kind"]
    deck = _deck(case, seed)
    if kind in ("ellipses", "flap_batch"):
        sim = GpuBatch(deck)
    else:
        sim = GpuSim(*deck[0])
    state = {"case": case, "sim": sim}
    if kind == "product":
        g = np.random.default_rng(seed)
        t = np.linspace(0.0, 2.0 * np.pi, sim.nf)
        state["x"] = np.cos(t + g.uniform(0, 6)) + 0.1 * g.standard_normal(sim.nf)  # surface forces
    elif kind != "matrix":
        for _ in range(WARM):
            sim.advance()
    return state


# -------------------------------------------------------------------- run
def run(state):
    c, sim = state["case"], state["sim"]
    kind = c["kind"]
    if kind == "product":
        return {"y": sim.schur_matvec(state["x"])}
    if kind == "matrix":
        return {"S": sim.schur_matrix()}
    if kind == "adjoint_fixed":
        J, dre, dw, gx, gy = sim.adjoint(c["steps"], 1.0, 0.5, position_grad=True)
        return {"J": J, "dRe": dre, "domega": dw, "dx": gx, "dy": gy}
    if kind == "adjoint_plate":
        J, dre, dw, gx, gy, dk, dg = sim.adjoint(c["steps"], 1.0, 0.5, position_grad=True, body_grad=True)
        return {"J": J, "dRe": dre, "domega": dw, "dx": gx, "dy": gy, "dK": dk, "dpitch": dg}
    if kind in ("ellipses", "flap_batch"):
        loads = []
        for _ in range(c["steps"]):
            sim.advance()
            loads.append(np.concatenate([np.concatenate(s.forces()) for s in sim.sims]))
        fields = [s.level(1) for s in sim.sims]
        body = [s.body() for s in sim.sims]
        out = {k: np.concatenate([f[k] for f in fields]) for k in fields[0]}
        out.update({k: np.concatenate([b[k] for b in body]) for k in body[0]})
        out["loads"] = np.array(loads)
        return out
    loads = []
    for _ in range(c["steps"]):
        sim.advance()
        loads.append(np.concatenate(sim.forces()))
    out = {"loads": np.array(loads), "levels": [sim.level(k) for k in range(1, sim.L + 1)], "body": sim.body()}
    if kind == "beam":
        out["beam"] = sim.beam(0)
    if c.get("pressure"):
        out["p"] = sim.pressure()
    return out


# ------------------------------------------------------- work and tolerance
def _fft_flops(m, n):
    return 5.0 * m * n * math.log2(4.0 * m * n)


def _step_work(m, n, L, nf, solves):
    """One time step: the state (vorticity, its history, both fluxes) read and written once, 7 transform pairs a level,
    and `solves` dense solves (0: one product with an inverse in hand)."""
    by = 8.0 * 8 * L * m * n + 8.0 * nf * nf * max(1, solves)
    fl = (7.0 * L + 2.0) * _fft_flops(m, n) + (2.0 / 3.0 * nf ** 3 * solves if solves else 2.0 * nf * nf)
    return by, fl


def work(case):
    kind = case["kind"]
    by = fl = 0.0
    for p, bodies in _deck(case, 1):
        m, n, L, nf = p.m, p.n, p.mgridlev, 2 * sum(b.npts for b in bodies)
        if kind == "product":
            by += 8.0 * 2 * L * m * n + 16.0 * nf
            fl += (2.0 * L + 2.0) * _fft_flops(m, n)
        elif kind == "matrix":
            by += 8.0 * nf * nf + nf * 8.0 * 2 * L * m * n
            fl += nf * (2.0 * L + 2.0) * _fft_flops(m, n)
        else:
            moving = any(b.fam > 1 for b in bodies)
            b1, f1 = _step_work(m, n, L, nf, 0 if p.num_stat else (3 if moving else 1))
            both = 2 if kind.startswith("adjoint") else 1  # the reverse sweep does what the forward one does
            saved = 1 if kind in ("ellipses", "flap_batch") else L
            by += case["steps"] * both * b1 + 8.0 * 5 * saved * m * n
            fl += case["steps"] * both * f1
    return {"bytes": by, "flops": fl}


# About four times what the same run differs by when its sums are taken in another order: the matrix-core form of the
# transforms against the FFT form, the staged GMRES against the cooperative one, over listed and drawn cases, and by what
# fixed bodies' forces differ from exact() (relative error, largest error).  A coupled solve stops at its own tolerance, and the condition of the Schur system (1e8 for the
# flap's closely spaced points) amplifies where it stops into the surface forces.
_TOL = {"small": (4e-11, 1e-10), "cylinder": (5e-5, 1e-4), "fixed": (4e-10, 2e-9), "plate": (2e-9, 4e-9),
        "beam": (2e-10, 6e-10), "airfoil_flap": (3e-5, 1e-3), "ellipses": (2e-10, 2e-9), "flap_batch": (3e-10, 4e-10),
        "adjoint_fixed": (1e-11, 3e-11), "adjoint_plate": (1e-11, 3e-11), "product": (1e-14, 1e-13),
        "matrix": (1e-14, 1e-13)}


def tolerance(case):
    rel, most = _TOL[case["kind"]]
    return {"rel": rel, "max": most}


# ------------------------------------------------------------------ exact
# The same numbers from plain dense algebra in 64 bits: the transforms as products with the sine matrix, the Schur system
# solved directly.  Only the linear operator and the steps past fixed bodies have such a value; a coupled step stops at
# an iterative solver's tolerance.
def _phi(r, dr):
    """The 3-cell smoothed delta function, whose short literals are single precision."""
    s = [float(np.float32(v)) for v in (-.1388888889, .2405626122, -.2405626122, -.3792313933, .1012731481, .6485698427,
                                         .4861111111, -1.143175026, -.1202813061, .8751991178, .3608439183,
                                         -.1548032407, -.2806563809, .1150173611, -.2638888889, 1.214391675,
                                         -2.449273192, .1523563211, 1.843201677)]
    q = np.abs(r) / dr

    def root(v):
        return np.sqrt(np.maximum(v, 0.0))

    def arc(v):
        return np.arcsin(np.clip(v, -1.0, 1.0))

    h = 0.5 * math.sqrt(3.0)
    a, b = arc(h * (2 * q - 1)), root(1 - 12 * q ** 2 + 12 * q)
    d1 = (0.4166666667e-1 * q ** 4 + (s[0] + 0.3472222222e-1 * b) * q ** 3
          + (-0.7121664902e-1 - 0.5208333333e-1 * b + s[1] * a) * q ** 2 + (s[2] * a + s[3] + s[4] * b) * q
          + 0.8018753741e-1 * a - 0.4195601852e-1 * b + s[5])
    a, b = arc(h * (2 * q - 3)), root(-23 + 36 * q - 12 * q ** 2)
    d2 = (-0.0625 * q ** 4 + (s[6] - 0.1736111111e-1 * b) * q ** 3 + (s[7] + 0.078125 * b + s[8] * a) * q ** 2
          + (s[9] + s[10] * a + s[11] * b) * q + s[12] * a + 0.822848104e-2 + s[13] * b)
    a, b = arc(h * (2 * q - 5)), root(-71 - 12 * q ** 2 + 60 * q)
    d3 = (0.2083333333e-1 * q ** 4 + (0.3472222222e-2 * b + s[14]) * q ** 3
          + (s[15] - 0.2604166667e-1 * b + 0.2405626122e-1 * a) * q ** 2 + (s[8] * a + s[16] + 0.7262731481e-1 * b) * q
          + s[17] * a + s[18] - 0.7306134259e-1 * b)
    return np.where(q <= 1, d1, np.where(q <= 2, d2, np.where(q <= 3, d3, 0.0))) / dr


class _Plain:
    """The operators of one simulation with rigid bodies; node arrays are (..., n - 1, m - 1)."""

    def __init__(self, p, bodies):
        self.p, self.m, self.n, self.L = p, p.m, p.n, p.mgridlev
        m, n = self.m, self.n
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.delta = p.len / m

        def sines(M):
            k = torch.arange(1, M, dtype=torch.int64, device=self.dev)
            return 2.0 * torch.sin(math.pi / M * ((k[:, None] * k) % (2 * M)).double())

        self.sx, self.sy = sines(m), sines(n)
        i = torch.arange(1, m, device=self.dev).double()
        j = torch.arange(1, n, device=self.dev).double()
        self.lam = -2.0 * (torch.cos(math.pi / m * i) + torch.cos(math.pi / n * j)[:, None] - 2.0)
        self.norm = 4.0 * m * n
        comp = np.concatenate([np.repeat([0, 1], b.npts) for b in bodies])
        xb = np.concatenate([np.tile(b.x, 2) for b in bodies])
        yb = np.concatenate([np.tile(b.y, 2) for b in bodies])
        self.nf, d = comp.size, self.delta
        ix, iy = ((xb + p.offsetx) / d).astype(int) + 1, ((yb + p.offsety) / d).astype(int) + 1
        o = np.arange(-3, 4)
        half = np.where(comp == 0, 0.0, 0.5 * d)
        wx = _phi(d * (ix[:, None] - 1 + o) - p.offsetx + half[:, None] - xb[:, None], d)
        wy = _phi(d * (iy[:, None] - 1 + o) - p.offsety + (0.5 * d - half)[:, None] - yb[:, None], d)
        ii, jj = ix[:, None, None] - 1 + o, (iy[:, None] - 1 + o)[:, :, None]
        wide = np.where(comp == 0, m + 1, m)[:, None, None]
        key = np.where(comp == 0, 0, (m + 1) * n)[:, None, None] + wide * jj + ii
        self.E = torch.zeros((self.nf, (m + 1) * n + m * (n + 1)), dtype=torch.float64, device=self.dev)
        self.E.scatter_(1, torch.from_numpy(key.reshape(self.nf, 49)).to(self.dev),
                        torch.from_numpy((d * d * wy[:, :, None] * wx[:, None, :]).reshape(self.nf, 49)).to(self.dev))

    def dst(self, a):
        return torch.matmul(self.sy, torch.matmul(a, self.sx))

    def del22(self, k):
        return self.delta ** 2 * 4.0 ** k

    def lam1i(self, k):
        return 1.0 / (1.0 + 0.5 * self.p.dt * self.lam / self.del22(k) / self.p.re)

    def ainv(self, a):
        return self.dst(self.lam1i(0) * self.dst(a) / self.norm)

    def split(self, q):
        cut = (self.m + 1) * self.n
        return (q[..., :cut].reshape(*q.shape[:-1], self.n, self.m + 1),
                q[..., cut:].reshape(*q.shape[:-1], self.n + 1, self.m))

    def rot(self, q):
        qx, qy = self.split(q)
        return qy[..., 1:-1, 1:] - qy[..., 1:-1, :-1] - qx[..., 1:, 1:-1] + qx[..., :-1, 1:-1]

    def edge(self, c, fac):
        """Values on the outline of the next finer level: (left, right, bottom, top)."""
        m, n = self.m, self.n
        i0, i1, j0, j1 = m // 4 - 1, 3 * m // 4 - 1, n // 4 - 1, 3 * n // 4 - 1

        def two(v):
            out = v.new_zeros(v.shape[:-1] + (2 * v.shape[-1] - 1,))
            out[..., ::2] = v
            out[..., 1::2] = 0.5 * (v[..., 1:] + v[..., :-1])
            return fac * out
        return (two(c[..., j0:j1 + 1, i0]), two(c[..., j0:j1 + 1, i1]), two(c[..., j0, i0:i1 + 1]),
                two(c[..., j1, i0:i1 + 1]))

    def ring(self, a, bc, fac=1.0):
        if bc is None:
            return a
        a = a.clone()
        a[..., :, 0] += fac * bc[0][..., 1:-1]
        a[..., :, -1] += fac * bc[1][..., 1:-1]
        a[..., 0, :] += fac * bc[2][..., 1:-1]
        a[..., -1, :] += fac * bc[3][..., 1:-1]
        return a

    def ext(self, a, bc):
        e = a.new_zeros(a.shape[:-2] + (self.n + 1, self.m + 1))
        e[..., 1:-1, 1:-1] = a
        if bc is not None:
            e[..., :, 0], e[..., :, -1], e[..., 0, :], e[..., -1, :] = bc
        return e

    def vort2flux(self, w):
        m, n = self.m, self.n
        w, s, q, bc = list(w), [None] * self.L, [None] * self.L, None
        for k in range(1, self.L):
            f = w[k - 1]
            c = f[..., 1:-1, 1:-1] + 0.5 * (f[..., 1:-1, 2:] + f[..., 2:, 1:-1] + f[..., 1:-1, :-2] + f[..., :-2, 1:-1]) \
                + 0.25 * (f[..., 2:, 2:] + f[..., :-2, 2:] + f[..., :-2, :-2] + f[..., 2:, :-2])
            w[k] = w[k].clone()
            w[k][..., n // 4:n // 4 + n // 2 - 1, m // 4:m // 4 + m // 2 - 1] = c[..., ::2, ::2]
        for k in range(self.L - 1, -1, -1):
            s[k] = self.dst(self.dst(self.ring(w[k], bc)) / self.lam / self.norm)
            e = self.ext(s[k], bc)
            q[k] = torch.cat([(e[..., 1:, :] - e[..., :-1, :]).flatten(-2), (e[..., :, :-1] - e[..., :, 1:]).flatten(-2)],
                             -1)
            bc = self.edge(s[k], 1.0)
        return w, s, q

    def product(self, x):
        """S x for the rows x (batch, nf)."""
        v = self.ainv(self.rot(x @ self.E))
        w = [v] + [torch.zeros_like(v) for _ in range(self.L - 1)]
        return self.vort2flux(w)[2][0] @ self.E.T

    def matrix(self):
        eye = torch.eye(self.nf, dtype=torch.float64, device=self.dev)
        return torch.cat([self.product(eye[a:a + 16]) for a in range(0, self.nf, 16)]).T

    def nonlinear(self, w, bc, q, k):
        e = self.ext(w, bc)
        qx, qy = self.split(q)
        u = torch.nn.functional.pad(qx + self.delta * 2.0 ** k, (0, 0, 1, 1))
        v = torch.nn.functional.pad(qy, (1, 1))
        ue, ve = 0.5 * (u[1:] + u[:-1]) * e, 0.5 * (v[:, 1:] + v[:, :-1]) * e
        nx, ny = 0.5 * (ve[1:] + ve[:-1]), -0.5 * (ue[:, 1:] + ue[:, :-1])
        return ny[1:-1, 1:] - ny[1:-1, :-1] - nx[1:, 1:-1] + nx[:-1, 1:-1]

    def steps(self, count):
        """`count` steps from rest past bodies held fixed; yields (omega, s, q, rhs, f) after each."""
        p, L = self.p, self.L
        A = torch.triu(self.matrix())
        A = A + torch.triu(A, 1).T
        lu = torch.linalg.lu_factor(A)
        q0 = torch.cat([torch.full(((self.m + 1) * self.n,), self.delta), torch.zeros(self.m * (self.n + 1))])
        q0 = q0.double().to(self.dev)
        q0[:(self.m + 1) * self.n] = self.delta
        w = [torch.zeros((self.n - 1, self.m - 1), dtype=torch.float64, device=self.dev) for _ in range(L)]
        q = [torch.zeros_like(q0) for _ in range(L)]
        old = None
        for _ in range(count):
            last = [self.edge(w[k + 1], 0.25) if k < L - 1 else None for k in range(L)]
            rhs = [self.nonlinear(w[k], last[k], q[k], k) for k in range(L)]
            old = old or rhs
            for k in range(L - 1, -1, -1):
                d2 = self.del22(k)
                r = 1.5 * p.dt / d2 / self.norm * rhs[k] - 0.5 * p.dt / d2 / self.norm * old[k]
                vfac = 0.5 * p.dt / p.re / d2 / self.norm
                r = self.ring(r, last[k], vfac)
                if k < L - 1:
                    r = self.ring(r, self.edge(w[k + 1], 0.25), vfac)
                lam1 = (1.0 - 0.5 * p.dt * self.lam / d2 / p.re) / self.norm
                w[k] = self.dst(self.lam1i(k) * (self.dst(r) + lam1 * self.dst(w[k])))
            old = rhs
            w, s, q = self.vort2flux(w)
            f = torch.linalg.lu_solve(*lu, (self.E @ (q[0] + q0))[:, None])[:, 0]
            w[0] = w[0] - self.ainv(self.rot(f @ self.E))
            w, s, q = self.vort2flux(w)
            yield w, s, q, rhs, f

    def spread_mean(self, f):
        den = self.E.sum(0)
        return self.E @ torch.where(den > 1e-10, (f @ self.E) / torch.where(den > 1e-10, den, torch.ones_like(den)), 0.0)


def _level(S, w, s, q, rhs, k):
    qx, qy = S.split(q[k])
    return {"omega": w[k].flatten(), "s": s[k].flatten(), "qx": qx.flatten(), "qy": qy.flatten(), "rhs_old": rhs[k].flatten()}


def _loads(S, bodies, f):
    out, at = [[], []], 0
    for b in bodies:
        for c in (0, 1):
            out[c].append(2.0 * S.delta * f[at:at + b.npts].sum() / S.p.dt)
            at += b.npts
    return torch.stack(out[0] + out[1])


def _body(S, bodies, f):
    none = torch.zeros(0)
    return {"f": f, "f_rdst": S.spread_mean(f), "xb": torch.from_numpy(np.concatenate([np.tile(b.x, 2) for b in bodies])),
            "yb": torch.from_numpy(np.concatenate([np.tile(b.y, 2) for b in bodies])),
            "theta": none, "thetad": none, "thetadd": none}


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("product", "matrix", "fixed", "ellipses"):
        return None
    got = []
    for p, bodies in _deck(case, seed):
        S = _Plain(p, bodies)
        if kind == "product":
            g = np.random.default_rng(seed)
            t = np.linspace(0.0, 2.0 * np.pi, S.nf)
            x = np.cos(t + g.uniform(0, 6)) + 0.1 * g.standard_normal(S.nf)
            return {"y": S.product(torch.from_numpy(x).to(S.dev)[None])[0]}
        if kind == "matrix":
            return {"S": S.matrix()}
        loads = []
        for i, (w, s, q, rhs, f) in enumerate(S.steps(WARM + case["steps"])):
            if i >= WARM:
                loads.append(_loads(S, bodies, f))
        saved = 1 if kind == "ellipses" else S.L
        got.append((torch.stack(loads), [_level(S, w, s, q, rhs, k) for k in range(saved)], _body(S, bodies, f)))
    if kind == "fixed":
        return {"loads": got[0][0], "levels": got[0][1], "body": got[0][2]}
    out = {k: torch.cat([g[1][0][k] for g in got]) for k in got[0][1][0]}
    out.update({k: torch.cat([g[2][k].cpu() for g in got]) for k in got[0][2]})
    out["loads"] = torch.cat([g[0] for g in got], 1)
    return out
