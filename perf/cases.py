"""Performance cases of falm_amd: what a program built on it spends its time in.

A program uses the framework in two ways.  It marches a simulation on the
device-resident step driver (falm_amd.runtime.Case) and takes a snapshot now
and then, or it writes its own main loop from the single operations of the C
ABI, as the reference's applications do through FalmCFD / FalmEq / FalmMV /
AlmHandler.  The cases cover both, forward and backward, in double, float and
mixed precision, on uniform and stretched meshes, from the smallest domains of
the tests and applications to the two-rotor segment.

A case is a dict of plain values with a "kind":

  predict   pseudo-velocity, face flux and Poisson right-hand side
  correct   boundary fills, projection, eddy viscosity, divergence and its
            norm, running time average: the rest of a step after the solve
  poisson   one pressure solve from the previous step's pressure
  rotor     actuator-line forces projected onto the grid
  smooth    a program's own iteration from sweeps, residual, product and dots
  backward  the vector-Jacobian products of a step's stages, in reverse order
  tunnel    the step driver on a wind-tunnel channel with rotors, and a snapshot
  cavity    the step driver on a lid-driven cavity, and a snapshot
  gradient  rotor power and its gradient through the window adjoint

run() makes the calls as such a program makes them.  exact() restates the
same algorithms in plain torch in 64 bits.
"""
import ctypes as C
import math

import numpy as np
import torch

from falm_amd import _abi as abi
from falm_amd import cases as setups
from falm_amd import runtime as rt

F64, F32 = torch.float64, torch.float32
SCHEMES = {"Upwind1": abi.ADV_UPWIND1, "Upwind3": abi.ADV_UPWIND3, "QUICK": abi.ADV_QUICK,
           "UTOPIA": abi.ADV_UTOPIA, "KK": abi.ADV_KK}
GC = 2


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the momentum half of a step of the 512 x 128 x 128 wind tunnel,
        # written as the applications write it, in the reference's precision
        dict(name="predict-512-f64", kind="predict", nx=512, ny=128, nz=128, prec="f64", scheme="Upwind3",
             stretch=0.0),
        # an odd-sized, stretched mesh in float with another scheme
        dict(name="predict-odd-f32", kind="predict", nx=133, ny=67, nz=45, prec="f32", scheme="QUICK", stretch=0.15),
        # the half after the solve, at the wind tunnel's size
        dict(name="correct-512-f64", kind="correct", nx=512, ny=128, nz=128, prec="f64", walls=False, stretch=0.0),
        # the pressure solve of the wind tunnel in mixed precision at the
        # tolerance the benchmark runs at (one SOR pass as preconditioner)
        dict(name="poisson-512-mixed", kind="poisson", nx=512, ny=128, nz=128, solver="PBiCGStab", mixed=True,
             outlet=True, declared=True, pc_maxit=1, pc_relax=1.0, tol=1.5e-8, stretch=0.0),
        # the cavity LES's solve in double (two passes, over-relaxed)
        dict(name="poisson-128-f64", kind="poisson", nx=128, ny=128, nz=128, solver="PBiCGStab", mixed=False,
             outlet=False, declared=True, pc_maxit=2, pc_relax=1.5, tol=1e-8, stretch=0.0),
        # two rotors' forces on a wide channel, every cell written
        dict(name="rotor-384-f64", kind="rotor", nx=384, ny=128, nz=128, prec="f64", rotors=2, cells_per_d=24,
             motion=True),
        # a program's own relaxation over the seven stored columns, at the
        # size of the two-rotor segment: the largest fields
        dict(name="smooth-1024-f64", kind="smooth", nx=1024, ny=256, nz=256, prec="f64", sweep="sor", stretch=0.0),
        # the stages' vector-Jacobian products at the adjoint report's size
        dict(name="backward-256", kind="backward", nx=256, ny=96, nz=96, scheme="Upwind3", stretch=0.0),
        # the flagship run: the mixed step driver with a rotor, 100 steps
        # between snapshots of a run that goes on
        dict(name="tunnel-512-mixed", kind="tunnel", nx=512, ny=128, nz=128, mixed=True, rotors=1, cells_per_d=32,
             tol=1.5e-8, pc_maxit=1, spin=20, steps=100),
        # a coarse channel as the tests and set-up runs use it, in double,
        # restarted: short kernels, where launches and waits count
        dict(name="tunnel-64-f64", kind="tunnel", nx=64, ny=33, nz=30, mixed=False, rotors=1, cells_per_d=12,
             tol=1e-6, pc_maxit=1, spin=60, steps=50),
        # the 2-D lid-driven cavity with its red-black SOR solver, restarted:
        # the smallest kernels and the most of them
        dict(name="cavity2d-128", kind="cavity", nx=128, ny=128, nz=1, mixed=False, tol=1e-8, spin=25, steps=5),
        # rotor power and its gradient over a short window
        dict(name="gradient-96", kind="gradient", nx=96, ny=48, nz=48, rotors=1, cells_per_d=16, tol=1e-12, spin=20,
             steps=4, ckpt=2),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, cells, lo=12, hi=640):
    """Interior sizes, spread over their logarithms, of at most `cells` cells."""
    while True:
        n = (_logint(rng, 2 * lo, hi), _logint(rng, lo, hi // 3), _logint(rng, lo, hi // 3))
        if n[0] * n[1] * n[2] <= cells:
            return dict(nx=n[0], ny=n[1], nz=n[2])


def draw(rng):
    kind = rng.choice(["predict", "predict", "correct", "correct", "poisson", "poisson", "poisson", "rotor", "smooth",
                       "smooth", "backward", "backward", "tunnel", "tunnel", "tunnel", "cavity", "cavity",
                       "gradient"])
    stretch = rng.choice([0.0, 0.0, round(rng.uniform(0.02, 0.25), 3)])
    prec = rng.choice(["f64", "f64", "f32"])
    if kind == "predict":
        return dict(kind=kind, **_box(rng, 8_400_000), prec=prec,
                    scheme=rng.choice(["Upwind3", "Upwind3", "Upwind1", "QUICK", "UTOPIA", "KK"]), stretch=stretch)
    if kind == "correct":
        return dict(kind=kind, **_box(rng, 8_400_000), prec=prec, walls=rng.random() < 0.4, stretch=stretch)
    if kind == "poisson":
        n = _box(rng, 8_400_000)
        cells = n["nx"] * n["ny"] * n["nz"]
        return dict(kind=kind, **n, solver="PBiCGStab", mixed=rng.random() < 0.5, outlet=rng.random() < 0.6,
                    declared=rng.random() < 0.85, pc_maxit=rng.choice([1, 1, 2, 3]),
                    pc_relax=rng.choice([1.0, 1.2, 1.5]), tol=rng.choice([1e-4, 1e-5]) / math.sqrt(cells),
                    stretch=min(stretch, 0.1))
    if kind == "rotor":
        n = _box(rng, 8_400_000, lo=36)
        return dict(kind=kind, **n, prec=prec, rotors=rng.choice([1, 2]), motion=rng.random() < 0.5,
                    cells_per_d=max(8, min(n["ny"], n["nz"]) // 3))
    if kind == "smooth":
        return dict(kind=kind, **_box(rng, 16_800_000, hi=1100), prec=prec, sweep=rng.choice(["sor", "sor", "jacobi"]),
                    stretch=stretch)
    if kind == "backward":
        return dict(kind=kind, **_box(rng, 2_400_000), scheme=rng.choice(["Upwind3", "UTOPIA", "KK"]), stretch=stretch)
    if kind == "tunnel":
        n = _box(rng, 6_000_000, lo=24)
        cells = n["nx"] * n["ny"] * n["nz"]
        return dict(kind=kind, **n, mixed=rng.random() < 0.6, rotors=rng.choice([0, 1, 1, 2]),
                    cells_per_d=max(8, min(n["ny"], n["nz"]) // 3), tol=rng.choice([1e-3, 2.5e-4]) / math.sqrt(cells),
                    pc_maxit=rng.choice([1, 1, 1, 2]), spin=20, steps=max(20, min(60, 200_000_000 // cells)))
    if kind == "cavity":
        if rng.random() < 0.5:
            m = _logint(rng, 32, 160)
            return dict(kind=kind, nx=m, ny=m, nz=1, mixed=False, tol=rng.choice([1e-7, 1e-8]), spin=25,
                        steps=rng.choice([3, 6]))
        m = _logint(rng, 24, 128)
        mixed = rng.random() < 0.5
        tol = (1e-4 if mixed else rng.choice([1e-3, 2e-4])) / m ** 1.5
        return dict(kind=kind, nx=m, ny=m, nz=m, mixed=mixed, tol=tol, spin=25, steps=20)
    m = _logint(rng, 28, 48)
    return dict(kind="gradient", nx=2 * m + rng.choice([0, 1]), ny=m, nz=m + rng.choice([0, 3]),
                rotors=rng.choice([1, 2]), cells_per_d=max(8, m // 3), tol=1e-12, spin=20, steps=rng.choice([3, 4]),
                ckpt=2)


def _n(case):
    return case["nx"], case["ny"], case["nz"]


def _cells(case):
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    """Each input of a pass read once, each output written once; a driver
    pass reads and writes the flow's state once per step."""
    N, kind = _cells(case), case["kind"]
    T = 4.0 if case.get("prec") == "f32" else 8.0
    if kind == "predict":  # un, u, uu, nut, kx, g, ja, ff -> ua, uu, rhs
        return dict(bytes=28.0 * T * N, flops=420.0 * N)
    if kind == "correct":  # ua, uua, p, kx, g, ja, means -> u, uu, nut, div, means
        return dict(bytes=30.0 * T * N, flops=110.0 * N)
    if kind == "poisson":  # b, x0 (and seven columns unless declared) -> x
        return dict(bytes=8.0 * N * (3.0 if case["declared"] and not case["stretch"] else 10.0), flops=400.0 * N)
    if kind == "rotor":  # ff written (the velocity is read at the points only)
        return dict(bytes=3.0 * T * N, flops=6.0 * N)
    if kind == "smooth":  # a, x, b -> x, r, A r
        return dict(bytes=12.0 * T * N, flops=70.0 * N)
    if kind == "backward":  # u, uu, nut, kx, g, ja, ub, uub, rhsb -> unb, uunb, uab, uusb, pb, nutb, ffb, usb
        return dict(bytes=(21.0 + 20.0) * 8.0 * N, flops=900.0 * N)
    S = 4.0 if case.get("mixed") else 8.0
    per_step = N * (2.0 * (7.0 * S + 8.0))  # u, uu, nut and the pressure
    if kind in ("tunnel", "cavity"):
        return dict(bytes=case["steps"] * per_step, flops=case["steps"] * 900.0 * N)
    return dict(bytes=3.0 * case["steps"] * per_step, flops=case["steps"] * 4000.0 * N)


def tolerance(case):
    """Single operations differ by rounding only (about 2e-15 in double and
    3e-6 in float at the divergence, the most cancelled result, against 64
    bits).  A solve that stops at a tolerance may stop an iteration earlier or
    later when a dot product rounds differently, and then moves by what the
    tolerance leaves open; in the drivers that happens in some of the steps."""
    kind = case["kind"]
    if kind in ("predict", "correct", "rotor", "smooth", "backward"):
        return {"rel": 1e-5} if case.get("prec") == "f32" else {"rel": 1e-13}
    if kind == "poisson":
        return {"rel": 1e-3} if case["mixed"] else {"rel": 1e-6}
    if kind == "tunnel":
        return {"rel": 1e-3} if case["mixed"] else {"rel": 1e-4}
    if kind == "cavity":
        return {"rel": 2e-2} if case["mixed"] else {"rel": 1e-9} if case["nz"] == 1 else {"rel": 1e-4}
    return {"rel": 1e-5}


# ---------------------------------------------------- meshes and fields
def _pad(n):
    return n[0] + 2 * GC, n[1] + 2 * GC, n[2] + 2 * GC


class _Mesh:
    """Cell centres and widths of the padded cells, the metric fields the
    single operations take (kx, g, ja, xyz), all in 64 bits, x fastest."""

    def __init__(self, n, h, stretch=0.0, fields=True):
        self.n, self.c, self.w = n, [], []
        for m in range(3):
            i = torch.arange(n[m] + 2 * GC, dtype=F64, device="cuda")
            w = h * (1.0 + stretch * torch.sin(2.0 * math.pi * (i - GC + 0.5) / n[m]))
            self.w.append(w)
            self.c.append(torch.cumsum(w, 0) - 0.5 * w - w[:GC].sum())
        if fields:
            hx, hy, hz = self.w[0][None, None, :], self.w[1][None, :, None], self.w[2][:, None, None]
            self.ja = (hx * hy * hz).contiguous()
            ones = torch.ones_like(self.ja)
            self.kx = torch.stack([ones / hx, ones / hy, ones / hz])
            self.g = self.ja * self.kx * self.kx

    @property
    def xyz(self):
        ones = torch.ones_like(self.ja)
        return torch.stack([ones * self.c[0][None, None, :], ones * self.c[1][None, :, None],
                            ones * self.c[2][:, None, None]])


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 13)


def _field(n, ncol, gen, base=0.0, amp=1.0, noise=0.05):
    """Large eddies of a seeded shape and phase plus fine-grained noise."""
    px, py, pz = _pad(n)
    x, y, z = (torch.linspace(0, 1, m, dtype=F64, device="cuda") for m in (px, py, pz))
    out = torch.empty((ncol, pz, py, px), dtype=F64, device="cuda")
    for c in range(ncol):
        a = (0.5 + 2.0 * torch.rand(6, generator=gen, dtype=F64, device="cuda")).tolist()
        out[c] = base + amp * (torch.sin(3.1 * a[0] * x + a[3])[None, None, :] *
                               torch.cos(2.3 * a[1] * y + a[4])[None, :, None] *
                               torch.sin(1.7 * a[2] * z + a[5])[:, None, None])
        if noise:
            out[c] += noise * amp * torch.randn((pz, py, px), generator=gen, dtype=F64, device="cuda")
    return out


def _I(a, di=0, dj=0, dk=0):
    """The interior of a field, shifted."""
    nz, ny, nx = a.shape[-3:]
    return a[..., GC + dk:nz - GC + dk, GC + dj:ny - GC + dj, GC + di:nx - GC + di]


def _Fb(a, di=0, dj=0, dk=0):
    """The face region of a field (the interior and the layer below it), shifted."""
    nz, ny, nx = a.shape[-3:]
    return a[..., GC - 1 + dk:nz - GC + dk, GC - 1 + dj:ny - GC + dj, GC - 1 + di:nx - GC + di]


E = ((1, 0, 0), (0, 1, 0), (0, 0, 1))


def _neg(e):
    return tuple(-v for v in e)


def _poisson_matrix(mesh, outlet, flat=False):
    """The applications' seven columns [c,w,e,s,n,b,t] divided by max |c|, and that maximum."""
    a = torch.zeros((7,) + tuple(mesh.ja.shape), dtype=F64, device="cuda")
    for d in range(2 if flat else 3):
        g = mesh.g[d]
        lo, hi = [slice(None)] * 3, [slice(None)] * 3
        lo[2 - d], hi[2 - d] = slice(0, 1), slice(-1, None)
        for sgn, colm in ((1, 2 + 2 * d), (-1, 1 + 2 * d)):
            e = E[d] if sgn > 0 else _neg(E[d])
            coef = 0.5 * (_I(g) + _I(g, *e)) / _I(mesh.ja)
            if sgn < 0:
                coef[tuple(lo)] = 0.0
            elif not (outlet and d == 0):
                coef[tuple(hi)] = 0.0
            _I(a[colm])[...] = coef
            _I(a[0])[...] -= coef
    md = float(a[0].abs().max())
    return a / md, md


# ------------------------------------------- the algorithms in 64 bits
def _pseudo_u(scheme, ReI, dt, un, u, uu, nut, kx, g, ja, ff):
    """ua on the interior cells."""
    J = _I(ja)
    out = []
    for d in range(3):
        q = u[d]
        adv = torch.zeros_like(J)
        vis = torch.zeros_like(J)
        qc = _I(q)
        for e in range(3):
            ep, em = E[e], _neg(E[e])
            p1, m1 = _I(q, *ep), _I(q, *em)
            JP, JM = _I(uu[e]), _I(uu[e], *em)
            Ua = (_I(u[e]) * _I(kx[e])).abs()
            if scheme == "Upwind1":
                fl = 0.5 * (JP * (p1 + qc) - JP.abs() * (p1 - qc)) - 0.5 * (JM * (qc + m1) - JM.abs() * (qc - m1))
                adv = adv + fl / J
            else:
                p2, m2 = _I(q, *(2 * v for v in ep)), _I(q, *(2 * v for v in em))
                if scheme == "QUICK":
                    t = JP * (-p2 + 9 * p1 + 9 * qc - m1) + JP.abs() * (p2 - 3 * p1 + 3 * qc - m1) \
                        - JM * (-p1 + 9 * qc + 9 * m1 - m2) - JM.abs() * (p1 - 3 * qc + 3 * m1 - m2)
                    adv = adv + t / (16.0 * J)
                else:
                    al = {"Upwind3": 1 / 24, "UTOPIA": 1 / 12, "KK": 1 / 4}[scheme]
                    L = JP * (-p2 + 27 * p1 - 27 * qc + m1) / 24
                    R = JM * (-p1 + 27 * qc - 27 * m1 + m2) / 24
                    adv = adv + 0.5 * (L + R) / J + Ua * (p2 - 4 * p1 + 6 * qc - 4 * m1 + m2) * al
            gc, gp, gm = _I(g[e]), _I(g[e], *ep), _I(g[e], *em)
            nc, npl, nm = _I(nut), _I(nut, *ep), _I(nut, *em)
            vis = vis + ((gc + gp) * (ReI + 0.5 * (nc + npl)) * (p1 - qc)
                         - (gc + gm) * (ReI + 0.5 * (nc + nm)) * (qc - m1)) / (2.0 * J)
        out.append(_I(un[d]) + dt * (-adv + vis + _I(ff[d])))
    return torch.stack(out)


def _face_flux(u, kx, ja):
    """The face fluxes of the face region."""
    return torch.stack([0.5 * (_Fb(ja) * _Fb(kx[d]) * _Fb(u[d]) +
                               _Fb(ja, *E[d]) * _Fb(kx[d], *E[d]) * _Fb(u[d], *E[d])) for d in range(3)])


def _div(uu, ja):
    s = sum(_I(uu[d]) - _I(uu[d], *_neg(E[d])) for d in range(3))
    return s / _I(ja)


def _project(dt, ua, uua, p, kx, g):
    """u on the interior, uu on the face region."""
    u = torch.stack([_I(ua[d]) - dt * 0.5 * _I(kx[d]) * (_I(p, *E[d]) - _I(p, *_neg(E[d]))) for d in range(3)])
    uu = torch.stack([_Fb(uua[d]) - dt * 0.5 * (_Fb(g[d]) + _Fb(g[d], *E[d])) * (_Fb(p, *E[d]) - _Fb(p))
                      for d in range(3)])
    return u, uu


def _smagorinsky(Cs, u, kx, ja):
    gr = [[0.5 * _I(kx[e]) * (_I(u[d], *E[e]) - _I(u[d], *_neg(E[e]))) for e in range(3)] for d in range(3)]
    S = sum(2 * gr[d][d] ** 2 for d in range(3)) + (gr[0][1] + gr[1][0]) ** 2 + (gr[1][2] + gr[2][1]) ** 2 \
        + (gr[0][2] + gr[2][0]) ** 2
    return (Cs ** 2) * _I(ja) ** (2.0 / 3.0) * torch.sqrt(S)


def _face_cells(a, f, pos):
    """Ghost (0, -1) or interior (1, 2) cells of face f, counted from the face."""
    d, plus = f // 2, f % 2
    ax = a.ndim - 1 - d
    n = a.shape[ax]
    at = n - GC - pos if plus else GC - 1 + pos
    sl = [slice(None)] * (a.ndim - 3) + [slice(GC, -GC)] * 3
    sl[ax] = at
    return a[tuple(sl)]


def _bc_velocity(u, uprev, walls, lid, u_in, cx, dt, noise=None, faces=6):
    """In place: the channel's fills (inlet, outflow, slip) or the cavity's."""
    for f in range(faces):
        o1, o2, i1, i2 = (_face_cells(u, f, p) for p in (0, -1, 1, 2))
        if walls:
            v = torch.zeros((3, 1, 1), dtype=F64, device="cuda")
            if f == 3:
                v[0] = lid
            o1[...], o2[...] = 2 * v - i1, 2 * v - i2
        elif f == 0:
            v = torch.zeros_like(o1)
            v[0] = u_in
            if noise is not None:
                v += noise
            o1[...] = v
            o2[...] = v
        elif f == 1:
            p1, q1, q2 = (_face_cells(uprev, f, p) for p in (0, 1, 2))
            n = cx.shape[0]
            dxi = 1.0 / (cx[n - GC] - cx[n - GC - 1])
            ub = p1 - dt * (0.5 * dxi * (3 * p1 - 4 * q1 + q2))
            o2[...] = 2 * ub - i1
            o1[...] = ub
        else:
            ub = i1.clone()
            ub[f // 2] = 0.0
            o2[...] = 2 * ub - i1
            o1[...] = ub


def _bc_pressure(p, walls, faces=6):
    for f in range(faces):
        _face_cells(p, f, 0)[...] = 0.0 if (f == 1 and not walls) else _face_cells(p, f, 1)


def _mv(a, x):
    """A x on the interior."""
    return (_I(a[0]) * _I(x) + _I(a[2]) * _I(x, 1, 0, 0) + _I(a[1]) * _I(x, -1, 0, 0) + _I(a[4]) * _I(x, 0, 1, 0)
            + _I(a[3]) * _I(x, 0, -1, 0) + _I(a[6]) * _I(x, 0, 0, 1) + _I(a[5]) * _I(x, 0, 0, -1))


def _colours(shape):
    """Interior cells of the black and the red colour."""
    k, j, i = (torch.arange(m, device="cuda") for m in shape)
    odd = (i[None, None, :] + j[None, :, None] + k[:, None, None]) % 2 == 1
    odd = _I(odd)
    return ~odd, odd


def _sor(a, x, b, omega, colour):
    """One half-sweep, in place."""
    xi = _I(x)
    xi[...] = torch.where(colour, xi + omega * ((_I(b) - _mv(a, x)) / _I(a[0])), xi)


def _bicgstab(a, x, b, tol, pc_maxit, omega_pc, maxit=1000):
    """Right-preconditioned BiCGStab with red-black SOR sweeps, in place on x."""
    N = _I(b).numel()
    cols = _colours(b.shape)

    def precondition(v):
        w, full = torch.zeros_like(x), torch.zeros_like(x)
        _I(full)[...] = v
        for _ in range(max(1, pc_maxit)):
            for c in cols:
                _sor(a, w, full, omega_pc, c)
        return w

    r = _I(b) - _mv(a, x)
    rr, p, q = r.clone(), None, None
    rho_old, alpha, omega, it = 1.0, 0.0, 1.0, 0
    while True:
        rho = float((r * rr).sum())
        if abs(rho) < 1.17549435e-38:
            break
        p = r.clone() if it == 0 else r + (rho * alpha) / (rho_old * omega) * (p - omega * q)
        pp = precondition(p)
        q = _mv(a, pp)
        alpha = rho / float((rr * q).sum())
        s = r - alpha * q
        ss = precondition(s)
        t = _mv(a, ss)
        omega = float((t * s).sum()) / float((t * t).sum())
        _I(x)[...] += alpha * _I(pp) + omega * _I(ss)
        r = s - omega * t
        rho_old = rho
        it += 1
        if not (it < maxit and math.sqrt(float((r * r).sum())) / N > tol):
            break


def _sor_solve(a, x, b, tol, omega, maxit=100000):
    N = _I(b).numel()
    cols = _colours(b.shape)
    for _ in range(maxit):
        for c in cols:
            _sor(a, x, b, omega, c)
        if math.sqrt(float(((_I(b) - _mv(a, x)) ** 2).sum())) / N <= tol:
            break


def _philox_normals(seed, step, ja, kb):
    """Three N(0, 1) deviates per inlet cell: Philox4x32-10 keyed by the seed, counter (step, j, k), Box-Muller."""
    m32 = np.uint64(0xFFFFFFFF)
    j, k = np.meshgrid(np.asarray(ja, np.uint64), np.asarray(kb, np.uint64), indexing="xy")
    c = [np.full_like(j, step & 0xFFFFFFFF), np.full_like(j, step >> 32), j, k]
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        hi0, lo0, hi1, lo1 = p0 >> np.uint64(32), p0 & m32, p1 >> np.uint64(32), p1 & m32
        c = [hi1 ^ c[1] ^ np.uint64(k0), lo1, hi0 ^ c[3] ^ np.uint64(k1), lo0]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    s = 2.3283064365386963e-10
    u = [c[0].astype(np.float64) * s + s, c[1].astype(np.float64) * s, c[2].astype(np.float64) * s + s,
         c[3].astype(np.float64) * s]
    r1, r2 = np.sqrt(-2 * np.log(u[0])), np.sqrt(-2 * np.log(u[2]))
    return torch.from_numpy(np.stack([r1 * np.cos(2 * np.pi * u[1]), r1 * np.sin(2 * np.pi * u[1]),
                                      r2 * np.cos(2 * np.pi * u[3])])).cuda()


def _turn(v, ang, kind):
    x, y, z = v
    c, s = math.cos(ang), math.sin(ang)
    if kind == 1:
        return [x, c * y + s * z, -s * y + c * z]
    if kind == 2:
        return [c * x - s * z, y, s * x + c * z]
    if kind == 3:
        return [c * x + s * y, -s * x + c * y, z]
    return [x, y, z]


def _turn_dt(v, w, ang, om, kind):
    x, y, z = v
    c, s = math.cos(ang), math.sin(ang)
    r = _turn(w, ang, kind)
    if kind == 1:
        return [r[0], om * (-s * y + c * z) + r[1], om * (-c * y - s * z) + r[2]]
    if kind == 2:
        return [om * (-s * x - c * z) + r[0], r[1], om * (c * x - s * z) + r[2]]
    if kind == 3:
        return [om * (-s * x + c * y) + r[0], om * (-c * x - s * y) + r[1], r[2]]
    return r


def _rotor_forces(alm, centres, u, t, pitch=None, offset=None):
    """(ff, point forces, torque, thrust) of the actuator lines; pitch per
    turbine and blade, twist offsets per section, in degrees."""
    cx = [c.cpu().numpy() for c in centres]
    nap, nb, napb = alm.n_ap, alm.n_blade, alm.n_ap_per_blade
    npt = nb * napb
    attack, cl, cd = alm.attack, alm.cl.reshape(-1, nap), alm.cd.reshape(-1, nap)
    dr = (alm.struct.radius - alm.struct.hub_radius) / napb
    pos, force = np.zeros((nap, 3)), np.zeros((nap, 3))
    torque, thrust = np.zeros(alm.n_turbine), np.zeros(alm.n_turbine)
    for tid in range(alm.n_turbine):
        T = alm.turbines[tid]
        kind, ang, om = T.angle_type, 0.0, 0.0
        base, bvel = np.array(T.base[:]), np.zeros(3)
        if kind:
            ang = T.motion[0] * math.sin(T.motion[1] * t + T.motion[2])
            om = T.motion[0] * T.motion[1] * math.cos(T.motion[1] * t + T.motion[2])
        if T.surge[0]:
            base[0] += T.surge[0] * math.sin(T.surge[1] * t + T.surge[2])
            bvel[0] += T.surge[0] * T.surge[1] * math.cos(T.surge[1] * t + T.surge[2])
        ids = np.arange(tid * npt, (tid + 1) * npt)
        r, chord, twist = alm.ap_r[ids], alm.ap_chord[ids], alm.ap_twist[ids]
        blade = (ids - tid * npt) // napb
        if pitch is not None:
            twist = twist + pitch[tid][blade] + offset[ids % napb]
        theta = T.tip_rate * t + 2 * math.pi / nb * blade
        P = np.stack(_turn([np.full(npt, T.hub[0]), T.hub[1] + r * np.cos(theta), T.hub[2] + r * np.sin(theta)],
                           -ang, kind), 1) + base
        pos[ids] = P
        idx = [np.searchsorted(cx[m], P[:, m], side="right") - 1 for m in range(3)]
        inside = np.ones(npt, bool)
        for m in range(3):
            inside &= (idx[m] >= GC - 1) & (idx[m] < len(cx[m]) - GC - 1)
            idx[m] = np.clip(idx[m], 0, len(cx[m]) - 2)
        fr = [(P[:, m] - cx[m][idx[m]]) / (cx[m][idx[m] + 1] - cx[m][idx[m]]) for m in range(3)]
        uap = np.zeros((npt, 3))
        for q in range(8):
            o = (q & 1, (q >> 1) & 1, q >> 2)
            w = np.prod([fr[m] if o[m] else 1 - fr[m] for m in range(3)], axis=0)
            at = [torch.from_numpy(idx[m] + o[m]).cuda() for m in range(3)]
            uap += w[:, None] * u[:, at[2], at[1], at[0]].T.cpu().numpy()
        ut = _turn_dt((P - base).T, (uap - bvel).T, ang, om, kind)
        utan = T.tip_rate * r + ut[1] * np.sin(theta) - ut[2] * np.cos(theta)
        rel2 = ut[0] ** 2 + utan ** 2
        phi = np.arctan(ut[0] / utan)
        att = np.degrees(phi) - twist
        CL = np.array([np.interp(v, attack, cl[:, i]) for v, i in zip(att, ids)])
        CD = np.array([np.interp(v, attack, cd[:, i]) for v, i in zip(att, ids)])
        fl, fd = 0.5 * CL * rel2 * chord * dr, 0.5 * CD * rel2 * chord * dr
        fx = np.where(inside, fl * np.cos(phi) + fd * np.sin(phi), 0.0)
        ft = np.where(inside, (fl * np.sin(phi) - fd * np.sin(phi)) * np.sign(T.tip_rate), 0.0)
        force[ids] = np.stack(_turn([-fx, ft * np.sin(theta), -ft * np.cos(theta)], -ang, kind), 1)
        torque[tid], thrust[tid] = np.sum(np.abs(ft) * r), np.sum(fx)
    eps = alm.struct.eps
    eta = 1.0 / (eps * math.sqrt(math.pi)) ** 3
    ex, ey, ez = (torch.exp(-((c[None, :] - torch.from_numpy(pos[:, m:m + 1].copy()).cuda()) / eps) ** 2)
                  for m, c in enumerate(centres))
    ff = torch.zeros((3,) + tuple(u.shape[1:]), dtype=F64, device="cuda")
    plane = (ey[:, :, None] * ex[:, None, :]).reshape(nap, -1)
    F = torch.from_numpy(force).cuda() * eta
    for m in range(3):
        _I(ff[m])[...] = _I(((ez * F[:, m:m + 1]).T.contiguous() @ plane).reshape(u.shape[1:]))
    return ff, force, torque, thrust


# ------------------------------------------------------------- inputs
def _cast(case, *arrays):
    t = F32 if case["prec"] == "f32" else F64
    return [a.to(t).contiguous() for a in arrays]


def _step_fields(case, seed):
    """A turbulent flow's fields on the case's mesh, dx = 1/32."""
    n, gen = _n(case), _gen(seed)
    mesh = _Mesh(n, 1.0 / 32, case.get("stretch", 0.0))
    u = _field(n, 3, gen, 0.0, 0.3)
    u[0] += 1.0
    uu = torch.zeros_like(u)
    _Fb(uu[0])[...], _Fb(uu[1])[...], _Fb(uu[2])[...] = _face_flux(u, mesh.kx, mesh.ja)
    nut = 1e-4 * (1.0 + _field(n, 1, gen, 0.0, 0.4)[0].abs())
    return n, gen, mesh, u, uu, nut


_DT = 0.1 / 32
_RE = 2.5e5


def _predict_inputs(case, seed):
    n, gen, mesh, u, uu, nut = _step_fields(case, seed)
    un = u + 1e-3 * _field(n, 3, gen)
    ff = _field(n, 3, gen, 0.0, 0.2)
    return dict(zip(("un", "u", "uu", "nut", "kx", "g", "ja", "ff"),
                    _cast(case, un, u, uu, nut, mesh.kx, mesh.g, mesh.ja, ff)))


def _correct_inputs(case, seed):
    n, gen, mesh, u, uu, nut = _step_fields(case, seed)
    p = _field(n, 1, gen, 0.0, 0.05)[0]
    uprev = u + 1e-3 * _field(n, 3, gen)
    return dict(zip(("ua", "uua", "p", "uprev", "um", "pm", "kx", "g", "ja", "xyz"),
                    _cast(case, u, uu, p, uprev, u + 0.01 * _field(n, 3, gen), p * 0.9, mesh.kx, mesh.g, mesh.ja,
                          mesh.xyz)))


def _poisson_inputs(case, seed):
    """The pressure of the previous step and a right-hand side whose
    solution it is up to the step's change."""
    n, gen = _n(case), _gen(seed)
    mesh = _Mesh(n, 1.0 / 32, case["stretch"])
    a, _ = _poisson_matrix(mesh, case["outlet"])
    p = _field(n, 1, gen, 0.0, 1.0, 0.0)[0]
    inner = torch.zeros_like(p)
    _I(inner)[...] = _I(p)
    b = torch.zeros_like(p)
    _I(b)[...] = _mv(a, inner)
    x0 = inner.clone()
    for width in (1, 2, 4, 8):  # the change has eddies of all sizes up to some cells
        part = torch.randn([1, 1] + [max(1, m // width) for m in p.shape], generator=gen, dtype=F64, device="cuda")
        if width > 1:
            part = torch.nn.functional.interpolate(part, tuple(p.shape), mode="trilinear")
        _I(x0)[...] += 2e-3 * width * _I(part[0, 0])
    return a, x0, b


def _smooth_inputs(case, seed):
    n, gen = _n(case), _gen(seed)
    mesh = _Mesh(n, 1.0 / 32, case["stretch"])
    a, _ = _poisson_matrix(mesh, True)
    x = torch.zeros_like(a[0])
    _I(x)[...] = _I(_field(n, 1, gen, 0.0, 1.0, 0.1)[0])
    b = torch.zeros_like(x)
    _I(b)[...] = 0.01 * _I(_field(n, 1, gen, 0.0, 1.0, 1.0)[0])
    return _cast(case, a, x, b)


def _backward_inputs(case, seed):
    n, gen, mesh, u, uu, nut = _step_fields(case, seed)
    d = dict(u=u, uu=uu, nut=nut, kx=mesh.kx.contiguous(), g=mesh.g.contiguous(), ja=mesh.ja, xyz=mesh.xyz)
    d["ub"] = _field(n, 3, gen, 0.0, 1.0, 0.3)
    d["uub"] = torch.zeros_like(uu)
    _Fb(d["uub"])[...] = _Fb(_field(n, 3, gen, 0.0, 1.0, 0.3))
    d["rhsb"] = torch.zeros_like(nut)
    _I(d["rhsb"])[...] = _I(_field(n, 1, gen, 0.0, 1.0, 0.3)[0])
    return d


def _rotor_setup(case, n, h):
    """Rotors in a row down the channel, the first on a moving platform on request."""
    D = case["cells_per_d"] * h
    mid = (0.5 * n[1] * h, 0.5 * n[2] * h)
    at = [(n[0] * h * f,) + mid for f in ((0.3,) if case["rotors"] == 1 else (0.25, 0.65))]
    kw = {}
    if case.get("motion"):
        kw = dict(angle_type=2, motion=(math.radians(3.0), 0.7, 0.5), surge=(0.1 * D, 0.7, 0.0))
    return setups.rotor(h, at[0], radius=0.5 * D, extra_bases=at[1:], chord=(0.08 * D, 0.02 * D), **kw)


def _driver_setup(case, seed):
    n = _n(case)
    precision = abi.CASE_MIXED if case.get("mixed") else abi.CASE_F64
    if case["kind"] == "cavity":
        if n[2] == 1:
            return setups.lid2d(n=n[0], tol=case["tol"])
        return setups.lid3d(n=n, dt=0.05 / n[0], precision=precision, tol=case["tol"])
    s = setups.windtunnel(n=n, cells_per_d=case["cells_per_d"], cfl=0.1, seed=int(seed) + 1, precision=precision,
                          with_rotor=False, pc_maxit=case.get("pc_maxit", 1), tol=case["tol"])
    if case["rotors"]:
        alm = _rotor_setup(dict(case, motion=case["rotors"] > 1), n, s.struct.h[0])
        s = setups.CaseSetup(s.struct, alm, s.name)
    return s


def _driver_start(case, seed, setup):
    """The fields (u, uu, nut) a run starts from: the driver's own uniform
    stream in a channel (its inlet noise is seeded), seeded eddies in a cavity."""
    n, gen, h = _n(case), _gen(seed), setup.struct.h[0]
    mesh = _Mesh(n, h)
    flat = n[2] == 1
    if case["kind"] == "cavity":
        u = _field(n, 3, gen, 0.0, 0.1, 0.0)
        for m in range(3):  # a flow that vanishes at the walls
            for ax in range(2 if flat else 3):
                i = torch.arange(n[ax] + 2 * GC, dtype=F64, device="cuda")
                w = torch.sin(math.pi * ((i - GC + 0.5) / n[ax]).clamp(0, 1))
                u[m] *= w.reshape([-1 if q == 2 - ax else 1 for q in range(3)])
        if flat:
            u[2] = 0.0
        _bc_velocity(u, u, True, 1.0, 0.0, None, 0.0, faces=4 if flat else 6)
        if flat:
            u[:] = u[:, GC:GC + 1].clone()
        if case["mixed"]:
            u = u.to(F32).to(F64)
    else:
        u = torch.zeros((3,) + tuple(mesh.ja.shape), dtype=F64, device="cuda")
        u[0] = 1.0
    uu = torch.zeros_like(u)
    _Fb(uu)[...] = _face_flux(u, mesh.kx, mesh.ja)
    nut = torch.zeros_like(u[0])
    if not flat:
        _I(nut)[...] = _smagorinsky(setup.struct.Cs, u, mesh.kx, mesh.ja)
    return mesh, u, uu, nut


_RESTART = (abi.FIELD_U, abi.FIELD_UU, abi.FIELD_P, abi.FIELD_NUT)


def _start_driver(case, seed):
    """The set-up, the run after its first `spin` steps and, for the smaller
    domains, the restart file every pass continues from."""
    setup = _driver_setup(case, seed)
    c = rt.Case(setup)
    if case["kind"] == "cavity":
        _, u, uu, nut = _driver_start(case, seed, setup)
        for f, v in ((abi.FIELD_U, u), (abi.FIELD_UU, uu), (abi.FIELD_NUT, nut)):
            c.set(f, v.cpu().numpy().reshape(-1))
    c.step(case["spin"])
    restart = [(f, c.get(f)) for f in _RESTART] if _cells(case) <= 600_000 and case["kind"] != "gradient" else []
    return setup, c, restart


def _angles(alm, seed):
    rng = np.random.default_rng(int(seed))
    return (torch.from_numpy(rng.uniform(-1, 1, (alm.n_turbine, alm.n_blade))),
            torch.from_numpy(rng.uniform(-0.5, 0.5, alm.n_ap_per_blade)))


def _dom(n):
    return abi.Domain.make(_pad(n), gc=GC)


def prepare(case, seed):
    rt.init(0)
    torch.cuda.set_device(0)
    n, kind = _n(case), case["kind"]
    s = dict(case=case, dom=_dom(n))
    if kind == "predict":
        s.update(_predict_inputs(case, seed))
        s["ua"], s["uu1"], s["rhs"] = s["u"].clone(), torch.zeros_like(s["uu"]), torch.zeros_like(s["nut"])
    elif kind == "correct":
        s.update(_correct_inputs(case, seed))
        s["u"], s["uu"] = torch.zeros_like(s["ua"]), torch.zeros_like(s["uua"])
        s["nut"], s["div"] = torch.zeros_like(s["p"]), torch.zeros_like(s["p"])
        s["faces"], s["pfaces"] = _faces(case["walls"])
    elif kind == "poisson":
        s["a"], s["x0"], s["b"] = _poisson_inputs(case, seed)
        s["x"] = torch.zeros_like(s["x0"])
        cfg = abi.solver_config(type=abi.LS_PBICGSTAB, maxit=1000, tol=case["tol"], pc_type=abi.LS_SOR,
                                pc_maxit=case["pc_maxit"], pc_relax=case["pc_relax"],
                                precision=abi.SOLVE_MIXED if case["mixed"] else abi.SOLVE_F64)
        s["solver"] = rt.Solver(s["dom"], cfg)
        if case["declared"]:
            s["solver"].set_matrix(s["a"])
    elif kind == "rotor":
        mesh, gen = _Mesh(n, 1.0 / case["cells_per_d"], fields=False), _gen(seed)
        u = _field(n, 3, gen, 0.0, 0.1)
        u[0] += 1.0
        (s["u"],) = _cast(case, u)
        s["ff"] = torch.zeros_like(s["u"])
        setup = _rotor_setup(case, n, 1.0 / case["cells_per_d"])
        s["alm"] = rt.Alm(s["dom"], setup, *[c.cpu().numpy() for c in mesh.c])
    elif kind == "smooth":
        s["a"], s["x"], s["b"] = _smooth_inputs(case, seed)
        s["r"], s["ar"], s["xn"] = (torch.zeros_like(s["x"]) for _ in range(3))
    elif kind == "backward":
        s.update(_backward_inputs(case, seed))
        s["faces"], s["pfaces"] = _faces(False)
        m = s["ja"].numel()
        s["out"] = torch.zeros(17 * m, dtype=F64, device="cuda")
        at = 0
        for name, ncol in (("usb", 3), ("unb", 3), ("uab", 3), ("uusb", 3), ("uunb", 3), ("pb", 1), ("nutb", 1)):
            shape = ((ncol,) if ncol > 1 else ()) + tuple(s["ja"].shape)
            s[name] = s["out"][at * m:(at + ncol) * m].view(shape)
            at += ncol
        s["ffb"] = torch.zeros_like(s["u"])
    elif kind in ("tunnel", "cavity"):
        s["setup"], s["run"], s["restart"] = _start_driver(case, seed)
    else:
        s["setup"], s["run"], _ = _start_driver(case, seed)
        s["pitch"], s["twist"] = _angles(s["setup"].alm, seed)
    return s


def _faces(walls):
    arr = (abi.FaceBC * 6)()
    if walls:
        for f in range(6):
            arr[f].type = abi.BC_REFLECT
        arr[3].value[0] = 1.0
        return arr, (C.c_int * 6)(*([abi.PBC_NEUMANN] * 6))
    for f, t in enumerate((abi.BC_INLET, abi.BC_CONVECTIVE, abi.BC_SLIP, abi.BC_SLIP, abi.BC_SLIP, abi.BC_SLIP)):
        arr[f].type = t
    arr[0].value[0] = 1.0
    return arr, (C.c_int * 6)(abi.PBC_NEUMANN, abi.PBC_ZERO, *([abi.PBC_NEUMANN] * 4))


_MAXDIAG = 6144.0
_CS = 0.1
_COUNT = 50  # steps in the running mean


def run(s):
    return globals()["_run_" + s["case"]["kind"]](s)


def _prec(s):
    return abi.F32 if s["case"]["prec"] == "f32" else abi.F64


def _P(s, *names):
    return [rt.ptr(s[k]) for k in names]


def _run_predict(s):
    dom, pr = C.byref(s["dom"]), _prec(s)
    rt.call("falm_pseudo_u", dom, pr, SCHEMES[s["case"]["scheme"]], 1.0 / _RE, _DT,
            *_P(s, "un", "u", "uu", "ua", "nut", "kx", "g", "ja", "ff"), None)
    rt.call("falm_u_to_uu", dom, pr, *_P(s, "ua", "uu1", "kx", "ja"), None)
    rt.call("falm_poisson_rhs", dom, pr, *_P(s, "uu1", "rhs", "ja"), _DT, _MAXDIAG, None)
    return dict(ua=s["ua"], uu=s["uu1"], rhs=s["rhs"])


def _run_correct(s):
    dom, pr = C.byref(s["dom"]), _prec(s)
    rt.call("falm_bc_pressure", dom, pr, s["pfaces"], rt.ptr(s["p"]), None)
    rt.call("falm_project_p", dom, pr, _DT, *_P(s, "u", "ua", "uu", "uua", "p", "kx", "g"), None)
    rt.call("falm_bc_velocity", dom, pr, s["faces"], *_P(s, "u", "uprev", "xyz"), _DT, None, None)
    rt.call("falm_sgs", dom, pr, abi.SGS_SMAGORINSKY, _CS, *_P(s, "u", "nut", "kx", "ja"), None)
    rt.call("falm_divergence", dom, pr, *_P(s, "uu", "div", "ja"), None)
    norm = C.c_double()
    rt.call("falm_norm2", dom, pr, rt.ptr(s["div"]), 1, C.byref(norm), None)
    w = 1.0 / _COUNT
    for mean, v in (("um", "u"), ("pm", "p")):
        rt.call("falm_vecaxby", pr, 1.0 - w, rt.ptr(s[mean]), w, rt.ptr(s[v]), rt.ptr(s[mean]), s[v].numel(), None)
    return dict(u=s["u"], uu=s["uu"], nut=s["nut"], div=s["div"], norm=norm.value, um=s["um"], pm=s["pm"])


def _run_poisson(s):
    s["x"].copy_(s["x0"])
    s["solver"].solve(s["a"], s["x"], s["b"], None)
    return s["x"]


def _run_rotor(s):
    s["alm"].step(_prec(s), s["u"], s["ff"], 0.37)
    _, force, torque, thrust = s["alm"].get()
    return dict(ff=s["ff"], force=force, torque=torque, thrust=thrust)


def _run_smooth(s):
    """A smoothing pass and a minimal-residual correction: x += w r with w = (r, A r) / (A r, A r)."""
    dom, pr = C.byref(s["dom"]), _prec(s)
    x = "x"
    if s["case"]["sweep"] == "sor":
        for colour in (abi.BLACK, abi.RED):
            rt.call("falm_sor_sweep", dom, pr, *_P(s, "a", "x", "b"), 1.2, colour, None)
    else:
        rt.call("falm_jacobi_sweep", dom, pr, *_P(s, "a", "xn", "x", "b"), None)
        x = "xn"
    rt.call("falm_residual", dom, pr, *_P(s, "a", x, "b", "r"), None)
    rt.call("falm_mv", dom, pr, *_P(s, "a", "r", "ar"), None)
    num, den = C.c_double(), C.c_double()
    rt.call("falm_dot", dom, pr, *_P(s, "r", "ar"), C.byref(num), None)
    rt.call("falm_norm2", dom, pr, rt.ptr(s["ar"]), 1, C.byref(den), None)
    w = num.value / den.value if den.value > 0.0 else 0.0
    rt.call("falm_vecaxby", pr, 1.0, rt.ptr(s[x]), w, rt.ptr(s["r"]), rt.ptr(s["x"]), s["x"].numel(), None)
    return dict(x=s["x"], r=s["r"], ar=s["ar"])


def _run_backward(s):
    dom = C.byref(s["dom"])
    s["out"].zero_()
    rt.call("falm_bc_velocity_vjp", dom, s["faces"], rt.ptr(s["xyz"]), _DT, *_P(s, "ub", "usb", "unb"), None)
    rt.call("falm_project_p_vjp", dom, _DT, *_P(s, "kx", "g", "usb", "uub", "uab", "uusb", "pb"), None)
    rt.call("falm_bc_pressure_vjp", dom, s["pfaces"], rt.ptr(s["pb"]), None)
    rt.call("falm_poisson_rhs_vjp", dom, rt.ptr(s["ja"]), _DT, _MAXDIAG, *_P(s, "rhsb", "uusb"), None)
    rt.call("falm_u_to_uu_vjp", dom, *_P(s, "kx", "ja", "uusb", "uab"), None)
    rt.call("falm_pseudo_u_vjp", dom, SCHEMES[s["case"]["scheme"]], 1.0 / _RE, _DT,
            *_P(s, "u", "uu", "nut", "kx", "g", "ja", "uab", "unb", "uunb", "nutb", "ffb"), None)
    rt.call("falm_sgs_vjp", dom, _CS, *_P(s, "u", "kx", "ja", "nutb", "unb"), None)
    return {k: s[k] for k in ("usb", "unb", "uab", "uusb", "uunb", "pb", "nutb", "ffb")}


def _run_tunnel(s):
    for field, values in s["restart"]:
        s["run"].set(field, values)
    s["run"].step(s["case"]["steps"])
    return dict(u=s["run"].get(abi.FIELD_U), p=s["run"].get(abi.FIELD_P))


_run_cavity = _run_tunnel


def _run_gradient(s):
    from falm_amd.adjoint import rotor_power
    pitch, twist = s["pitch"].clone().requires_grad_(), s["twist"].clone().requires_grad_()
    J = rotor_power(s["run"], pitch, twist, s["case"]["steps"], s["case"]["ckpt"], 1e-11)
    J.backward()
    return dict(power=J.detach(), pitch=pitch.grad, twist=twist.grad)


# -------------------------------------------------------------- 64 bits
def exact(case, seed):
    rt.init(0)
    torch.cuda.set_device(0)
    f = globals().get("_exact_" + case["kind"])
    return None if f is None else f(case, seed)


def _full(shape, part, where):
    out = torch.zeros(shape, dtype=F64, device="cuda")
    where(out)[...] = part
    return out


def _exact_predict(case, seed):
    d = {k: v.to(F64) for k, v in _predict_inputs(case, seed).items()}
    ua = d["u"].clone()
    _I(ua)[...] = _pseudo_u(case["scheme"], 1.0 / _RE, _DT, *(d[k] for k in ("un", "u", "uu", "nut", "kx", "g", "ja",
                                                                             "ff")))
    uu = _full(ua.shape, _face_flux(ua, d["kx"], d["ja"]), _Fb)
    return dict(ua=ua, uu=uu, rhs=_full(d["ja"].shape, _div(uu, d["ja"]) / (_DT * _MAXDIAG), _I))


def _exact_correct(case, seed):
    d = {k: v.to(F64) for k, v in _correct_inputs(case, seed).items()}
    walls = case["walls"]
    _bc_pressure(d["p"], walls)
    ui, uuf = _project(_DT, d["ua"], d["uua"], d["p"], d["kx"], d["g"])
    u, uu = _full(d["ua"].shape, ui, _I), _full(d["ua"].shape, uuf, _Fb)
    _bc_velocity(u, d["uprev"], walls, 1.0, 1.0, d["xyz"][0][0, 0], _DT)
    nut = _full(d["ja"].shape, _smagorinsky(_CS, u, d["kx"], d["ja"]), _I)
    div = _full(d["ja"].shape, _div(uu, d["ja"]), _I)
    w = 1.0 / _COUNT
    return dict(u=u, uu=uu, nut=nut, div=div, norm=float((div ** 2).sum()), um=(1 - w) * d["um"] + w * u,
                pm=(1 - w) * d["pm"] + w * d["p"])


def _exact_poisson(case, seed):
    a, x, b = _poisson_inputs(case, seed)
    _bicgstab(a, x, b, case["tol"], case["pc_maxit"], case["pc_relax"])
    return x


def _exact_rotor(case, seed):
    n = _n(case)
    mesh, gen = _Mesh(n, 1.0 / case["cells_per_d"], fields=False), _gen(seed)
    u = _field(n, 3, gen, 0.0, 0.1)
    u[0] += 1.0
    u = _cast(case, u)[0].to(F64)
    ff, force, torque, thrust = _rotor_forces(_rotor_setup(case, n, 1.0 / case["cells_per_d"]), mesh.c, u, 0.37)
    return dict(ff=ff, force=force, torque=torque, thrust=thrust)


def _exact_smooth(case, seed):
    a, x, b = (v.to(F64) for v in _smooth_inputs(case, seed))
    if case["sweep"] == "sor":
        for c in _colours(x.shape):
            _sor(a, x, b, 1.2, c)
    else:
        x = _full(x.shape, _I(x) + (_I(b) - _mv(a, x)) / _I(a[0]), _I)
    r = _full(x.shape, _I(b) - _mv(a, x), _I)
    ar = _full(x.shape, _mv(a, r), _I)
    return dict(x=x + float((r * ar).sum()) / float((ar * ar).sum()) * r, r=r, ar=ar)


def _vjp(f, inputs, cot):
    with torch.enable_grad():
        xs = [x.detach().clone().requires_grad_() for x in inputs]
        return torch.autograd.grad(f(*xs), xs, cot)


def _exact_backward(case, seed):
    d = _backward_inputs(case, seed)
    u, uu, nut, kx, g, ja = (d[k] for k in ("u", "uu", "nut", "kx", "g", "ja"))
    zero = torch.zeros_like(u)

    def fill(us, un):  # the boundary fill of the interior us with the previous un
        v = _full(us.shape, _I(us), _I)
        _bc_velocity(v, un, False, 0.0, 1.0, d["xyz"][0][0, 0], _DT)
        return v

    usb, unb = _vjp(fill, (u, u), d["ub"])
    p0 = torch.zeros_like(ja)

    def project(ua, uua, p):
        a, b = _project(_DT, ua, uua, p, kx, g)
        return _full(u.shape, a, _I), _full(u.shape, b, _Fb)

    uab, uusb, pb = _vjp(project, (zero, zero, p0), (usb * _full(u.shape, 1.0, _I), d["uub"]))

    def pfill(p):
        q = p.clone()
        _bc_pressure(q, False)
        return q

    (pb,) = _vjp(pfill, (p0,), pb)
    uusb = uusb + _vjp(lambda f: _full(ja.shape, _div(f, ja) / (_DT * _MAXDIAG), _I), (zero,), d["rhsb"])[0]
    uab = uab + _vjp(lambda v: _full(u.shape, _face_flux(v, kx, ja), _Fb), (zero,), uusb)[0]
    gu, guu, gn, gf = _vjp(lambda v, f, nu, ff: _full(u.shape, _pseudo_u(case["scheme"], 1.0 / _RE, _DT, v, v, f, nu,
                                                                         kx, g, ja, ff), _I),
                           (u, uu, nut, zero), uab)
    unb = unb + gu + _vjp(lambda v: _full(ja.shape, _smagorinsky(_CS, v, kx, ja), _I), (u,), gn)[0]
    return dict(usb=usb, unb=unb, uab=uab, uusb=uusb, uunb=guu, pb=pb, nutb=gn, ffb=gf)


def _march(case, seed, pitch=None, twist=None):
    """The driver's first steps and the pass's; returns u and the pass's mean rotor power."""
    n, walls, flat = _n(case), case["kind"] == "cavity", case["nz"] == 1
    setup = _driver_setup(case, seed)
    st = setup.struct
    mesh, u, uu, nut = _driver_start(case, seed, setup)
    a, md = _poisson_matrix(mesh, not walls, flat)
    p, ff = torch.zeros_like(nut), torch.zeros_like(u)
    nf, power = 4 if flat else 6, 0.0

    def flatten(v):
        if flat:
            v[...] = v[..., GC:GC + 1, :, :].clone()

    spin, steps = case["spin"], case["steps"]
    for it in range(1, spin + steps + 1):
        t = st.dt * it
        uprev = u.clone()
        if setup.alm is not None:
            turned = (pitch, twist) if it > spin else (None, None)
            ff, _, torque, _ = _rotor_forces(setup.alm, mesh.c, u, t, *turned)
            if it > spin:
                power += float(sum(setup.alm.turbines[q].tip_rate * torque[q] for q in range(len(torque))))
        u = uprev.clone()
        _I(u)[...] = _pseudo_u("Upwind3", 1.0 / st.Re, st.dt, uprev, uprev, uu, nut, mesh.kx, mesh.g, mesh.ja, ff)
        _Fb(uu)[...] = _face_flux(u, mesh.kx, mesh.ja)
        if walls:
            for f in range(nf):
                _face_cells(uu[f // 2], f, f % 2)[...] = 0.0
        rhs = _full(p.shape, _div(uu, mesh.ja) / (st.dt * md), _I)
        if flat:
            _sor_solve(a, p, rhs, st.solver.tol, st.solver.relax)
        else:
            _bicgstab(a, p, rhs, st.solver.tol, st.solver.pc_maxit, st.solver.pc_relax)
        _bc_pressure(p, walls, nf)
        flatten(p)
        ui, uuf = _project(st.dt, u, uu, p, mesh.kx, mesh.g)
        _I(u)[...] = ui
        _Fb(uu)[...] = uuf
        noise = None
        if not walls:
            noise = st.inlet_intensity * _philox_normals(st.seed, it, range(GC, GC + n[1]), range(GC, GC + n[2]))
        _bc_velocity(u, uprev, walls, st.lid_velocity, st.u_inflow, mesh.c[0], st.dt, noise, nf)
        flatten(u)
        if not flat:
            _I(nut)[...] = _smagorinsky(st.Cs, u, mesh.kx, mesh.ja)
    return u, power / steps


def _exact_tunnel(case, seed):
    """The pressure is left out: the solve's tolerance leaves its smoothest
    modes open, and the velocity does not feel them."""
    u, _ = _march(case, seed)
    return dict(u=u.reshape(-1), p=None)


_exact_cavity = _exact_tunnel


def _exact_gradient(case, seed):
    """The power by the forward window; the gradient has no 64-bit
    restatement that is quick enough."""
    pitch, twist = _angles(_driver_setup(case, seed).alm, seed)
    _, power = _march(case, seed, pitch.numpy(), twist.numpy())
    return dict(power=torch.tensor(power, dtype=F64), pitch=None, twist=None)
