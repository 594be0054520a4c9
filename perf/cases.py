"""Performance cases of the HO-CXX time-step path on one GPU, through the package's entry points.

Each case is what a program using the framework does again and again: advance a flow, solve the
stream function of a vorticity field, apply the Poisson operator inside a loop of its own, run an
outer step of a hybrid coupling, or take the gradient of a run.  Handles are set up in `prepare`
(a program sets a mesh up once and then marches), and every pass restarts from the same given
vorticity, so that a pass is the same work however often it ran before.

`exact` restates the flux-reconstruction discretisation for uniform cavities in plain torch
(FP64, dense: on such a mesh the Poisson operator is a Kronecker sum, solved by its eigenvectors).
"""
import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "ho-cxx_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "ho-cxx_amd"))

import hoc  # noqa: E402
from hoc import meshes  # noqa: E402

# rho(J^-1 A) / n^2 of the FR Laplacian on an n x n unit cavity (K: points per direction)
RHO = {2: 48.0, 3: 149.4, 4: 373.9, 5: 799.5, 6: 1523.0}
REAL_LIMIT = {1: 2.0, 2: 2.0, 4: 2.785}  # |z| on the negative real axis inside the RK stability region
SCRATCH = 64 << 20                       # bytes of face traces the no-allocation operator apply takes


def listed():
    return [
        # the operator inside a caller's own loop (a Krylov method, a spectrum): the smallest call,
        # where launches are all there is, and the largest the entry point takes (its 64 MiB scratch)
        dict(name="laplacian_16_K3", path="laplacian", mesh="cavity", n=16, jitter=0.0, K=3),
        dict(name="laplacian_440_K5", path="laplacian", mesh="cavity", n=440, jitter=0.0, K=5),
        # stream function of a given vorticity from a zero guess (initialisation, diagnostics)
        dict(name="poisson_101_K6", path="poisson", mesh="cavity", n=101, jitter=0.0, K=6, precision="fp64", tol=1e-12),
        # the parity-size cavity run of the reference's own decks: latency-bound marching
        dict(name="step_cavity32_K4", path="step", mesh="cavity", n=32, jitter=0.0, K=4, precision="fp64", Re=100.0,
             integ=4, adv=1, tol=1e-12, steps=10),
        # an ordinary run at a higher Reynolds number, odd size
        dict(name="step_cavity127_K5", path="step", mesh="cavity", n=127, jitter=0.0, K=5, precision="fp64", Re=1000.0,
             integ=4, adv=1, tol=1e-12, steps=8),
        # the benchmark cavity, plain FP64: the largest march
        dict(name="step_cavity512_K5", path="step", mesh="cavity", n=512, jitter=0.0, K=5, precision="fp64", Re=100.0,
             integ=4, adv=1, tol=1e-10, steps=5),
        # mixed precision (FP32 preconditioner) at an ordinary large size
        dict(name="step_cavity320_K5_mixed", path="step", mesh="cavity", n=320, jitter=0.0, K=5, precision="mixed",
             Re=400.0, integ=4, adv=1, tol=1e-12, steps=5),
        # backward-facing step at the size of the reference's case: distorted elements, BiCGSTAB,
        # inflow and outflow
        dict(name="step_bfs384_K5", path="step", mesh="bfs", n=384, jitter=0.1, K=5, precision="fp64", Re=400.0,
             integ=4, adv=1, tol=1e-12, steps=3),
        # curved quadratic elements around a cylinder, the highest order
        dict(name="step_cylinder96_K6", path="step", mesh="cylinder", n=96, jitter=0.0, K=6, precision="fp64", Re=100.0,
             integ=4, adv=1, tol=1e-13, steps=2),
        # many small cavities of ragged sizes advanced together (parameter sweeps)
        dict(name="ensemble_K5", path="ensemble", mesh="cavity", sizes="16,91,33,64,47,24,72,57,38,19,83,28", K=5,
             precision="fp64", integ=4, adv=1, tol=1e-12, steps=3),
        # one outer step of a hybrid (vortex-particle) coupling: driver values in, sub-steps, field out
        dict(name="hybrid_open48_K4", path="hybrid", mesh="cavity", n=48, jitter=0.0, K=4, precision="fp64", Re=200.0,
             integ=2, adv=2, tol=1e-12, steps=4),
        # gradient of the final enstrophy with respect to the initial field and the lid: forward
        # and reverse sweep
        dict(name="adjoint_24_K4", path="adjoint", mesh="cavity", n=24, jitter=0.0, K=4, precision="fp64", Re=1000.0,
             integ=4, adv=1, tol=1e-13, steps=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    p = rng.random()
    K = rng.choice([2, 3, 4, 4, 5, 5, 6])
    if p < 0.15:
        n = _log(rng, 12, min(440, int(math.sqrt(SCRATCH / (64.0 * K)))))
        jit = rng.choice([0.0, 0.0, 0.1])
        return dict(path="laplacian", mesh="cavity", n=n, jitter=jit, K=K)
    if p < 0.25:
        return dict(path="poisson", mesh="cavity", n=_log(rng, 12, 256), jitter=0.0, K=K,
                    precision=rng.choice(["fp64", "mixed"]), tol=1e-12)
    if p < 0.62:
        n = _log(rng, 12, 400)
        return dict(path="step", mesh="cavity", n=n, jitter=0.0, K=K, precision=rng.choice(["fp64", "fp64", "mixed"]),
                    Re=round(math.exp(rng.uniform(math.log(100.0), math.log(3200.0))), 1),
                    integ=rng.choice([4, 4, 4, 2, 1]), adv=rng.choice([1, 1, 2]), tol=1e-12,
                    steps=max(2, min(10, 1200 // n)))
    if p < 0.72:
        return dict(path="step", mesh="bfs", n=12 * _log(rng, 4, 32), jitter=0.1, K=K,
                    precision=rng.choice(["fp64", "mixed"]), Re=400.0, integ=4, adv=1, tol=1e-12, steps=2)
    if p < 0.80:
        return dict(path="step", mesh="cylinder", n=_log(rng, 16, 96), jitter=0.0, K=max(K, 4),
                    precision="fp64", Re=100.0, integ=4, adv=1, tol=1e-13, steps=2)
    if p < 0.90:
        m = rng.randint(3, 16)
        return dict(path="ensemble", mesh="cavity", sizes=",".join(str(_log(rng, 12, 96)) for _ in range(m)), K=K,
                    precision=rng.choice(["fp64", "mixed"]), integ=4, adv=1, tol=1e-12, steps=2)
    if p < 0.96:
        return dict(path="hybrid", mesh="cavity", n=_log(rng, 12, 128), jitter=0.0, K=K, precision="fp64", Re=200.0,
                    integ=rng.choice([2, 4]), adv=2, tol=1e-12, steps=rng.randint(2, 5))
    return dict(path="adjoint", mesh="cavity", n=_log(rng, 12, 40), jitter=0.0, K=K, precision="fp64", Re=1000.0,
                integ=4, adv=1, tol=1e-13, steps=2)


# ---- meshes, time steps and inputs -------------------------------------------------------------
@functools.lru_cache(maxsize=8)
def _mesh(kind, n, jitter):
    if kind == "cavity":
        return meshes.cavity(n, 2, jitter=jitter, seed=7 if jitter else None)
    if kind == "bfs":
        return meshes.backward_facing_step(n, n // 6, 2, jitter=jitter, seed=2)
    return meshes.cylinder_ogrid(n, 2 * n, 3)


def _sizes(case):
    return [int(s) for s in case["sizes"].split(",")]


def _ensemble_params(case):
    """Re and dt of the instances: Re log-spaced over [100, 3200] by position."""
    ns = _sizes(case)
    re = [100.0 * 32.0 ** (i / max(1, len(ns) - 1)) for i in range(len(ns))]
    return ns, re, [_dt(n, case["K"], r, case["integ"]) for n, r in zip(ns, re)]


def _dt(n, K, Re, integ):
    """Half the explicit diffusion limit of an n x n unit cavity, capped by an advective bound."""
    return min(0.5 * REAL_LIMIT[integ] / (RHO[K] * n * n / Re), 0.05 / n)


def _case_dt(case):
    if case["mesh"] == "bfs":
        return 5e-4 * (384.0 / case["n"]) ** 2 * min(1.0, RHO[5] / RHO[case["K"]])
    if case["mesh"] == "cylinder":
        return 5e-7 * (256.0 / case["n"]) ** 2
    return _dt(case["n"], case["K"], case["Re"], case["integ"])


def _field(xy, seed, amp=1.0):
    """A smooth random field: eight plane waves of random direction, wavelength and phase."""
    rng = np.random.default_rng(seed)
    k, ph, a = rng.standard_normal((8, 2)) * 8.0, rng.uniform(0.0, 2 * np.pi, 8), rng.standard_normal(8)
    x = torch.as_tensor(xy, device="cuda" if torch.cuda.is_available() else "cpu")
    w = torch.zeros(x.shape[0], dtype=torch.float64, device=x.device)
    for i in range(8):
        w += (amp * a[i]) * torch.cos(x[:, 0] * k[i, 0] + x[:, 1] * k[i, 1] + ph[i])
    return w


def _handle(case):
    prec = hoc.HOC_MIXED if case.get("precision") == "mixed" else hoc.HOC_FP64
    kw = dict(K=case["K"], precision=prec, tol=case.get("tol", 1e-12), maxiter=500,
              time_integration_type=case.get("integ", 4), advection_type=case.get("adv", 1))
    if case["path"] == "ensemble":
        ns, re, dts = _ensemble_params(case)
        m, off = meshes.concat([_mesh("cavity", n, 0.0) for n in ns])
        g = hoc.HO2D(problem_type=1, Re=re[0], dt=dts[0], **kw)
        g.load_mesh(m)
        g.set_instances(off, re, dts)
        g.setup()
        return g
    m = _mesh(case["mesh"], case["n"], case["jitter"])
    if case["path"] in ("laplacian", "poisson"):
        g = hoc.HO2D(problem_type=1, Re=100.0, dt=1e-4, **kw)
    elif case["path"] == "hybrid":
        names = ["wall", "open"]
        ids = np.array([1 if nm == "top" else 0 for nm in m.bnames], dtype=np.int32)[m.bedge_bdry]
        m = meshes.QuadMesh(m.lnod, m.xy, m.elem, m.bedges, ids, names)
        g = hoc.HO2D(problem_type=11, Re=case["Re"], dt=1.0, **kw)
    else:
        g = hoc.HO2D(problem_type={"cavity": 1, "bfs": 2, "cylinder": 3}[case["mesh"]], Re=case["Re"],
                     dt=_case_dt(case), **kw)
    g.load_mesh(m)
    g.setup()
    return g


def prepare(case, seed):
    g = _handle(case)
    xy = g.solution_points()
    path = case["path"]
    s = {"g": g, "path": path}
    if path == "laplacian":
        s["x"] = _field(xy, seed)
        s["y"] = torch.empty_like(s["x"])
        s["stream"] = torch.cuda.Stream()
        return s
    if path == "ensemble":  # another field per instance
        K2 = case["K"] ** 2
        parts, e0 = [], 0
        for i, n in enumerate(_sizes(case)):
            parts.append(_field(xy[e0 * K2:(e0 + n * n) * K2], seed * 131 + i).cpu().numpy())
            e0 += n * n
        s["w0"] = np.concatenate(parts)
    elif case["mesh"] == "cylinder":
        s["w0"] = np.random.default_rng(seed).uniform(-1e-3, 1e-3, g.D)
    else:
        s["w0"] = _field(xy, seed).cpu().numpy()
    s["steps"] = case.get("steps", 1)
    s["t0"] = 20.0 / 3.0 if case["mesh"] in ("bfs", "cylinder") else 0.0
    if path == "poisson":
        s["zero"] = np.zeros(g.D)
    if path == "hybrid":
        s["outer"] = (_dt(case["n"], case["K"], case["Re"], case["integ"]) * s["steps"], s["steps"], case["integ"], case["Re"])
        op = g.open_points()
        g.set_p2g_weights(np.where(xy[:, 1] > 0.8, 0.3, 0.0))
        s["ends"] = []
        for k in range(2):
            f = _field(op, seed * 17 + k, 0.1).cpu().numpy()
            s["ends"].append((np.stack([np.sin(np.pi * op[:, 0]) * (1.0 + 0.1 * k) + f, 0.05 * op[:, 0]], 1), f,
                              _field(xy, seed * 19 + k).cpu().numpy()))
    if path == "adjoint":
        s["areas"] = g.solution_areas()
    return s


def run(s):
    g, path = s["g"], s["path"]
    if path == "laplacian":
        g.apply_laplacian_device(s["x"].data_ptr(), s["y"].data_ptr(), s["stream"].cuda_stream)
        return s["y"]
    if path == "poisson":
        g.set_streamfunction(s["zero"])
        return g.poisson(s["w0"])
    g.set_vorticity(s["w0"])
    if path == "hybrid":
        for uv, w, target in s["ends"]:  # values at the start and at the end of the outer step
            g.set_open_velocities(uv)
            g.set_open_vorticity(w)
            g.set_vorticity_target(target)
        g.solveto(*s["outer"])
        return {"w": g.get_vorticity(), "psi": g.get_streamfunction()}
    g.set_time(s["t0"])
    if path == "adjoint":
        g.adjoint_forward(s["steps"], 0)
        w = g.get_vorticity()
        gw, gp = g.adjoint_backward(s["areas"] * w)
        return {"w": w, "grad_w0": gw, "grad_wall": gp}
    g.step(s["steps"])
    return {"w": g.get_vorticity(), "psi": g.get_streamfunction()}


def work(case):
    """Inputs read once, outputs written once, and the operations of the least arithmetic that
    takes one to the other: per stage one solve (as one operator application), the velocity, the
    diffusion and the advection of every element, at 4 K^3 fused operations per 2-D derivative pair."""
    K = case["K"]
    if case["path"] == "ensemble":
        N = sum(n * n for n in _sizes(case))
    elif case["mesh"] == "bfs":
        N = case["n"] * (case["n"] // 6) - round(case["n"] / 6) * (case["n"] // 6 // 2)
    elif case["mesh"] == "cylinder":
        N = 2 * case["n"] ** 2
    else:
        N = case["n"] ** 2
    D = N * K * K
    op = 16.0 * K ** 3 * N  # derivative pair and divergence pair, multiply and add
    if case["path"] in ("laplacian", "poisson"):
        return {"bytes": 16.0 * D, "flops": op}
    stages = case["steps"] * case["integ"]  # integ 1, 2, 4: that many stages
    # a stage reads its vorticity and writes the next; a step's state passes through memory
    bytes_ = stages * 16.0 * D
    flops = stages * 3.0 * op
    if case["path"] == "adjoint":  # forward, and the transpose of each stage
        bytes_, flops = 3.0 * bytes_, 3.0 * flops
    return {"bytes": bytes_, "flops": flops}


# ---- the discretisation on a uniform cavity, in plain torch ------------------------------------
def _tables(K):
    x, w = np.polynomial.legendre.leggauss(K)
    P = np.polynomial.legendre.Legendre.basis
    one = np.ones(1)
    basis, lv, ld, D = [], np.zeros((K, 2)), np.zeros((K, 2)), np.zeros((K, K))
    for m in range(K):
        others = np.delete(x, m)
        p = np.polynomial.Polynomial.fromroots(others) / np.prod(x[m] - others)
        lv[m] = p(-1.0), p(1.0)
        ld[m] = p.deriv()(-1.0), p.deriv()(1.0)
        D[m] = p.deriv()(x)  # D[m, k] = l_m'(x_k)
        basis.append(p)
    gl = ((-1) ** K * 0.5) * (P(K) - P(K - 1))  # the left Radau correction, 1 at -1 and 0 at +1
    gv = np.stack([gl(x), gl(-x)], 1)
    gd = np.stack([gl.deriv()(x), -gl.deriv()(-x)], 1)
    assert abs(gl(-one)[0] - 1) < 1e-12
    gp = np.array([-0.5 * K * (K + 1), 0.5 * K * (K + 1)])  # the interface coefficient of the scheme
    t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=_dev())  # noqa: E731
    return dict(x=t(x), w=t(w), lv=t(lv), ld=t(ld), D=t(D), gv=t(gv), gd=t(gd), gp=gp)


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


class _Uniform:
    """n x n cells of the unit square, K points per direction: fields [row, j, column, i]."""

    def __init__(self, n, K, Re, dt, adv):
        self.n, self.K, self.Re, self.dt, self.adv = n, K, Re, dt, adv
        self.T = _tables(K)
        self.h = 1.0 / n
        self.J = self.h * self.h / 4
        self.vecs = None

    def shape(self, flat):
        n, K = self.n, self.K
        return torch.as_tensor(flat, dtype=torch.float64, device=_dev()).reshape(n, n, K, K).permute(0, 2, 1, 3)

    def flat(self, u):
        return u.permute(0, 2, 1, 3).reshape(-1)

    # one direction at a time: lines [..., cell, point]
    def _flux(self, u, wall, wall_kind):
        """Corrected gradient at the points, common values and common fluxes at the ends of the
        cells of every line; wall = (lower, upper) values, kind 'value' or 'flux'."""
        T, gp = self.T, self.T["gp"]
        v = u @ T["lv"]
        g = u @ T["ld"]
        cv, F = torch.empty_like(v), torch.empty_like(v)
        mid = 0.5 * (v[..., :-1, 1] + v[..., 1:, 0])
        cv[..., :-1, 1], cv[..., 1:, 0] = mid, mid
        F[..., :-1, 1] = g[..., :-1, 1] + (mid - v[..., :-1, 1]) * gp[1]
        F[..., 1:, 0] = g[..., 1:, 0] + (mid - v[..., 1:, 0]) * gp[0]
        avg = 0.5 * (F[..., :-1, 1] + F[..., 1:, 0])
        F[..., :-1, 1], F[..., 1:, 0] = avg, avg
        for c, b in ((0, 0), (self.n - 1, 1)):
            if wall_kind == "value":
                cv[..., c, b] = wall[b]
                F[..., c, b] = g[..., c, b] + (cv[..., c, b] - v[..., c, b]) * gp[b]
            else:
                F[..., c, b] = wall[b]
                cv[..., c, b] = v[..., c, b] + (F[..., c, b] - g[..., c, b]) / gp[b]
        grad = u @ T["D"] + (cv - v) @ T["gd"].T
        return grad, cv, F

    def _second(self, u, wall, kind):
        grad, cv, F = self._flux(u, wall, kind)
        return grad @ self.T["D"] + (F - grad @ self.T["lv"]) @ self.T["gd"].T, cv

    def _xy(self, f, u):
        """f on the x lines and on the y lines of u; results back in the field's layout."""
        fx = f(u, 0)
        fy = f(u.permute(2, 3, 0, 1), 1)
        return fx, tuple(r.permute(2, 3, 0, 1) for r in fy)

    def laplacian(self, u):
        zero = (0.0, 0.0)
        fx, fy = self._xy(lambda v, d: (self._second(v, zero, "value")[0],), u)
        return fx[0] + fy[0]

    def poisson(self, w):
        """psi of -laplacian = w with psi = 0 on the walls (the operator is the sum over both
        directions of one line operator, symmetric under the quadrature weights)."""
        n, K = self.n, self.K
        if self.vecs is None:
            eye = torch.eye(n * K, dtype=torch.float64, device=_dev()).reshape(n * K, n, K)
            M = self._second(eye, (0.0, 0.0), "value")[0].reshape(n * K, n * K).T
            s = self.T["w"].sqrt().repeat(n)
            A = (s[:, None] * M / s[None, :]).cpu()
            lam, Q = torch.linalg.eigh(0.5 * (A + A.T))
            self.vecs = (lam.to(_dev()), Q.to(_dev()) / s.cpu().to(_dev())[:, None], Q.to(_dev()) * s[:, None])
        lam, R, L = self.vecs
        b = (-self.J * w).reshape(n * K, n * K)
        solve = lambda r: R @ ((L.T @ r @ L) / (lam[:, None] + lam[None, :])) @ R.T  # noqa: E731
        psi = solve(b)
        r = b - self.laplacian(psi.reshape(n, K, n, K)).reshape(n * K, n * K)
        return (psi + solve(r)).reshape(n, K, n, K)

    def stage(self, w):
        """(k, psi, wall values): k = dt (advection + diffusion) of one Runge-Kutta stage."""
        T, n = self.T, self.n
        psi = self.poisson(w)
        # velocity: corrected gradient of psi, its flux corrected by the common fluxes
        def velocity(v, d):
            grad, _, F = self._flux(v, (0.0, 0.0), "value")
            return grad + (F - grad @ T["lv"]) @ T["gv"].T, F
        (px, Fx), (py, Fy) = velocity(psi, 0), velocity(psi.permute(2, 3, 0, 1), 1)
        py = py.permute(2, 3, 0, 1)
        hh = self.h / 2
        U1, U2 = py, -px                    # contravariant fluxes: hh u = dpsi/d(eta), -hh v = dpsi/d(xi)
        # wall vorticity flux: (slip + wall speed) Re / dt; the lid moves at -1 in its tangent
        q = self.Re / self.dt
        wx = (hh * q * (Fx[..., 0, 0] / hh), hh * q * (Fx[..., n - 1, 1] / hh))
        wy = (hh * q * (Fy[..., 0, 0] / hh), hh * q * (Fy[..., n - 1, 1] / hh - 1.0))
        dx, cx = self._second(w, wx, "flux")
        dy, cy = self._second(w.permute(2, 3, 0, 1), wy, "flux")
        diff = dx + dy.permute(2, 3, 0, 1)
        ax = self._advect(w, U1)
        ay = self._advect(w.permute(2, 3, 0, 1), U2.permute(2, 3, 0, 1)).permute(2, 3, 0, 1)
        return self.dt * (ax + ay + diff / self.Re) / self.J, psi

    def _advect(self, w, U):
        """-d(U w) on lines: upwind fluxes at the cell ends, no flux through the walls."""
        T = self.T
        wv, uv = w @ T["lv"], U @ T["lv"]
        f = torch.zeros_like(wv)
        if self.adv == 1:
            fl, fr = (uv * wv)[..., :-1, 1], (uv * wv)[..., 1:, 0]
            dw = wv[..., :-1, 1] - wv[..., 1:, 0]
            # |a| dw with a = (fl - fr) / dw, switched on where the jump is above 1e-4
            up = 0.5 * (fl + fr) + torch.where(dw.abs() > 1e-4, 0.5 * (fl - fr).abs() * dw.sign(), torch.zeros_like(dw))
        else:
            c = 0.5 * (uv[..., :-1, 1] + uv[..., 1:, 0])
            up = torch.where(c > 0, c * wv[..., :-1, 1], c * wv[..., 1:, 0])
            cu = torch.zeros_like(uv)
            cu[..., :-1, 1], cu[..., 1:, 0] = c, c
            U = U + (cu - uv) @ T["gv"].T
        f[..., :-1, 1], f[..., 1:, 0] = up, up
        F = U * w
        return -(F @ T["D"] + (f - F @ T["lv"]) @ T["gd"].T)

    def step(self, w, integ):
        k1, psi = self.stage(w)
        if integ == 1:
            return w + k1, psi
        if integ == 2:
            k2, psi = self.stage(w + k1)
            return w + 0.5 * (k1 + k2), psi
        k2, _ = self.stage(w + 0.5 * k1)
        k3, _ = self.stage(w + 0.5 * k2)
        k4, psi = self.stage(w + k3)
        return w + (k1 + 2 * k2 + 2 * k3 + k4) / 6, psi


def _points(n, K):
    x = np.polynomial.legendre.leggauss(K)[0]
    p = ((np.arange(n)[:, None] + 0.5 * (1 + x)[None, :]) / n)
    xx = np.broadcast_to(p[None, :, None, :], (n, n, K, K))
    yy = np.broadcast_to(p[:, None, :, None], (n, n, K, K))
    return np.stack([xx.ravel(), yy.ravel()], 1)


def exact(case, seed):
    path = case["path"]
    if case["mesh"] != "cavity" or case.get("jitter", 0.0) or path in ("hybrid", "adjoint"):
        return None  # no closed form of the operator on these meshes; the gradient has none
    K = case["K"]
    if path == "ensemble":
        ws, psis = [], []
        for i, (n, re, dt) in enumerate(zip(*_ensemble_params(case))):
            m = _Uniform(n, K, re, dt, case["adv"])
            w = m.shape(_field(_points(n, K), seed * 131 + i))
            for _ in range(case["steps"]):
                w, psi = m.step(w, case["integ"])
            ws.append(m.flat(w))
            psis.append(m.flat(psi))
        return {"w": torch.cat(ws).cpu().numpy(), "psi": torch.cat(psis).cpu().numpy()}
    n = case["n"]
    if path != "laplacian" and n * K > 2600:
        return None  # the dense eigenvectors take too long
    f = _field(_points(n, K), seed)
    if path == "laplacian":
        m = _Uniform(n, K, 100.0, 1e-4, 1)
        return m.flat(m.laplacian(m.shape(f)))
    if path == "poisson":
        m = _Uniform(n, K, 100.0, 1e-4, 1)
        return m.flat(m.poisson(m.shape(f))).cpu().numpy()
    m = _Uniform(n, K, case["Re"], _case_dt(case), case["adv"])
    w = m.shape(f)
    for _ in range(case["steps"]):
        w, psi = m.step(w, case["integ"])
    return {"w": m.flat(w).cpu().numpy(), "psi": m.flat(psi).cpu().numpy()}
