"""The work that programs have this framework do, as cases that can be timed.

`listed()` holds the sizes that the repository's own benchmark and tests use
(the 256 x 256 Rayleigh-Benard step above all), next to the smallest, ragged and
batched forms of the same calls; `draw` gives further cases of the same ranges.
Every case goes through the public entry points: the drop-in `NavierStokes`
and `NavierStokesAdjoint`, the batches (`RBCBatch`, `HeteroBatch`), the
differentiable trajectory, the bases' transforms, the solver plans and the
field operations.  Everything is 64-bit floating point, the only type the
framework has.
"""
import functools
import math

import numpy as np
import torch

F64 = torch.float64


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest production run: a 64 x 64 box, where launches and their
        # latency are all there is
        dict(name="step_64", kind="step", n0=64, n1=64, case="rbc", integrator="eu", beta=1.0,
             ra=1e5, dt=0.01, steps=20),
        # the headline: one 256 x 256 box at Ra = 1e8
        dict(name="step_256", kind="step", n0=256, n1=256, case="rbc", integrator="eu", beta=1.0,
             ra=1e8, dt=1e-3, steps=20),
        # one large box
        dict(name="step_512", kind="step", n0=512, n1=512, case="rbc", integrator="eu", beta=1.0,
             ra=1e8, dt=1e-3, steps=10),
        # odd and unequal lengths (an odd dealiased grid has no mirror folds),
        # isothermal sidewalls
        dict(name="step_129x101", kind="step", n0=129, n1=101, case="linear", integrator="eu",
             beta=1.0, ra=1e6, dt=2e-3, steps=20),
        # the three-stage scheme with half of the diffusion explicit, a wide
        # box with the sidewall profile
        dict(name="rk3_128x96", kind="step", n0=128, n1=96, case="zero", integrator="rk3",
             beta=0.5, ra=1e6, dt=2e-3, steps=10),
        # a parameter study: 64 boxes of one shape advanced together
        dict(name="batch_64x256", kind="batch", n0=256, n1=256, count=64, ra=1e8, dt=1e-3,
             steps=4),
        # a parameter study over resolutions: 64 boxes of 16 shapes, one launch
        # per operator for all of them
        dict(name="mixed_64", kind="mixed", sizes="64,96,128,192", count=64, steps=4),
        # the gradient of a trajectory's mean Nusselt number with respect to
        # its initial temperature, forward and backward
        dict(name="gradient_128", kind="gradient", n0=128, n1=128, ra=1e6, dt=2e-3, steps=20),
        # steady-state search by adjoint descent
        dict(name="descent_128", kind="descent", n0=128, n1=128, ra=1e5, dt=2e-4, steps=4),
        # transforms of many fields there and back (post-processing, data sets)
        dict(name="transform_512x256", kind="transform", n0=256, n1=256, count=512),
        # Helmholtz and Poisson plans on many fields: right-hand sides, banded
        # solves and projections
        dict(name="solve_512x256", kind="solve", n0=256, n1=256, count=512, lam=0.01),
        # a program that works on one small field at a time, op by op
        dict(name="field_96x80", kind="field", n0=96, n1=80),
    ]


def _size(rng, lo, hi):
    """A length spread over the logarithm of [lo, hi], odd ones among them."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.4:
        n += n % 2
    return min(max(n, lo), hi)


def _pair(rng, lo, hi):
    a, b = _size(rng, lo, hi), _size(rng, lo, hi)
    return (a, a) if rng.random() < 0.4 else (a, b)


def draw(rng):
    kind = rng.choice(["step", "step", "step", "batch", "mixed", "gradient", "descent",
                       "transform", "solve", "field"])
    c = dict(kind=kind)
    if kind == "step":
        c["n0"], c["n1"] = _pair(rng, 48, 400)
        c["case"] = rng.choice(["rbc", "rbc", "linear", "zero"])
        c["integrator"], c["beta"] = rng.choice([("eu", 1.0), ("eu", 1.0), ("eu", 0.5),
                                                 ("rk3", 1.0), ("rk3", 0.5)])
        # the three-stage scheme and explicit diffusion run fused on even
        # dealiased lengths
        if c["integrator"] == "rk3" or c["beta"] != 1.0:
            c["n0"], c["n1"] = c["n0"] // 4 * 4, c["n1"] // 4 * 4
        c["ra"], c["dt"] = rng.choice([(1e5, 5e-3), (1e6, 2e-3), (1e8, 1e-3)])
        c["steps"] = rng.choice([7, 10, 13, 20])
    elif kind == "batch":
        c["n0"], c["n1"] = _pair(rng, 48, 256)
        area = c["n0"] * c["n1"]
        c["count"] = max(2, min(64, int(rng.uniform(0.1, 1.0) * 64 * 65536 / area)))
        c["ra"], c["dt"], c["steps"] = 1e7, 1e-3, rng.choice([2, 3, 4])
    elif kind == "mixed":
        c["sizes"] = ",".join(str(n) for n in sorted({2 * _size(rng, 32, 96) // 4 * 4
                                                      for _ in range(3)}))
        c["count"], c["steps"] = rng.randrange(9, 49), rng.choice([2, 3, 4])
    elif kind == "gradient":
        c["n0"], c["n1"] = _pair(rng, 48, 160)
        c["ra"], c["dt"], c["steps"] = 1e6, 2e-3, rng.choice([5, 10, 15])
    elif kind == "descent":
        c["n0"], c["n1"] = _pair(rng, 48, 160)
        c["ra"], c["dt"], c["steps"] = 1e5, 2e-4, rng.choice([2, 3])
    elif kind in ("transform", "solve"):
        c["n0"], c["n1"] = _pair(rng, 48, 400)
        most = 512 * 65536 // max(c["n0"] * c["n1"], 1)
        c["count"] = max(1, min(4096, int(math.exp(rng.uniform(0.0, math.log(most))))))
        if kind == "solve":
            c["lam"] = 10.0 ** rng.uniform(-4, -1)
    else:
        c["n0"], c["n1"] = _pair(rng, 48, 160)
    return c


def _mixed_specs(case, seed):
    """Shapes in turn over all pairs of sizes; Ra spread over 1e5 ... 1e8."""
    sizes = [int(s) for s in case["sizes"].split(",")]
    shapes = [(a, b) for a in sizes for b in sizes]
    rng = np.random.default_rng([seed, 5])
    specs = []
    for i in range(case["count"]):
        ra = 10.0 ** rng.uniform(5.0, 8.0)
        specs.append(dict(shape=shapes[i % len(shapes)], ra=ra, pr=1.0,
                          dt=float(np.clip(0.01 * math.sqrt(1e5 / ra), 1e-3, 1e-2))))
    return specs


def _batch_params(case, seed):
    rng = np.random.default_rng([seed, 6])
    return [dict(ra=case["ra"] * 10.0 ** rng.uniform(-1.0, 0.0), pr=float(rng.uniform(0.7, 2.0)),
                 dt=case["dt"]) for _ in range(case["count"])]


# ---------------------------------------------------------------------------
# inputs: smooth spectral fields, coefficients that fall off with the mode
# number like those of a developed flow
# ---------------------------------------------------------------------------
def _noise(seed, tag, shape):
    g = torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1) + tag)
    return torch.randn(shape, generator=g, dtype=F64, device="cuda")


def _coefs(seed, tag, shape, amplitude):
    x = _noise(seed, tag, shape)
    for ax in (-2, -1):
        n = shape[ax]
        k = torch.arange(n, dtype=F64, device="cuda")
        w = torch.exp(-12.0 * k / n) / (1.0 + 0.3 * k)
        x = x * (w[:, None] if ax == -2 else w)
    return amplitude * x


@functools.lru_cache(maxsize=64)
def _wall_modes(n):
    """Dirichlet coefficients [n-2, K] of (1 - x^2)^2 T_k(x) and of their
    derivatives, k < K."""
    cheb = np.polynomial.chebyshev
    K = n // 4
    A, D = np.zeros((n, K)), np.zeros((n, K))
    for k in range(K):
        t = np.zeros(k + 1)
        t[k] = 1.0
        c = cheb.chebmul(cheb.chebmul([0.5, 0.0, -0.5], [0.5, 0.0, -0.5]), t)
        d = cheb.chebder(c)
        A[:len(c), k], D[:len(d), k] = c, d
    P = np.linalg.pinv(_stencil(n, "CD"))
    return _t(P @ A), _t(P @ D)


def _state(seed, tag, lead, n0, n1):
    """(X [*lead, 3, n0-2, n1-2], pres [*lead, n0, n1]): coefficients of a flow in
    a box with walls (the velocities of a random stream function, so free of
    divergence), its temperature and its pressure."""
    X = _coefs(seed, 10 * tag + 1, tuple(lead) + (3, n0 - 2, n1 - 2), 0.2)
    pres = _coefs(seed, 10 * tag + 2, tuple(lead) + (n0, n1), 0.01)
    (ax, dx), (ay, dy) = _wall_modes(n0), _wall_modes(n1)
    kx = torch.arange(ax.shape[1], dtype=F64, device="cuda")
    ky = torch.arange(ay.shape[1], dtype=F64, device="cuda")
    psi = _noise(seed, 10 * tag + 3, tuple(lead) + (ax.shape[1], ay.shape[1]))
    psi = 0.2 * psi / ((1.0 + kx[:, None]) ** 2 * (1.0 + ky) ** 2)
    X[..., 0, :, :] = _y(dy, _x(ax, psi))
    X[..., 1, :, :] = -_y(ay, _x(dx, psi))
    return X, pres


def _ns_kwargs(case):
    return dict(shape=(case["n0"], case["n1"]), ra=case["ra"], pr=1.0, dt=case["dt"], tsave=None,
                dealias=True, integrator=case.get("integrator", "eu"),
                beta=case.get("beta", 1.0), aspect=1.0)


def prepare(case, seed):
    import pypde_amd as pypde
    kind = case["kind"]
    st = dict(case)
    if kind == "step":
        from pypde_amd.navier import NavierStokes
        ns = NavierStokes(case=case["case"], **_ns_kwargs(case))
        st["X"], st["pres"] = _state(seed, 1, (), case["n0"], case["n1"])
        ns.set_state(U=st["X"][0], V=st["X"][1], T=st["X"][2], pres=st["pres"])
        ns.prepare_graphs()
        st["ns"] = ns
    elif kind == "batch":
        from pypde_amd.engine import RBCBatch
        eng = RBCBatch((case["n0"], case["n1"]), _batch_params(case, seed), case="rbc")
        st["X"], st["pres"] = _state(seed, 2, (case["count"],), case["n0"], case["n1"])
        eng.capture(1)
        st["eng"] = eng
    elif kind == "mixed":
        from pypde_amd.batch import HeteroBatch
        hb = HeteroBatch(_mixed_specs(case, seed), case="rbc", persistent=True)
        st["init"] = [_state(seed, 100 + c, (e.B,), *hb.shapes[c])
                      for c, e in enumerate(hb.classes)]
        hb.capture(1)
        st["hb"] = hb
    elif kind == "gradient":
        from pypde_amd.adjoint import Trajectory
        from pypde_amd.engine import RBCBatch
        eng = RBCBatch((case["n0"], case["n1"]), [dict(ra=case["ra"], pr=1.0, dt=case["dt"])],
                       case="rbc")
        st["X"], st["pres"] = _state(seed, 3, (1,), case["n0"], case["n1"])
        st["traj"] = Trajectory(eng)
    elif kind == "descent":
        from pypde_amd.navier import NavierStokesAdjoint
        st["X"], st["pres"] = _state(seed, 4, (), case["n0"], case["n1"])
        st["zero"] = torch.zeros_like(st["pres"])
        ns = NavierStokesAdjoint(case="rbc", **_ns_kwargs(case))
        for _ in range(3):   # op by op, the capture, one replay
            _descent_set(ns, st)
            ns.update()
        st["ns"] = ns
    elif kind == "transform":
        st["x"] = pypde.Base(case["n0"], "CH")
        st["y"] = pypde.Base(case["n1"], "CH")
        st["c"] = _coefs(seed, 51, (case["count"], case["n0"], case["n1"]), 1.0)
    elif kind == "solve":
        bx, by = pypde.Base(case["n0"], "CD"), pypde.Base(case["n1"], "CD")
        st["bx"], st["by"] = bx, by
        st["hh"] = pypde.solverplan_hholtz2d_adi([bx, by], case["lam"])
        st["po"] = pypde.solverplan_poisson2d([bx, by], singular=False)
        st["f"] = _coefs(seed, 61, (case["count"], case["n0"], case["n1"]), 1.0)
    elif kind == "field":
        n0, n1 = case["n0"], case["n1"]
        st["v"] = pypde.Field([pypde.Base(n0, "CD", dealias=1.5), pypde.Base(n1, "CD", dealias=1.5)])
        st["w"] = pypde.Field([pypde.Base(n0, "CH", dealias=1.5), pypde.Base(n1, "CH", dealias=1.5)])
        st["hh"] = pypde.solverplan_hholtz2d_adi(st["v"].xs, 0.02)
        st["po"] = pypde.solverplan_poisson2d(st["v"].xs, singular=False)
        st["vhat"] = _coefs(seed, 71, (n0 - 2, n1 - 2), 0.3)
    else:
        raise ValueError("unknown kind %r" % kind)
    return st


def _descent_set(ns, st):
    """The iteration's state: fields, pressure and the inner step's pressure."""
    for f, v in ((ns.U, st["X"][0]), (ns.V, st["X"][1]), (ns.T, st["X"][2]),
                 (ns.pres, st["pres"])):
        f.vhat.copy_(v)
    ns.NS.set_state(pres=st["zero"])


def run(st):
    kind = st["kind"]
    if kind == "step":
        ns = st["ns"]
        ns.set_state(U=st["X"][0], V=st["X"][1], T=st["X"][2], pres=st["pres"])
        ns.update_many(st["steps"])
        return [ns.U.vhat, ns.V.vhat, ns.T.vhat, ns.pres.vhat]
    if kind == "batch":
        eng = st["eng"]
        eng.X.copy_(st["X"])
        eng.pres.copy_(st["pres"])
        eng.step(st["steps"])
        return [eng.X, eng.pres]
    if kind == "mixed":
        hb = st["hb"]
        for e, (X, pres) in zip(hb.classes, st["init"]):
            e.X.copy_(X)
            e.pres.copy_(pres)
        hb.step(st["steps"])
        return [t for e in hb.classes for t in (e.X, e.pres)]
    if kind == "gradient":
        from pypde_amd.adjoint import TimeAveragedNusselt
        T0 = st["X"][:, 2].clone().requires_grad_(True)
        J = TimeAveragedNusselt.apply(T0, st["traj"], st["X"], st["pres"], st["steps"])
        J.sum().backward()
        return [J.detach(), T0.grad]
    if kind == "descent":
        ns = st["ns"]
        _descent_set(ns, st)
        for _ in range(st["steps"]):
            ns.update()
        return [ns.U.vhat, ns.V.vhat, ns.T.vhat, ns.pres.vhat]
    if kind == "transform":
        v = st["y"].backward_fft(st["x"].backward_fft(st["c"], axis=0), axis=1)
        return [v, st["y"].forward_fft(st["x"].forward_fft(v, axis=0), axis=1)]
    if kind == "solve":
        f, hh, po = st["f"], st["hh"], st["po"]
        old = st["by"].from_chebyshev(st["bx"].from_chebyshev(f, axis=0), axis=1)
        u = hh.solve_lhs(hh.solve_rhs(f) + hh.solve_old(old))
        return [old, u, po.solve_lhs(po.solve_rhs(f))]
    if kind == "field":
        import pypde_amd as pypde
        v, w = st["v"], st["w"]
        v.vhat = st["vhat"]
        v.backward()
        dx = pypde.grad(v, (1, 0))
        ux = v.dealias.backward(v.vhat)
        conv = pypde.convective_term(v, ux, ux, deriv_field=w, dealias=True)
        u = st["hh"].solve_lhs(st["hh"].solve_rhs(conv) + st["hh"].solve_old(v.vhat))
        p = st["po"].solve_lhs(st["po"].solve_rhs(dx))
        return [v.v, v.forward(v.v), dx, conv, u, p]
    raise ValueError(kind)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _step_work(n0, n1, stages=1, diffusion=False):
    """One time step of one box: the state read and written once; the dense
    operators with half of their terms (every one of them maps even and odd
    modes separately or is mirror-symmetric), eight dealiased fields from the
    three of the state, three products, and the velocity correction and Poisson
    mixing.  Banded operators are left out of the operation count."""
    m0, m1, l0, l1 = n0 - 2, n1 - 2, n0 * 3 // 2, n1 * 3 // 2
    fl = 2 * 3 * l0 * m1 * m0            # three fields, values and x-derivatives: 6 products / 2
    fl += 8 * l0 * l1 * m1               # eight fields along y
    fl += 3 * l0 * m1 * l1 + 3 * m0 * m1 * l0        # forward, y then x
    fl += 2 * m0 * m1 * m1               # Poisson mixing there and back
    fl += 2 * m0 * m0 * m1 + 2 * m0 * m1 * m1        # velocity projections
    by = 8 * 2 * (3 * m0 * m1 + n0 * n1)
    return stages * fl, stages * by


def work(case):
    kind = case["kind"]
    if kind in ("step", "batch", "gradient", "descent", "transform", "solve", "field"):
        n0, n1 = case["n0"], case["n1"]
        m0, m1, l0, l1 = n0 - 2, n1 - 2, n0 * 3 // 2, n1 * 3 // 2
    if kind in ("step", "batch"):
        fl, by = _step_work(n0, n1, 3 if case.get("integrator") == "rk3" else 1)
        n = case["steps"] * case.get("count", 1)
        return dict(bytes=float(n * by), flops=float(n * fl))
    if kind == "mixed":
        fl = by = 0
        for s in _mixed_specs(case, 0):
            f, b = _step_work(*s["shape"])
            fl, by = fl + f, by + b
        return dict(bytes=float(case["steps"] * by), flops=float(case["steps"] * fl))
    if kind == "gradient":
        # the value, the states again for the backward sweep, and the reverse
        # step (the dealiased fields again and the transposed operators)
        fl, by = _step_work(n0, n1)
        return dict(bytes=float(4.0 * case["steps"] * by), flops=float(4.0 * case["steps"] * fl))
    if kind == "descent":
        # the inner step, three Poisson smoothings, and dealiased products of
        # the adjoint fields (16 backward, 3 forward transforms), the projection
        fl, by = _step_work(n0, n1)
        fl += 3 * 2 * m0 * m1 * m1 + 19 * (l0 * m0 * m1 + l0 * l1 * m1) + 2 * m0 * m1 * (m0 + m1)
        return dict(bytes=float(2 * case["steps"] * by), flops=float(case["steps"] * fl))
    if kind == "transform":
        b = case["count"]
        return dict(bytes=float(3 * 8 * b * n0 * n1), flops=float(2.0 * b * n0 * n1 * (n0 + n1)))
    if kind == "solve":
        b = case["count"]
        return dict(bytes=float(8 * b * (n0 * n1 + 3 * m0 * m1)),
                    flops=float(b * m0 * m1 * (2.0 * m1 + 120)))
    fl = l0 * m0 * m1 * 3 + l0 * l1 * m1 * 3 + l0 * n1 * l1 + n0 * n1 * l0
    fl += 2 * n0 * n1 * (m0 + m1) + 2 * m0 * m1 * m1
    return dict(bytes=float(8 * (6 * n0 * n1 + m0 * m1)), flops=float(fl))


# ---------------------------------------------------------------------------
# the same results in plain 64-bit torch / numpy: dense operators throughout
# ---------------------------------------------------------------------------
def _grid(n):
    return -np.cos(np.pi * np.arange(n) / (n - 1))


def _to_values(L, N):
    """Values at L Gauss-Lobatto points (increasing) of N Chebyshev modes."""
    j, k = np.arange(L)[:, None], np.arange(N)[None, :]
    return (-1.0) ** k * np.cos(np.pi * ((j * k) % (2 * (L - 1))) / (L - 1))


def _to_coefs(N, L):
    """The first N Chebyshev modes of L samples."""
    j, k = np.arange(L)[None, :], np.arange(N)[:, None]
    c = (-1.0) ** k * np.cos(np.pi * ((j * k) % (2 * (L - 1))) / (L - 1)) * 2.0 / (L - 1)
    c[:, 0] *= 0.5
    c[:, -1] *= 0.5
    c[0] *= 0.5
    if N == L:
        c[-1] *= 0.5
    return c


def _diff(N):
    D = np.zeros((N, N))
    for n in range(N):
        D[n, n + 1::2] = 2.0 * np.arange(n + 1, N, 2)
    D[0] *= 0.5
    return D


def _stencil(N, key):
    S = np.zeros((N, N - 2))
    k = np.arange(N - 2)
    S[k, k] = 1.0
    S[k + 2, k] = -1.0 if key == "CD" else -(k / (k + 2.0)) ** 2
    return S


def _integrate2(N):
    """Pseudo-inverse of the second derivative, rows 2 and up."""
    B = np.zeros((N, N))
    i = np.arange(2, N, dtype=float)
    B[np.arange(2, N), np.arange(N - 2)] = 1.0 / (4.0 * i * (i - 1.0))
    B[2, 0] *= 2.0
    i = np.arange(2, N - 2)
    B[i, i] = -1.0 / (2.0 * (i.astype(float) ** 2 - 1.0))
    i = np.arange(2, N - 4)
    B[i, i + 2] = 1.0 / (4.0 * i * (i + 1.0))
    return B[2:]


class _Axis:
    """Dense operators of one axis: N points, L dealiased, half length s."""

    def __init__(self, N, s):
        L = int(N * 1.5)
        self.N, self.L, self.s = N, L, s
        self.S = {k: _stencil(N, k) for k in ("CD", "CN")}
        self.T = {k: np.linalg.solve(S.T @ S, S.T) for k, S in self.S.items()}
        self.D = _diff(N) / s
        self.B = _integrate2(N)
        self.V, self.F = _to_values(L, N), _to_coefs(N, L)
        self.I2 = np.eye(N)[2:]

    def helmholtz(self, key, lam):
        return self.B @ self.S[key] - lam / self.s ** 2 * self.I2 @ self.S[key]


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=F64, device="cuda")


def _x(A, v):
    return torch.matmul(A, v)


def _y(A, v):
    return torch.matmul(v, A.T)


def _inv_by_parity(A):
    """Inverses of a stack of matrices that couple modes of equal parity only."""
    out = np.zeros_like(A)
    for p in (0, 1):
        out[..., p::2, p::2] = np.linalg.inv(A[..., p::2, p::2])
    return out


class _Poisson:
    """nabla^2 p = f between Galerkin bases: along y by eigenvectors, along x
    one dense inverse per eigenvalue.  For the singular mode (Neumann) the mean
    is left out and set to zero."""

    def __init__(self, ax, ay, kx, ky, sx, sy):
        Ax, Cx = ax.I2 @ ax.S[kx] / sx ** 2, ax.B @ ax.S[kx]
        Ay, Cy = ay.I2 @ ay.S[ky] / sy ** 2, ay.B @ ay.S[ky]
        n = Ay.shape[0]
        w, Q, Qi = np.zeros(n), np.zeros((n, n)), np.zeros((n, n))
        K = np.linalg.solve(Cy, Ay)
        for p in (0, 1):
            lam, vec = np.linalg.eig(K[p::2, p::2])
            w[p::2] = lam.real
            Q[p::2, p::2] = vec.real
            Qi[p::2, p::2] = np.linalg.inv(vec.real)
        H = Qi @ np.linalg.solve(Cy, ay.B)
        inv = np.empty((n,) + Ax.shape)
        for j in range(0, n, 64):   # some lines at a time
            inv[j:j + 64] = 0.0
            for i in range(j, min(j + 64, n)):
                M = Ax + w[i] * Cx
                if abs(w[i]) < 1e-8:
                    M = M.copy()
                    M[0, :], M[:, 0] = 0.0, 0.0
                    M[0, 0] = 1.0
                inv[i] = M
            inv[j:j + 64] = _inv_by_parity(inv[j:j + 64])
            for i in range(j, min(j + 64, n)):
                if abs(w[i]) < 1e-8:
                    inv[i, 0, 0] = 0.0
        self.Bx, self.H, self.Q, self.inv = _t(ax.B), _t(H), _t(Q), _t(inv)

    def __call__(self, f):
        """f [..., N0, N1] Chebyshev coefficients -> [..., M0, M1]."""
        g = _y(self.H, _x(self.Bx, f))
        lead = g.shape[:-2]
        g = g.reshape((-1,) + g.shape[-2:])
        p = torch.bmm(self.inv, g.permute(2, 1, 0).contiguous()).permute(2, 1, 0)
        return _y(self.Q, p).reshape(lead + p.shape[1:])


def _sidewall(n, s):
    """Boundary temperature of the "zero" case along y: 1/2 at the bottom, -1/2
    at the top, zero in between."""
    y = _grid(n) * s
    k, z = 0.02, y * 2.0 / (y[-1] - y[0])
    return np.where(z < 0, -k * z / (k + z + 1.0) * 0.5, k * z / (k - z + 1.0) * -0.5)


class _Flow:
    """The incompressible Boussinesq step for boxes of one shape, dense."""

    def __init__(self, n0, n1, params, case="rbc", integrator="eu", beta=1.0):
        self.ax, self.ay = _Axis(n0, 0.5), _Axis(n1, 0.5)
        ax, ay = self.ax, self.ay
        self.case, self.beta = case, beta
        self.side = side = "CN" if case == "rbc" else "CD"
        self.keys = ("CD", "CD", side)
        if integrator == "rk3":
            self.abc = ((8 / 15, 8 / 15, 0.0), (2 / 15, 5 / 12, -17 / 60), (1 / 3, 3 / 4, -5 / 12))
        else:
            self.abc = ((1.0, 1.0, 0.0),)
        col = lambda v: _t(np.asarray(v, float)).reshape(-1, 1, 1)
        nu = np.array([math.sqrt(p["pr"] / p["ra"]) for p in params])
        ka = np.array([math.sqrt(1.0 / p["pr"] / p["ra"]) for p in params])
        dt = np.array([p["dt"] for p in params])
        self.nu, self.ka, self.dt = col(nu), col(ka), col(dt)
        self.Sx, self.Sy = {k: _t(ax.S[k]) for k in ax.S}, {k: _t(ay.S[k]) for k in ay.S}
        self.Tx, self.Ty = {k: _t(ax.T[k]) for k in ax.T}, {k: _t(ay.T[k]) for k in ay.T}
        self.Dx, self.Dy, self.Bx, self.By = _t(ax.D), _t(ay.D), _t(ax.B), _t(ay.B)
        self.Vx, self.Vy, self.Fx, self.Fy = _t(ax.V), _t(ay.V), _t(ax.F), _t(ay.F)
        cache = {}

        def inv(axis, a, key, lam):
            k = (a, key, float(lam))
            if k not in cache:
                cache[k] = _inv_by_parity(axis.helmholtz(key, lam))
            return cache[k]
        # per stage and field: inverses of the implicit operators along x and y
        self.Hx, self.Hy = [], []
        for a, _, _ in self.abc:
            hx, hy = [], []
            for f, key in enumerate(self.keys):
                lam = dt * a * beta * (nu if f < 2 else ka)
                hx.append(_t(np.stack([inv(ax, 0, key, v) for v in lam])))
                hy.append(_t(np.stack([inv(ay, 1, "CD", v) for v in lam])))
            self.Hx.append(hx)
            self.Hy.append(hy)
        self.poisson = _Poisson(ax, ay, "CN", "CN", 0.5, 0.5)
        # boundary temperature: Chebyshev coefficients, its y-derivatives
        tb = np.zeros((n0, n1))
        if case == "zero":
            tb[0] = _to_coefs(n1, n1) @ _sidewall(n1, 0.5)
        else:
            tb[0, 1] = -0.5
        self.tb = _t(tb)
        self.tb2 = _y(self.Dy, _y(self.Dy, self.tb))
        self.tb1 = self.values(_y(self.Dy, self.tb))

    def cheb(self, v, f):
        return _y(self.Sy["CD"], _x(self.Sx[self.keys[f]], v))

    def galerkin(self, c, f):
        return _y(self.Ty["CD"], _x(self.Tx[self.keys[f]], c))

    def values(self, c):
        return _y(self.Vy, _x(self.Vx, c))

    def forward(self, v):
        return _y(self.Fy, _x(self.Fx, v))

    def slopes(self, c):
        return self.values(_x(self.Dx, c)), self.values(_y(self.Dy, c))

    def project(self, U, V):
        """(divergence, pressure potential coefficients, corrected U and V)."""
        div = _x(self.Dx, self.cheb(U, 0)) + _y(self.Dy, self.cheb(V, 1))
        P = self.poisson(div)
        mask = torch.ones_like(P)
        mask[..., 0, 0] = 0.0
        p = _y(self.Sy["CN"], _x(self.Sx["CN"], P * mask))
        return div, p, U - self.galerkin(_x(self.Dx, p), 0), V - self.galerkin(_y(self.Dy, p), 1)

    def step(self, X, pres):
        U, V, T = X
        dt, nu, ka = self.dt, self.nu, self.ka
        old = None
        for s, (a, b, c) in enumerate(self.abc):
            ch = [self.cheb(v, f) for f, v in enumerate((U, V, T))]
            ux, uz = self.values(ch[0]), self.values(ch[1])
            rhs = []
            for f in range(3):
                gx, gy = self.slopes(ch[f])
                bc = self.tb1 if f == 2 else 0.0
                conv = b * (gx * ux + gy * uz + bc * uz)
                if c != 0.0:
                    conv = conv + c * (gx * old[0] + gy * old[1] + bc * old[1])
                r = -dt * self.forward(conv)
                if self.beta != 1.0:
                    lap = _x(self.Dx, _x(self.Dx, ch[f])) + _y(self.Dy, _y(self.Dy, ch[f]))
                    r = r + dt * a * (1.0 - self.beta) * (nu if f < 2 else ka) * lap
                rhs.append(r)
            rhs[0] = rhs[0] - dt * a * _x(self.Dx, pres)
            rhs[1] = rhs[1] - dt * a * _y(self.Dy, pres) + dt * a * (ch[2] + self.tb)
            rhs[2] = rhs[2] + dt * a * ka * self.tb2
            new = []
            for f in range(3):
                g = _y(self.By, _x(self.Bx, rhs[f] + ch[f]))
                new.append(torch.matmul(torch.matmul(self.Hx[s][f], g),
                                        self.Hy[s][f].transpose(1, 2).contiguous()))
            div, p, U, V = self.project(new[0], new[1])
            T = new[2]
            pres = pres - nu * self.beta * div + p / (dt * a)
            old = (ux, uz)
        return [U, V, T], pres


def _wall_weights(flow):
    """a, b with Nu = 1 + a^T T b: the mean wall gradient of the temperature."""
    n0, n1 = flow.ax.N, flow.ay.N
    x = _grid(n0)
    e = np.concatenate([x[:1], 0.5 * (x[1:] + x[:-1]), x[-1:]])
    w = np.diff(e) / (x[-1] - x[0])
    a = w @ _to_values(n0, n0) @ flow.ax.S[flow.side]
    g = _to_values(n1, n1) @ flow.ay.D @ flow.ay.S["CD"]
    return _t(a), _t(-0.5 * (g[0] + g[-1]))


def _flow(case, params):
    return _Flow(case["n0"], case["n1"], params, case=case.get("case", "rbc"),
                 integrator=case.get("integrator", "eu"), beta=case.get("beta", 1.0))


def _exact_steps(flow, X, pres, n):
    X = [X[:, f] for f in range(3)]
    for _ in range(n):
        X, pres = flow.step(X, pres)
    return torch.stack(X, dim=1), pres


def _exact_descent(case, seed):
    n0, n1 = case["n0"], case["n1"]
    X, pres = _state(seed, 4, (), n0, n1)
    flow = _flow(case, [dict(ra=case["ra"], pr=1.0, dt=case["dt"])])
    nu, ka, dt = flow.nu, flow.ka, case["dt"]
    smooth = [_Poisson(flow.ax, flow.ay, k, "CD", 0.5, 0.5) for k in ("CD", flow.side)]
    U, V, T, pres = X[0][None], X[1][None], X[2][None], pres[None]
    inner = torch.zeros_like(pres)
    tbv = flow.values(flow.tb)
    for _ in range(case["steps"]):
        cu, cv, ct = (flow.cheb(v, f) for f, v in enumerate((U, V, T)))
        ux, uz, te = flow.values(cu), flow.values(cv), flow.values(ct)
        (Un, Vn, Tn), inner = flow.step([U, V, T], inner)
        r = [flow.cheb((n - o) / dt, f) for f, (n, o) in enumerate(((Un, U), (Vn, V), (Tn, T)))]
        A = [smooth[f == 2](r[f]) / (nu if f < 2 else ka) for f in range(3)]
        cA = [flow.cheb(v, f) for f, v in enumerate(A)]
        g = [flow.slopes(c) for c in cA]
        out = []
        for d, (f, v) in enumerate(((0, U), (1, V))):
            grad = _x(flow.Dx, pres) if d == 0 else _y(flow.Dy, pres)
            own = g[f][0] * ux + g[f][1] * uz
            adj = g[0][d] * ux + g[1][d] * uz + g[2][d] * (te + tbv)
            out.append(v + dt * flow.galerkin(flow.forward(own + adj) - grad + r[f], f))
        _, p, U, V = flow.project(*out)
        pres = pres + p / dt
        T = T + dt * flow.galerkin(flow.forward(g[2][0] * ux + g[2][1] * uz) + r[2] + cA[1], 2)
    return [U[0], V[0], T[0], pres[0]]


@functools.lru_cache(maxsize=4)
def _plain_axes(n0, n1):
    return _Axis(n0, 1.0), _Axis(n1, 1.0)


def _exact_helmholtz(ax, ay, lam, f, old):
    g = _y(_t(ay.B), _x(_t(ax.B), f)) + _y(_t(ay.B @ ay.S["CD"]), _x(_t(ax.B @ ax.S["CD"]), old))
    return _y(_t(_inv_by_parity(ay.helmholtz("CD", lam))),
              _x(_t(_inv_by_parity(ax.helmholtz("CD", lam))), g))


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        X, pres = _state(seed, 1, (), case["n0"], case["n1"])
        flow = _flow(case, [dict(ra=case["ra"], pr=1.0, dt=case["dt"])])
        X, pres = _exact_steps(flow, X[None], pres[None], case["steps"])
        return [X[0, 0], X[0, 1], X[0, 2], pres[0]]
    if kind == "batch":
        X, pres = _state(seed, 2, (case["count"],), case["n0"], case["n1"])
        return list(_exact_steps(_flow(case, _batch_params(case, seed)), X, pres, case["steps"]))
    if kind == "mixed":
        by_shape = {}
        for s in _mixed_specs(case, seed):
            by_shape.setdefault(s["shape"], []).append(s)
        out = []
        for c, shape in enumerate(sorted(by_shape)):
            X, pres = _state(seed, 100 + c, (len(by_shape[shape]),), *shape)
            out += list(_exact_steps(_Flow(*shape, by_shape[shape]), X, pres, case["steps"]))
        return out
    if kind == "gradient":
        X, pres = _state(seed, 3, (1,), case["n0"], case["n1"])
        flow = _flow(case, [dict(ra=case["ra"], pr=1.0, dt=case["dt"])])
        a, b = _wall_weights(flow)
        T0 = X[:, 2].clone().requires_grad_(True)
        S, J = [X[:, 0], X[:, 1], T0], 0.0
        for _ in range(case["steps"]):
            S, pres = flow.step(S, pres)
            J = J + (1.0 + torch.matmul(torch.matmul(a, S[2]), b)) / case["steps"]
        J.sum().backward()
        return [J.detach(), T0.grad]
    if kind == "descent":
        return _exact_descent(case, seed)
    n0, n1 = case["n0"], case["n1"]
    ax, ay = _plain_axes(n0, n1)
    if kind == "transform":
        c = _coefs(seed, 51, (case["count"], n0, n1), 1.0)
        return [_y(_t(_to_values(n1, n1)), _x(_t(_to_values(n0, n0)), c)), c]
    if kind == "solve":
        f = _coefs(seed, 61, (case["count"], n0, n1), 1.0)
        old = _y(_t(ay.T["CD"]), _x(_t(ax.T["CD"]), f))
        return [old, _exact_helmholtz(ax, ay, case["lam"], f, old),
                _Poisson(ax, ay, "CD", "CD", 1.0, 1.0)(f)]
    vh = _coefs(seed, 71, (n0 - 2, n1 - 2), 0.3)
    c = _y(_t(ay.S["CD"]), _x(_t(ax.S["CD"]), vh))
    dx = _x(_t(ax.D), c)
    Vx, Vy = _t(ax.V), _t(ay.V)
    u = _y(Vy, _x(Vx, c))
    conv = _y(Vy, _x(Vx, dx)) * u + _y(Vy, _x(Vx, _y(_t(ay.D), c))) * u
    conv = _y(_t(ay.F), _x(_t(ax.F), conv))
    return [_y(_t(_to_values(n1, n1)), _x(_t(_to_values(n0, n0)), c)), vh, dx, conv,
            _exact_helmholtz(ax, ay, 0.02, conv, vh),
            _Poisson(ax, ay, "CD", "CD", 1.0, 1.0)(dx)]
