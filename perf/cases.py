"""Timing cases of the framework: what a user's program has it do.

Most cases advance a simulation by a few steps and read the fields back, as
a program that writes or looks at frames does; the others call the parts
that a program can use by themselves (projection solver, narrow band with
extension, the learned guess's network).
"""
import math

import numpy as np
import torch

import incrmt_amd as ia
from incrmt_amd import workloads as wl
from incrmt_amd.conv import conv_test_case
from incrmt_amd.ensemble import Ensemble

FRAME = 4 * math.pi / 240  # ftest's frame interval


def listed():
    return [
        # the smallest run in use (smoke test, ensemble members): launches and latency
        dict(name="spin_64", kind="spin", m=64, mixed=False, guess=0, steps=32),
        # `ftest simple-spin 128` with the reference's own solver settings
        dict(name="spin_128", kind="spin", m=128, mixed=False, guess=0, steps=32),
        # the benchmark's grid and solver: single-precision V-cycles, quadratic starts
        dict(name="spin_1024", kind="spin", m=1024, mixed=True, guess=2, steps=24),
        # the same grid with the plain double-precision solver
        dict(name="spin_1024_fp64", kind="spin", m=1024, mixed=False, guess=0, steps=24),
        # the sediment-style run: many solids, the largest grid
        dict(name="circles_2048", kind="circles", m=2048, count=64, mixed=True, steps=8),
        # conv_test's periodic box at one of its odd-factor sizes, a heavy circle
        dict(name="conv_360", kind="conv", m=360, ctype=4, steps=12),
        # horizontal flow past a soft circle, zero pressure at the outflow
        dict(name="flow_256", kind="flow", m=256, n=128, y_prd=True, steps=24),
        # independent rotors of uneven size side by side
        dict(name="ensemble_16", kind="ensemble", count=16, largest=256, steps=8),
        # the standalone nodal projection to 1e-10, from host arrays
        dict(name="fem_1024", kind="fem", m=1024, n=1024, mixed=True, zpr=False),
        # the standalone cell projection with a solid's density and an outflow edge
        dict(name="mac_256", kind="mac", m=256, n=128, mixed=False, zpr=True),
        # the narrow band and the extension by themselves
        dict(name="band_512", kind="band", m=512, n=512, shape="rotor"),
        # the learned guess's network: prediction, loss and gradient
        dict(name="net_257", kind="net", m=257, n=257),
    ]


def draw(rng):
    kind = rng.choice(["spin", "spin", "circles", "conv", "flow", "ensemble", "fem", "mac", "band", "net"])

    def grid(lo, hi):  # a size that halves down to 4..7, spread over the logarithm
        got = [a << k for k in range(1, 10) for a in (4, 5, 6, 7) if lo <= a << k <= hi]
        want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return min(got, key=lambda v: abs(math.log(v / want)))

    def whole(lo, hi):
        return round(math.exp(rng.uniform(math.log(lo), math.log(hi))))

    def outflow():  # grids that halve down to the few points a zero-pressure edge needs
        n = rng.choice([32, 64, 128, 256, 512, 48, 96, 192, 384])
        m = n * 4 // 3 if n % 3 == 0 else n * rng.choice([1, 2])
        return dict(m=m, n=n) if m <= 512 else dict(m=n, n=n)

    def nodes():  # any even count, or an odd one that halves
        m = 2 * whole(17, 640) if rng.random() < 0.7 else grid(32, 1280) + 1
        return dict(m=m, n=m if rng.random() < 0.4 else 2 * round(0.5 * m * rng.uniform(0.6, 1.0)))

    if kind == "spin":
        return dict(kind=kind, m=grid(64, 1280), mixed=rng.random() < 0.5, guess=rng.choice([0, 1, 2]),
                    steps=rng.randint(8, 24))
    if kind == "circles":
        return dict(kind=kind, m=grid(512, 1280), count=rng.randint(2, 40), mixed=rng.random() < 0.7,
                    steps=rng.randint(4, 8))
    if kind == "conv":
        return dict(kind=kind, m=whole(64, 640), ctype=rng.choice([0, 2, 3, 4, 5, 7]), steps=rng.randint(4, 12))
    if kind == "flow":
        return dict(kind=kind, y_prd=rng.random() < 0.5, steps=rng.randint(8, 24), **outflow())
    if kind == "ensemble":
        return dict(kind=kind, count=rng.randint(3, 20), largest=rng.choice([128, 256, 512]), steps=rng.randint(2, 6))
    if kind == "fem":
        return dict(kind=kind, mixed=rng.random() < 0.5, zpr=False, **nodes())
    if kind == "mac":
        return dict(kind=kind, mixed=rng.random() < 0.5, zpr=True, **outflow())
    if kind == "band":
        m = whole(72, 1400)
        return dict(kind=kind, m=m, n=round(m * rng.uniform(0.8, 1.0)), shape=rng.choice(["rotor", "wavy", "two"]))
    return dict(kind=kind, m=whole(33, 520), n=whole(33, 520))


# ------------------------------------------------------------------ inputs
def _precision(c):
    return ia.PREC_MIXED if c["mixed"] else ia.PREC_FP64


def _sim(c, seed):
    """An initialised simulation and its timestep; the seed sets the rotor's
    speed, the circles' places or the solid's place."""
    r = np.random.default_rng(seed)
    if c["kind"] == "spin":
        f = ia.simple_spin(c["m"], omega=r.uniform(0.5, 2.0), precision=_precision(c), guess=c["guess"])
        return f, f.timestep_select(FRAME)[1]
    if c["kind"] == "circles":
        f = ia.multibody(c["m"], c["count"], seed=seed, precision=_precision(c))
        return f, f.dt_reg
    if c["kind"] == "conv":
        f = conv_test_case(c["m"], c["ctype"], coarsest=min(280, c["m"]))
        f.set("u", f.get("u") * r.uniform(0.5, 1.0))  # a weaker or stronger pulse
        return f, f.timestep_select(0.02)[1]
    f = ia.Fluid2D(c["m"], c["n"], visc=1e-2, rhof=1.0, ax=-1.0, bx=-1.0 + 2.0 * c["m"] / c["n"], ay=-1.0, by=1.0,
                   y_prd=c["y_prd"])
    f.add_circle(r.uniform(-0.3, 0.3), r.uniform(-0.2, 0.2), r.uniform(0.25, 0.35), 0.0, G=2.0, rhos=1.5)
    f.set_horizontal_flow(1.0)
    f.initialize(0.8, 0.4, 0.8)
    return f, f.dt_reg


def _density(m, n, r):
    """Cell densities with one ghost layer: a disk of three times the fluid's
    density, and a smooth variation."""
    X, Y = np.meshgrid((np.arange(m + 2) - 0.5) / m, (np.arange(n + 2) - 0.5) / n)
    R = np.where(np.hypot(X - r.uniform(0.4, 0.6), Y - r.uniform(0.4, 0.6)) < 0.3, 3.0, 1.0)
    return R * (1 + 0.2 * np.sin(2 * np.pi * (X * r.uniform(1, 3) + Y * r.uniform(1, 3))))


def _mac_irho(R, m, n):
    """Face inverse densities in the solver's layout: left and lower face of
    each cell, then the right-edge and the top-edge faces."""
    K = 1 / R
    fx = 0.5 * (K[1:-1, 1:] + K[1:-1, :-1])  # n x (m+1)
    fy = 0.5 * (K[1:, 1:-1] + K[:-1, 1:-1])  # (n+1) x m
    cells = np.stack([fx[:, :m], fy[:n, :]], axis=2).ravel()
    return np.concatenate([cells, fx[:, m], fy[n, :]]), fx, fy


def _mac_system(c, seed):
    m, n, r = c["m"], c["n"], np.random.default_rng(seed)
    h = 2.0 / n
    irho, fx, fy = _mac_irho(_density(m, n, r), m, n)
    x, y = np.meshgrid((np.arange(m) + 0.5) / m, (np.arange(n) + 0.5) / n)
    b = sum(r.standard_normal() / (k + 1) * np.cos(np.pi * (k + 1) * x + r.uniform(0, 6)) *
            np.cos(np.pi * r.integers(1, 9) * y) for k in range(12))
    return h, irho, fx, fy, b + 0.05 * r.standard_normal(b.shape)


def _fem_system(c, seed):
    """The nodal divergence of a seeded smooth velocity between walls."""
    m, n, r = c["m"], c["n"], np.random.default_rng(seed)
    h = 1.0 / (m - 1)
    xs, ys = (np.arange(m - 1) + 0.5) / (m - 1), (np.arange(n - 1) + 0.5) / (n - 1)
    kx, ky = r.integers(1, 17, 32), r.integers(1, 17, 32)
    sx, sy = np.sin(np.pi * np.outer(kx, xs)), np.sin(np.pi * np.outer(ky, ys))
    u, v = (sy.T @ ((r.standard_normal(32) / (kx * kx + ky * ky))[:, None] * sx) for _ in range(2))
    b = wl.fem_source(u, v, h, h)
    return h, b - b.mean()


def _band_input(c, seed):
    m, n, r = c["m"], c["n"], np.random.default_rng(seed)
    d = 2.0 / min(m, n)
    X, Y = np.meshgrid(d * (np.arange(m) - 0.5 * (m - 1)), d * (np.arange(n) - 0.5 * (n - 1)))
    a = r.uniform(0.1, 1.0)
    xr, yr = math.cos(a) * X + math.sin(a) * Y, math.cos(a) * Y - math.sin(a) * X
    if c["shape"] == "rotor":
        t = np.cos(3 * np.arctan2(yr, xr))
        phi = np.hypot(xr, yr) - 0.8 / 1.625 * (0.875 + t * (0.5 + 0.25 * t))
    elif c["shape"] == "wavy":
        phi = np.hypot(X - 0.08 * a, Y) - 0.4 + 0.18 * np.sin(11 * X) + 0.13 * np.sin(13.5 * Y + a)
    else:
        phi = np.minimum(np.hypot(X - 0.35, Y - 0.1 * a) - 0.25, np.hypot(X + 0.35, Y + 0.1 * a) - 0.3)
    inside = phi < 0
    return d, X, Y, phi, np.where(inside, (X + 0.5 * Y) ** 2, 0.0), np.where(inside, np.sin(3 * X) * Y, 0.0)


# input channels, second input's channels (the skip), output channels, stride, ReLU
_NET = [(4, 0, 16, 1, True), (16, 0, 16, 1, True), (16, 0, 32, 2, True), (32, 0, 32, 1, True),
        (32, 0, 48, 2, True), (48, 0, 48, 1, True), (48, 0, 64, 2, True), (64, 0, 64, 1, True),
        (64, 48, 48, 1, True), (48, 32, 32, 1, True), (32, 16, 16, 1, True), (16, 0, 1, 1, False)]


def _net_input(c, seed):
    m, n, r = c["m"], c["n"], np.random.default_rng(seed)
    y, x = np.meshgrid(np.linspace(0, 1, n), np.linspace(0, 1, m), indexing="ij")
    a = np.stack([np.sin(3 * x + 2 * y) + 0.3 * r.standard_normal((n, m)),
                  np.tanh(4 * (np.hypot(x - 0.5, y - 0.5) - 0.3)),
                  np.cos(5 * x * y) + 0.3 * r.standard_normal((n, m))], axis=2).astype(np.float32)
    p = []
    for c1, c2, co, _, _ in _NET:  # He-scaled weights, small biases
        p.append(r.standard_normal(co * 9 * (c1 + c2)) * math.sqrt(2.0 / (9 * (c1 + c2))))
        p.append(0.05 * r.standard_normal(co))
    p = torch.tensor(np.concatenate(p)).bfloat16().float().numpy()  # values the network holds exactly
    return p, torch.tensor(a).bfloat16().float().numpy(), (np.sin(2 * x) * np.cos(3 * y)).astype(np.float32)


# ------------------------------------------------------------------- calls
class _Held:
    """What a program holds of one case; closes it with the last reference."""

    def __init__(self, case, **kw):
        self.case = case
        self.__dict__.update(kw)

    def __del__(self):
        for h in ("sim", "solver", "net"):
            if hasattr(self, h):
                getattr(self, h).close()


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("spin", "circles", "conv", "flow"):
        f, dt = _sim(c, seed)
        return _Held(c, sim=f, dt=dt)
    if kind == "ensemble":
        r = np.random.default_rng(seed)
        return _Held(c, sim=Ensemble([(m, r.uniform(0.5, 2.0)) for m in _members(c)], precision=ia.PREC_MIXED,
                                     guess=ia.GUESS_QUADRATIC))
    if kind == "fem":
        h, b = _fem_system(c, seed)
        return _Held(c, solver=ia.MgSolver(ia.MG_FEM, c["m"], c["n"], h, h), b=b, z0=np.zeros(b.size))
    if kind == "mac":
        h, irho, _, _, b = _mac_system(c, seed)
        s = ia.MgSolver(ia.MG_MAC, c["m"], c["n"], h, h, zpr=c["zpr"])
        s.set_irho(irho)
        return _Held(c, solver=s, b=b, z0=np.zeros(b.size))
    if kind == "band":
        d, X, Y, phi, fx, fy = _band_input(c, seed)
        return _Held(c, args=(c["m"], c["n"], float(X[0, 0]), float(Y[0, 0]), d, d, -7 * d, 7 * d), fields=(phi, fx, fy))
    p, a, t = _net_input(c, seed)
    net = ia.UNet(c["m"], c["n"])
    net.set_params(p)
    return _Held(c, net=net, a=a, t=t)


def _members(c):
    sizes = [s for s in (64, 128, 256, 512) if s <= c["largest"]]
    return [sizes[k % len(sizes)] for k in range(c["count"])]


def run(state):
    c = state.case
    kind = c["kind"]
    if kind in ("spin", "circles", "conv", "flow"):
        f = state.sim
        f.steps(state.dt, c["steps"])
        out = {k: f.get(k) for k in ("u", "v", "p")}
        if f.nobj and kind != "circles":
            out.update({k: f.get(k) for k in ("X", "Y", "phi")})
        elif f.nobj:  # the fields that see every solid, and one solid's own
            out.update(rho=f.get("rho"), X=f.get("X"), Y=f.get("Y"))
        return out
    if kind == "ensemble":
        state.sim.steps(c["steps"])
        return [[f.get("u"), f.get("v"), f.get("p")] for f in state.sim.members]
    if kind in ("fem", "mac"):
        z = state.solver.solve(state.b, rel_tol=1e-10, precision=_precision(c), z=state.z0)[0]
        if not c["zpr"]:
            z -= z.mean()  # between walls the solution is known up to a constant
        return z
    if kind == "band":
        phi, status, fx, fy, _ = ia.extrapolate(*state.args, *state.fields)
        return dict(phi=phi, status=status, fx=fx, fy=fy)
    prediction = state.net.forward(state.a)
    loss, grad = state.net.gradient(state.a, state.t)
    return dict(prediction=prediction, loss=loss, grad=grad)


def work(case):
    """What a pass cannot do without. A step reads and writes velocity and
    pressure and one reference map with its level set once, and spends
    about a thousand operations a cell (sweeps, stresses and the least
    multigrid work that solves both projections); a projection from zero
    reads b and writes z with about 600 operations a point; the network's
    operations are its multiply-adds, forward twice and backward once."""
    c, kind = case, case["kind"]
    if kind == "ensemble":
        cells = sum(m * m for m in _members(c))
    else:
        cells = c["m"] * c.get("n", c["m"])
    if kind in ("spin", "circles", "conv", "flow", "ensemble"):
        return {"bytes": 96.0 * cells * c["steps"], "flops": 1000.0 * cells * c["steps"]}
    if kind in ("fem", "mac"):
        return {"bytes": (16.0 if kind == "fem" else 32.0) * cells, "flops": 600.0 * cells}
    if kind == "band":
        return {"bytes": 52.0 * cells, "flops": 100.0 * cells}
    macs = sum(9 * (c1 + c2) * co / 4 ** lv for (c1, c2, co, _, _), lv in
               zip(_NET, (0, 0, 1, 1, 2, 2, 3, 3, 2, 1, 0, 0)))
    return {"bytes": 24.0 * cells, "flops": 2.0 * 4 * macs * cells}


# ------------------------------------------------------- the same in 64 bits
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.tensor(a, dtype=torch.float64, device=_device())


def _exact_fem(c, seed):
    """Bilinear elements of constant density are a sum of two tensor products
    of one-dimensional stiffness and mass matrices."""
    h, b = _fem_system(c, seed)

    def line(k):
        K = 2 * np.eye(k) - np.eye(k, k=1) - np.eye(k, k=-1)
        M = 4 * np.eye(k) + np.eye(k, k=1) + np.eye(k, k=-1)
        K[0, 0] = K[-1, -1] = 1
        M[0, 0] = M[-1, -1] = 2
        L = torch.linalg.cholesky(_t(M / 6))
        Li = torch.linalg.inv(L)
        w, V = torch.linalg.eigh(Li @ _t(K) @ Li.T)
        w[0] = 0
        return w, Li.T @ V  # K v = w M v, v^T M v = 1

    (wx, Vx), (wy, Vy) = line(c["m"]), line(c["n"])
    q = Vy.T @ _t(b) @ Vx
    d = wy[:, None] + wx[None, :]
    d[0, 0] = 1
    q = q / d
    q[0, 0] = 0
    z = Vy @ q @ Vx.T
    return (z - z.mean()).ravel()


def _exact_mac(c, seed):
    """Conjugate gradients on the face-flux operator, preconditioned by the
    direct solve of the constant-density one."""
    h, _, fx, fy, b = _mac_system(c, seed)
    m, n = c["m"], c["n"]
    kx, ky = _t(fx) / h ** 2, _t(fy) / h ** 2
    kx[:, 0] = 0
    kx[:, m] *= 2  # half a cell to the zero-pressure edge
    ky[0] = 0
    ky[n] = 0

    def apply(q):  # minus the operator: positive definite
        fl = torch.zeros(n, m + 1, dtype=q.dtype, device=q.device)
        fl[:, 1:m] = q[:, 1:] - q[:, :-1]
        fl[:, m] = -q[:, -1]
        up = torch.zeros(n + 1, m, dtype=q.dtype, device=q.device)
        up[1:n] = q[1:] - q[:-1]
        fl, up = fl * kx, up * ky
        return fl[:, :-1] - fl[:, 1:] + up[:-1] - up[1:]

    def line(k, right):
        K = 2 * np.eye(k) - np.eye(k, k=1) - np.eye(k, k=-1)
        K[0, 0], K[-1, -1] = 1, right
        return torch.linalg.eigh(_t(K / h ** 2))

    (wx, Vx), (wy, Vy) = line(m, 3), line(n, 1)
    d = 0.6 * (wy[:, None] + wx[None, :])
    f = -_t(b)
    z, r = torch.zeros_like(f), f.clone()
    p, rho = None, None
    for _ in range(200):
        s = Vy @ ((Vy.T @ r @ Vx) / d) @ Vx.T
        new = float((r * s).sum())
        p = s if p is None else s + (new / rho) * p
        rho = new
        q = apply(p)
        a = rho / float((p * q).sum())
        z, r = z + a * p, r - a * q
        if float(r.norm()) < 1e-14 * float(f.norm()):
            break
    return z.ravel()


def _exact_net(c, seed):
    p, a, t = _net_input(c, seed)
    m, n = c["m"], c["n"]
    p = _t(p).requires_grad_()
    at = 0

    def conv(k, x):
        nonlocal at
        c1, c2, co, stride, relu = _NET[k]
        cin = c1 + c2
        W = p[at:at + co * 9 * cin].view(co, 3, 3, cin).permute(0, 3, 1, 2)
        bias = p[at + co * 9 * cin:at + co * 9 * cin + co]
        at += co * 9 * cin + co
        H, Wd = x.shape[1:]
        Ho, Wo = -(-H // stride), -(-Wd // stride)
        xp = torch.nn.functional.pad(x, (1, 1, 1, 1))
        y = bias[:, None].expand(co, Ho * Wo)
        for dy in range(3):
            for dx in range(3):
                part = xp[:, dy:dy + stride * (Ho - 1) + 1:stride, dx:dx + stride * (Wo - 1) + 1:stride]
                y = y + W[:, :, dy, dx] @ part.reshape(cin, -1)
        y = y.view(co, Ho, Wo)
        return torch.relu(y) if relu else y

    def up(x, H, Wd):  # vertex-centred linear interpolation, clamped past the last node
        def line(k, kc):
            U = torch.zeros(k, kc, dtype=torch.float64, device=x.device)
            for i in range(k):
                U[i, i // 2] += 0.5
                U[i, min(i // 2 + i % 2, kc - 1)] += 0.5
            return U
        return line(H, x.shape[1]) @ x @ line(Wd, x.shape[2]).T

    x = torch.zeros(4, n, m, dtype=torch.float64, device=_device())
    x[:3] = _t(a).permute(2, 0, 1)
    e0 = conv(1, conv(0, x))
    e1 = conv(3, conv(2, e0))
    e2 = conv(5, conv(4, e1))
    y = conv(7, conv(6, e2))
    for k, e in ((8, e2), (9, e1), (10, e0)):
        y = conv(k, torch.cat([up(y, *e.shape[1:]), e]))
    y = conv(11, y)[0]
    loss = 0.5 * ((y - _t(t)) ** 2).mean()
    loss.backward()
    return dict(prediction=y.detach(), loss=float(loss.detach()), grad=p.grad)


def exact(case, seed):
    """The solutions and the network's values as 64-bit linear algebra gives
    them; a simulation's fields and a marched band have no such short form."""
    return {"fem": _exact_fem, "mac": _exact_mac, "net": _exact_net}.get(case["kind"], lambda c, s: None)(case, seed)
