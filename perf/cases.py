"""Performance cases: what programs written on this package have it do.

Each case is one call sequence through the public entry points (Numerics,
Batch, FusedSolver, Stepper): the plain line operators, batches of uneven
subdomains, whole RK4 steps of the fused solver (viscous and inviscid,
constant and per-point metrics, FP64 and FP32 intermediates), the adjoint of
a step, and a step of the per-operator layer with walls.  `exact` evaluates
the same quantities with dense operators in plain torch, FP64.

A case is a dict of plain values: `kind`, the grid `nx, ny, nz`, the faces of
each axis as a letter (P periodic, N non-reflective, W viscous wall) and the
options of the kind.
"""
import math

import numpy as np
import torch

import compact_schemes_amd as cs
from compact_schemes_amd.batch import Batch
from compact_schemes_amd.fused import FusedSolver
from compact_schemes_amd.stepper import Stepper

GAM = 1.4
PRANDTL = 0.71
ALPHA_F = 0.49
MU = 1e-4
CODES = {"P": 45, "N": 10, "W": 25}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the plain method on a small periodic block (six line operators): the
        # smallest calls, where launches and latency count
        {"name": "ops_64", "kind": "ops", "nx": 64, "ny": 64, "nz": 64, "faces": "PPP"},
        # the same six operators on one large block of uneven, odd sizes with closures
        {"name": "ops_ragged", "kind": "ops", "nx": 292, "ny": 271, "nz": 284, "faces": "NNN"},
        # many subdomains of unrelated sizes in [48, 320] per axis, captured once and replayed
        {"name": "batch_16", "kind": "batch", "count": 16, "lo": 48, "hi": 320, "sizes": 3, "faces": "PPP"},
        # one RK4 step of a small viscous block: latency of a whole step
        {"name": "step_small", "kind": "step", "nx": 48, "ny": 40, "nz": 32, "faces": "NNN", "viscous": True,
         "f32": False, "curv": False},
        # an ordinary block whose sizes split into no equal chunks
        {"name": "step_ragged", "kind": "step", "nx": 150, "ny": 133, "nz": 97, "faces": "NNN", "viscous": True,
         "f32": False, "curv": False},
        # the headline block: viscous, non-reflective faces, time step, four stages, filter
        {"name": "step_256", "kind": "step", "nx": 256, "ny": 256, "nz": 256, "faces": "NNN", "viscous": True,
         "f32": False, "curv": False},
        # the forward step of an acoustic rollout (inviscid, periodic in x)
        {"name": "step_euler", "kind": "step", "nx": 128, "ny": 128, "nz": 128, "faces": "PNN", "viscous": False,
         "f32": False, "curv": False},
        # long lines in x and y, viscous intermediates stored in FP32
        {"name": "step_f32", "kind": "step", "nx": 512, "ny": 288, "nz": 96, "faces": "PPP", "viscous": True,
         "f32": True, "curv": False},
        # a curvilinear block: metrics, Jacobian and face normals per point
        {"name": "step_curv", "kind": "step", "nx": 192, "ny": 160, "nz": 144, "faces": "NPN", "viscous": True,
         "f32": False, "curv": True},
        # forward step with its tape, then the adjoint of the step
        {"name": "adjoint_128", "kind": "adjoint", "nx": 128, "ny": 128, "nz": 128, "faces": "PNN"},
        # a channel between viscous walls through the per-operator layer
        {"name": "walls", "kind": "walls", "nx": 160, "ny": 128, "nz": 96, "faces": "PWP"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_dims(rng, lo, hi, points, step=1):
    while True:
        d = [max(lo, _log_int(rng, lo, hi) // step * step) for _ in range(3)]
        if d[0] * d[1] * d[2] <= points:
            return dict(zip(("nx", "ny", "nz"), d))


def draw(rng):
    kind = rng.choice(["ops", "ops", "batch", "step", "step", "step", "step", "adjoint", "walls"])
    if kind == "ops":
        return {"kind": kind, "faces": rng.choice(["PPP", "NNN", "PNP"]), **_log_dims(rng, 40, 320, 320 ** 3)}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(6, 16), "lo": 48, "hi": rng.randint(96, 320),
                "sizes": rng.randint(10, 10 ** 6), "faces": rng.choice(["PPP", "NNN"])}
    if kind == "step":
        curv = rng.random() < 0.25
        viscous = curv or rng.random() < 0.75
        return {"kind": kind, "faces": rng.choice(["NNN", "PPP", "PNN", "NPN"]), "viscous": viscous,
                "f32": viscous and rng.random() < 0.3, "curv": curv,
                **_log_dims(rng, 24, 512, 12_000_000 if not curv else 5_000_000, rng.choice([1, 1, 8, 16]))}
    if kind == "adjoint":
        return {"kind": kind, "faces": rng.choice(["PNN", "PPP", "NNN"]),
                **_log_dims(rng, 32, 160, 2_500_000, rng.choice([8, 8, 1]))}
    return {"kind": kind, "faces": rng.choice(["PWP", "NWP"]), **_log_dims(rng, 32, 192, 3_000_000)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda")


def _dims(case):
    return case["nx"], case["ny"], case["nz"]


def _nbc(case):
    row = [CODES[c] for c in case["faces"]]
    return [row, list(row)]


def _axes(dims):
    nx, ny, nz = dims
    ar = lambda n: torch.arange(n, dtype=torch.float64, device=_device())
    return ar(nx).view(1, 1, nx), ar(ny).view(1, ny, 1), ar(nz).view(nz, 1, 1)


def _waves(dims, rng, modes, kmax):
    """Sum of seeded plane waves (periodic on the block), amplitude about 1 each."""
    x, y, z = _axes(dims)
    f = torch.zeros((dims[2], dims[1], dims[0]), dtype=torch.float64, device=_device())
    for _ in range(modes):
        k = rng.integers(1, kmax + 1, size=3)
        phi = float(rng.uniform(0.0, 2.0 * np.pi))
        w = [2.0 * np.pi * float(k[a]) / dims[a] for a in range(3)]
        f += torch.sin(w[0] * x + w[1] * y + w[2] * z + phi)
    return f


def _scalar_field(dims, seed):
    """Eight plane waves of wavenumbers 1..20 plus 1e-3 noise, flat."""
    rng = np.random.default_rng(seed)
    f = _waves(dims, rng, 8, 20)
    g = torch.Generator(device=_device())
    g.manual_seed(int(seed))
    f += 1e-3 * torch.randn(f.shape, generator=g, device=_device(), dtype=torch.float64)
    return f.reshape(-1).contiguous()


def _flow(case, seed):
    """Conserved variables [5][lmx], flat: uniform flow carried by the frame
    velocity, a Gaussian pressure pulse and smooth waves of 1e-3 in every
    variable; between walls a velocity profile that vanishes on them."""
    dims = _dims(case)
    rng = np.random.default_rng(seed)
    x, y, z = _axes(dims)
    cen = [rng.uniform(0.3 * n, 0.7 * n) for n in dims]
    r2 = (x - cen[0]) ** 2 + (y - cen[1]) ** 2 + (z - cen[2]) ** 2
    pulse = 1e-2 * torch.exp(-math.log(2.0) * r2 / 64.0)
    wave = [1e-3 * _waves(dims, rng, 2, 3) for _ in range(5)]
    rho = 1.0 + pulse + wave[0]
    p = 1.0 / GAM + pulse + wave[4]
    u, v, w = wave[1], wave[2], wave[3]
    if "W" in case["faces"]:
        s = torch.sin(np.pi * y / (dims[1] - 1))
        u = u * s - _umf(case)[0] * (1.0 - s)
        v, w = v * s, w * s
        p = (1.0 / GAM + (pulse + wave[4]) * s) * torch.ones_like(rho)
        rho = 1.0 + (pulse + wave[0]) * s
    E = p / (GAM - 1.0) + 0.5 * rho * (u * u + v * v + w * w)
    return torch.stack([rho, rho * u, rho * v, rho * w, E]).reshape(-1).contiguous()


def _umf(case):
    return (0.1, 0.0, 0.0) if "W" in case["faces"] else (0.5, 0.0, 0.0)


def _skewed_metrics(dims, s=0.3):
    """Metric rows [axis][component], Jacobian and unit face normals of the
    grid x = i + s sin(2 pi j/Ny), y = j + s sin(2 pi k/Nz), z = k + s sin(2 pi i/Nx)."""
    x, y, z = _axes(dims)
    nx, ny, nz = dims
    tw = 2.0 * np.pi
    full = torch.zeros((nz, ny, nx), dtype=torch.float64, device=_device())
    A = s * tw / ny * torch.cos(tw * y / ny) + full
    B = s * tw / nz * torch.cos(tw * z / nz) + full
    C = s * tw / nx * torch.cos(tw * x / nx) + full
    one = torch.ones_like(full)
    rows = [[one, -A, A * B], [B * C, one, -B], [-C, A * C, one]]
    J = 1.0 / (1.0 + A * B * C)
    cm = []
    for a in range(3):
        n = dims[a]
        faces = []
        for face in range(2):
            r = torch.stack([c.select(2 - a, face * (n - 1)).reshape(-1) for c in rows[a]])
            faces.append(r / torch.sqrt((r * r).sum(0)))
        cm.append(torch.stack(faces))
    return rows, J, cm


def _unit_normals(dims):
    nx, ny, nz = dims
    out = []
    for a, fs in enumerate((ny * nz, nx * nz, nx * ny)):
        c = torch.zeros((2, 3, fs), dtype=torch.float64, device=_device())
        c[:, a] = 1.0
        out.append(c)
    return out


def _boundary_weights(dims):
    w = np.zeros((dims[2], dims[1], dims[0]))
    w[0], w[-1], w[:, 0], w[:, -1], w[:, :, 0], w[:, :, -1] = (1.0,) * 6
    return w.reshape(-1)


def _state(case):
    """The geometry a program hands to the solvers (numpy, reference layout)."""
    dims = _dims(case)
    lmx = dims[0] * dims[1] * dims[2]
    st = {"umf": _umf(case), "ssk": np.broadcast_to(np.float64(MU), (lmx,)), "sbcc": _boundary_weights(dims)}
    if case.get("curv"):
        rows, J, cm = _skewed_metrics(dims)
        for key, r in zip(("xim", "etm", "zem"), rows):
            st[key] = torch.stack(r).reshape(-1).cpu().numpy()
        st["yaco"] = J.reshape(-1).cpu().numpy()
        st["cm"] = [c.reshape(-1).cpu().numpy() for c in cm]
    else:
        # unit spacing: (1,0,0), (0,1,0), (0,0,1) as three views of one buffer
        buf = np.zeros(5 * lmx)
        buf[2 * lmx:3 * lmx] = 1.0
        st["xim"], st["etm"], st["zem"] = buf[2 * lmx:], buf[lmx:4 * lmx], buf[:3 * lmx]
        st["yaco"] = np.broadcast_to(np.float64(1.0), (lmx,))
        st["cm"] = [c.reshape(-1) for c in _unit_normals(dims)]
    return st


def _batch_dims(case):
    rng = np.random.default_rng(case["sizes"])
    return [tuple(int(v) for v in rng.integers(case["lo"], case["hi"] + 1, size=3)) for _ in range(case["count"])]


def prepare(case, seed):
    dev = _device()
    kind = case["kind"]
    if kind == "batch":
        dims = _batch_dims(case)
        f = [_scalar_field(d, 1000 * seed + i) for i, d in enumerate(dims)]
        d = [torch.empty_like(f[i // 3]) for i in range(3 * len(f))]
        b = Batch(dims, _nbc(case))
        b.bind(f, d)
        b.set_persistent(2)
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        b.capture(stream)
        torch.cuda.current_stream().wait_stream(stream)
        return {"case": case, "batch": b, "f": f, "d": d}
    dims = _dims(case)
    if kind == "ops":
        f = _scalar_field(dims, seed)
        out = [torch.empty_like(f) for _ in range(4)]
        return {"case": case, "num": cs.Numerics(dims, _nbc(case)), "f": f, "out": out, "tmp": torch.empty_like(f)}
    q = _flow(case, seed)
    if kind == "walls":
        st = _state(case)
        npex = torch.zeros(dims[0] * dims[1] * dims[2], dtype=torch.int32, device=dev)
        return {"case": case, "stepper": Stepper(dims, _nbc(case), True, st["umf"], st), "q": q, "npex": npex}
    viscous = case.get("viscous", False)
    sv = FusedSolver(dims, _nbc(case), _state(case), viscous=viscous, curvilinear=case.get("curv", False))
    if case.get("f32"):
        sv.set_precision(1)
    if kind == "step":
        return {"case": case, "solver": sv, "q": q}
    # adjoint: the gradient of a loss on the state after the step
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) + 1)
    lam = torch.randn(q.shape, generator=g, device=dev, dtype=torch.float64)
    return {"case": case, "solver": sv, "q": q, "lam": lam, "tape": sv.new_tape(), "dt": 0.5 * sv.time_step(q)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["case"]["kind"]
    if kind == "ops":
        num, f, out, tmp = state["num"], state["f"], state["out"], state["tmp"]
        for axis in range(3):
            num.deriv(axis, f, out[axis])
        num.filter(0, f, out[3])
        num.filter(1, out[3], tmp)
        num.filter(2, tmp, out[3])
        return out
    if kind == "batch":
        state["batch"].replay()
        return state["f"] + state["d"]
    if kind == "step":
        state["solver"].rk4_step(state["q"])
        return state["q"]
    if kind == "walls":
        st = state["stepper"]
        st.rk4_step(state["q"], cfl=0.5)
        cs.wall_condition_update(st.num, state["q"], state["npex"], st.umf)
        return state["q"]
    sv, dt = state["solver"], state["dt"]
    x, lam = state["q"].clone(), state["lam"].clone()
    sv.rk4_step_tape(x, state["tape"], dt=dt)
    sv.rk4_vjp_tape(state["tape"], lam, dt)
    return [x, lam]


def work(case):
    """Compulsory bytes (inputs once, outputs once) and the operations of the
    method itself: 11 a point for a derivative (6 right-hand side, 5 solve),
    22 for a filter pass, and the pointwise arithmetic of the physics."""
    if case["kind"] == "batch":
        n = sum(a * b * c for a, b, c in _batch_dims(case))
        return {"bytes": 40.0 * n, "flops": 99.0 * n}
    n = float(case["nx"] * case["ny"] * case["nz"])
    if case["kind"] == "ops":
        return {"bytes": 40.0 * n, "flops": 99.0 * n}
    visc = case.get("viscous", True) if case["kind"] != "adjoint" else False
    stage = (27 * 11 + 250 if visc else 15 * 11 + 90) + 15
    step = 4.0 * stage + 15 * 22 + 30
    if case["kind"] == "adjoint":
        return {"bytes": 160.0 * n, "flops": 2.5 * step * n}
    return {"bytes": (80.0 + (80.0 if case.get("curv") or case["kind"] == "walls" else 0.0)) * n, "flops": step * n}


# ---------------------------------------------------------------------------
# the same in plain torch, FP64: dense line operators, pointwise physics
# ---------------------------------------------------------------------------
def _interface_rows():
    """The two quasi-disjoint seam rows (own side, far side): rows 8 and 9 of
    R P^-1 Q for the 16-point two-block system."""
    n = 16
    P, Q = np.zeros((n, n)), np.zeros((n, n))
    for i in range(2, n - 2):
        P[i, i - 1:i + 2] = [1 / 3, 1, 1 / 3]
        Q[i, i - 2:i + 3] = [-1 / 36, -7 / 9, 0, 7 / 9, 1 / 36]
    P[0, :2], P[1, :3] = [1, 2], [0.25, 1, 0.25]
    P[-1, -2:], P[-2, -3:] = [2, 1], [0.25, 1, 0.25]
    Q[0, :3], Q[1, :3] = [-2.5, 2, 0.5], [-0.75, 0, 0.75]
    Q[-1, -3:], Q[-2, -3:] = [2.5, -2, -0.5], [-0.75, 0, 0.75]
    R = P.copy()
    R[7, 8] = R[8, 7] = 0.0
    M = R @ np.linalg.solve(P, Q)
    return M[8:10, 8:], M[8:10, :8][:, ::-1]


def _solve(A, B):
    """A^-1 B of a (cyclic) tridiagonal A, refined once with residuals in extended precision."""
    X, i = np.linalg.solve(A, B), np.arange(len(A))
    Xl = X.astype(np.longdouble)
    R = B.astype(np.longdouble)
    for o in (-1, 0, 1):
        R -= A[i, (i + o) % len(A)][:, None].astype(np.longdouble) * Xl[(i + o) % len(A)]
    return (Xl + np.linalg.solve(A, R.astype(np.float64))).astype(np.float64)


def _deriv_matrix(n, seam):
    A, B = np.eye(n), np.zeros((n, n))
    for i in range(n):
        if i > 0:
            A[i, i - 1] = 1 / 3
        if i < n - 1:
            A[i, i + 1] = 1 / 3
        if 2 <= i < n - 2:
            B[i, i - 2:i + 3] = [-1 / 36, -7 / 9, 0, 7 / 9, 1 / 36]
    if not seam:
        A[0, :2], A[1, :3], A[-1, -2:], A[-2, -3:] = [1, 2], [0.25, 1, 0.25], [2, 1], [0.25, 1, 0.25]
        B[0, :3], B[1, :3] = [-2.5, 2, 0.5], [-0.75, 0, 0.75]
        B[-1, -3:], B[-2, -3:] = [-0.5, -2, 2.5], [-0.75, 0, 0.75]
    else:
        own, far = _interface_rows()
        for r in range(2):
            B[r, :8] += own[r]
            B[r, n - 8:] += far[r][::-1]
            B[n - 1 - r, n - 8:] -= own[r][::-1]
            B[n - 1 - r, :8] -= far[r]
    return _solve(A, B)


def _filter_coefficients(M, af):
    """Order-2M centred filter: T(0) = 1, T(pi) = 0 and flat to order 2M at 0."""
    A, r = np.zeros((M + 1, M + 1)), np.zeros(M + 1)
    A[0], r[0] = 1.0, 1.0 + 2.0 * af
    for m in range(1, M):
        A[m], r[m] = np.arange(M + 1.0) ** (2 * m), 2.0 * af
    A[M] = (-1.0) ** np.arange(M + 1)
    return np.linalg.solve(A, r)


def _filter_matrix(n, seam):
    A, B = np.zeros((n, n)), np.zeros((n, n))
    edge = (0.0, 0.2, 0.3, 0.4, 0.45)
    for i in range(n):
        d = 5 if seam else min(i, n - 1 - i, 5)
        A[i, i] = 1.0
        if d == 0:
            B[i, i] = 1.0
            continue
        af = ALPHA_F if d == 5 else min(ALPHA_F, edge[d])
        A[i, (i - 1) % n] += af
        A[i, (i + 1) % n] += af
        a = _filter_coefficients(d, af)
        for m in range(d + 1):
            B[i, (i - m) % n] += 0.5 * a[m]
            B[i, (i + m) % n] += 0.5 * a[m]
    return _solve(A, B)


def _along(M, f, axis):
    """The dense line operator M along `axis` of f [..., nz, ny, nx]."""
    M = torch.as_tensor(M, dtype=torch.float64, device=f.device)
    if axis == 0:
        return (f.reshape(-1, f.shape[-1]) @ M.T).reshape(f.shape)
    if axis == 1:
        return torch.stack([M @ s for s in f.reshape(-1, *f.shape[-2:])]).reshape(f.shape)
    s = f.reshape(-1, f.shape[-3], f.shape[-2] * f.shape[-1])
    return torch.stack([M @ p for p in s]).reshape(f.shape)


class _Flow:
    """The right-hand side and RK4 step of one block, dense operators."""

    def __init__(self, case, viscous):
        self.dims = _dims(case)
        self.faces = case["faces"]
        self.viscous = viscous
        self.umf = _umf(case)
        self.D = [torch.as_tensor(_deriv_matrix(n, c == "P"), device=_device())
                  for n, c in zip(self.dims, self.faces)]
        self.F = [torch.as_tensor(_filter_matrix(n, c == "P"), device=_device())
                  for n, c in zip(self.dims, self.faces)]
        if case.get("curv"):
            self.m, self.J, self.cm = _skewed_metrics(self.dims)
        else:
            self.m = [[1.0 if a == k else 0.0 for k in range(3)] for a in range(3)]
            self.J, self.cm = 1.0, _unit_normals(self.dims)

    @staticmethod
    def primitives(q):
        rho, E = q[0], q[4]
        u = [q[1 + i] / rho for i in range(3)]
        p = (GAM - 1.0) * (E - 0.5 * (q[1] * u[0] + q[2] * u[1] + q[3] * u[2]))
        return u, p, GAM * p / rho

    def time_step(self, q, cfl):
        u, _, c2 = self.primitives(q)
        U = [u[k] + self.umf[k] for k in range(3)]
        one = torch.ones_like(c2)
        rr1 = sum(self.m[a][k] * self.m[a][k] for a in range(3) for k in range(3)) * one
        rr2 = sum(torch.abs(sum(self.m[a][k] * U[k] for k in range(3))) for a in range(3))
        J = self.J * one
        m0 = ((torch.sqrt(c2 * rr1) + rr2) * J.abs()).max()
        m1 = (MU / q[0] * rr1 * J * J).max()
        return float(torch.minimum(cfl / m0, 0.5 / m1))

    def stress(self, u, c2):
        comp = list(u) + [c2]
        g = []
        for f in comp:
            d = [_along(self.D[a], f, a) for a in range(3)]
            g.append([sum(self.m[a][k] * d[a] for a in range(3) if self.curved or a == k) for k in range(3)])
        b0 = MU * self.J
        div = 2.0 / 3.0 * (g[0][0] + g[1][1] + g[2][2])
        tau = [[None] * 3 for _ in range(3)]
        for i in range(3):
            for k in range(3):
                tau[i][k] = b0 * (g[i][k] + g[k][i]) if i != k else b0 * (2.0 * g[i][i] - div)
        b1 = b0 / ((GAM - 1.0) * PRANDTL)
        heat = [b1 * g[3][i] + sum(u[k] * tau[i][k] for k in range(3)) for i in range(3)]
        return tau, heat

    @property
    def curved(self):
        return torch.is_tensor(self.J)

    def rhs(self, q, dtwi=0.0):
        u, p, c2 = self.primitives(q)
        U = [u[k] + self.umf[k] for k in range(3)]
        if self.viscous:
            tau, heat = self.stress(u, c2)
        de, drv = 0.0, []
        for a in range(3):
            m = self.m[a]
            ss = sum(m[k] * U[k] for k in range(3))
            F = [q[0] * ss] + [q[1 + i] * ss + m[i] * p for i in range(3)]
            F.append((q[4] + p) * ss - p * sum(m[k] * self.umf[k] for k in range(3)))
            if self.viscous:
                for i in range(3):
                    F[1 + i] = F[1 + i] - sum(m[k] * tau[i][k] for k in range(3))
                F[4] = F[4] - sum(m[k] * heat[k] for k in range(3))
            d = torch.stack([_along(self.D[a], f, a) for f in F])
            drv.append(d)
            de = de + d
        corr = []
        for a in range(3):
            if self.faces[a] == "P":
                continue
            n = self.dims[a]
            for face in range(2):
                i = face * (n - 1)
                pick = lambda f: f.select(2 - a, i).reshape(-1)
                src = drv[a] if self.faces[a] == "N" else de
                Jf = pick(self.J) if self.curved else self.J
                c = self.characteristic(face, self.cm[a][face], [pick(q[v]) for v in range(5)], pick(p),
                                        [pick(src[v]) for v in range(5)], Jf, self.faces[a] == "W", dtwi)
                corr.append((a, i, c))
        for a, i, c in corr:
            add = torch.zeros_like(de)
            sl = add.select(3 - a, i)
            sl += torch.stack(c).reshape(sl.shape)
            de = de + add
        return de

    def characteristic(self, face, n, q, p, drv, J, wall, dtwi):
        """Change of de at a face point: the amplitudes L (J drv) with the
        incoming acoustic waves removed (non-reflective) or reflected (wall)."""
        rho = q[0]
        a = torch.sqrt(GAM * p / rho)
        u = [q[1 + i] / rho for i in range(3)]
        hv2 = 0.5 * sum(c * c for c in u)
        vn = sum(n[k] * u[k] for k in range(3))
        vs = sum(n[k] * self.umf[k] for k in range(3))
        x = [J * d for d in drv]
        g1 = (GAM - 1.0) / (a * a)
        # acoustic amplitudes: pressure change / c^2 plus, minus rho times the
        # change of the normal velocity over c
        dp = g1 * (hv2 * x[0] - u[0] * x[1] - u[1] * x[2] - u[2] * x[3] + x[4])
        dv = (n[0] * x[1] + n[1] * x[2] + n[2] * x[3] - vn * x[0]) / a
        ch3, ch4 = dp + dv, dp - dv
        ra0 = 1.0 - 2.0 * face
        if wall:
            d3, d4 = torch.zeros_like(ch3), torch.zeros_like(ch4)
            refl = 2.0 * ra0 / a * rho * (dtwi * (vn + vs))
            if face == 0:
                d3 = ch4 + refl - ch3
            else:
                d4 = ch3 + refl - ch4
        else:
            d3 = torch.where(ra0 * (vn + vs + a) > 0, -ch3, torch.zeros_like(ch3))
            d4 = torch.where(ra0 * (vn + vs - a) > 0, -ch4, torch.zeros_like(ch4))
        h = hv2 + a * a / (GAM - 1.0)
        out = [0.5 * (d3 + d4)]
        out += [0.5 * (u[k] * (d3 + d4) + a * n[k] * (d3 - d4)) for k in range(3)]
        out.append(0.5 * (h * (d3 + d4) + a * vn * (d3 - d4)))
        return [c / J for c in out]

    def step(self, q, dt):
        q0, x = q, q
        for k in range(1, 5):
            x = q0 - dt / (5 - k) * self.J * self.rhs(x, 1.0 / dt)
        for a in range(3):
            x = torch.stack([_along(self.F[a], f, a) for f in x])
        return x


def _exact_ops(dims, faces, f):
    nx, ny, nz = dims
    f = f.view(nz, ny, nx)
    d = [_along(_deriv_matrix(n, c == "P"), f, a).reshape(-1) for a, (n, c) in enumerate(zip(dims, faces))]
    for a, (n, c) in enumerate(zip(dims, faces)):
        f = _along(_filter_matrix(n, c == "P"), f, a)
    return d, f.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "ops":
        d, f = _exact_ops(_dims(case), case["faces"], _scalar_field(_dims(case), seed))
        return d + [f]
    if kind == "batch":
        fs, ds = [], []
        for i, dims in enumerate(_batch_dims(case)):
            d, f = _exact_ops(dims, case["faces"], _scalar_field(dims, 1000 * seed + i))
            fs.append(f)
            ds += d
        return fs + ds
    nx, ny, nz = _dims(case)
    q = _flow(case, seed).view(5, nz, ny, nx)
    if kind == "step":
        fl = _Flow(case, case["viscous"])
        return fl.step(q, fl.time_step(q, 0.95)).reshape(-1)
    if kind == "walls":
        fl = _Flow(case, True)
        x = fl.step(q, fl.time_step(q, 0.5))
        # no-slip isothermal walls in the moving frame
        for j in (0, ny - 1):
            rho = x[0, :, j].clone()
            for k in range(3):
                x[1 + k, :, j] = -rho * fl.umf[k]
            x[4, :, j] = rho / (GAM * (GAM - 1.0)) + 0.5 * rho * sum(c * c for c in fl.umf)
        return x.reshape(-1)
    fl = _Flow(case, False)
    g = torch.Generator(device=q.device)
    g.manual_seed(int(seed) + 1)
    lam = torch.randn(q.numel(), generator=g, device=q.device, dtype=torch.float64)
    dt = 0.5 * fl.time_step(q, 0.95)
    q = q.clone().requires_grad_(True)
    x = fl.step(q, dt)
    grad, = torch.autograd.grad(x, q, lam.view_as(x))
    return [x.detach().reshape(-1), grad.reshape(-1)]
