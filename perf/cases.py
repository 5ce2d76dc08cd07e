"""What a program built on this library asks of it, as measurable cases.

A case is one call sequence through the public entry points of
`glemur_amd`, as a user's program makes it:

  relax     upload an initial state, advance it a number of attempted steps
            (one call per step, batches, or batches replayed as a graph) and
            download the positions it reached;
  ensemble  the same for several braids advanced together;
  row       one time-series row of a state on the device: the fields and
            every reduction the reference writes;
  unet      one sample through the warm-start network: the prediction, or
            the loss and every weight gradient;
  train     one epoch over samples resident on the device: the updated
            parameters;
  warm      a warm-started relaxation: prediction, settling steps, checks.

Initial states are braids of twisted blobs in a line-tied or periodic box,
with amplitudes from the seed.  `exact` evaluates the same equations in
64-bit torch from their definitions.
"""
import math
import os

import numpy as np
import torch

import glemur_amd as g
from glemur_amd import warmstart

BOX = (8.0, 8.0, 48.0)
ORIGIN = (-4.0, -4.0, -24.0)
MAX_ERROR = 1e-5
ENSEMBLE_SIZES = ((33, 33, 97), (49, 49, 145), (65, 65, 193))   # the ensemble workload's grids


def listed():
    return [
        # a small FP64 run that looks at every step before the next: call
        # latency and launches (the 33 x 33 x 97 braid of the test configuration)
        {"name": "f64_small_steps", "kind": "relax", "nx": 33, "ny": 33, "nz": 97, "prec": "f64", "api": "step",
         "attempts": 100, "pressure": False, "xp": False, "yp": False, "zp": False, "eps": False, "inertia": False},
        # the same braid as a long unattended run in FP32 with compensation,
        # batches replayed as a graph
        {"name": "f32k_small_graph", "kind": "relax", "nx": 33, "ny": 33, "nz": 97, "prec": "f32k", "api": "graph",
         "attempts": 200, "pressure": False, "xp": False, "yp": False, "zp": False, "eps": False, "inertia": False},
        # the headline braid in FP64
        {"name": "f64_medium", "kind": "relax", "nx": 129, "ny": 129, "nz": 385, "prec": "f64", "api": "run",
         "attempts": 50, "pressure": False, "xp": False, "yp": False, "zp": False, "eps": False, "inertia": False},
        # the headline braid in FP32 with compensation
        {"name": "f32k_medium", "kind": "relax", "nx": 129, "ny": 129, "nz": 385, "prec": "f32k", "api": "run",
         "attempts": 150, "pressure": False, "xp": False, "yp": False, "zp": False, "eps": False, "inertia": False},
        # the largest configured grid, with pressure
        {"name": "f32k_large_pressure", "kind": "relax", "nx": 257, "ny": 257, "nz": 769, "prec": "f32k", "api": "run",
         "attempts": 60, "pressure": True, "xp": False, "yp": False, "zp": False, "eps": False, "inertia": False},
        # a ragged grid with periodic x and y, pressure and a friction profile
        {"name": "f32k_periodic_odd", "kind": "relax", "nx": 61, "ny": 47, "nz": 150, "prec": "f32k", "api": "run",
         "attempts": 100, "pressure": True, "xp": True, "yp": True, "zp": False, "eps": True, "inertia": False},
        # the equation of motion with inertia (the reference's call structure)
        {"name": "f64_inertia", "kind": "relax", "nx": 65, "ny": 65, "nz": 193, "prec": "f64", "api": "run",
         "attempts": 30, "pressure": False, "xp": False, "yp": False, "zp": False, "eps": False, "inertia": True},
        # braids of mixed sizes advanced together, as for training data
        {"name": "ensemble_f32k", "kind": "ensemble", "members": 12, "prec": "f32k", "attempts": 60},
        # a time-series row of the headline grid
        {"name": "row_medium", "kind": "row", "nx": 129, "ny": 129, "nz": 385, "prec": "f32k", "pressure": False},
        # the gradient of one sample on a small network grid
        {"name": "unet_grad_small", "kind": "unet", "nx": 33, "ny": 33, "nz": 97, "part": "grad"},
        # one optimiser step over a mini-batch at the network's own grid
        {"name": "unet_train", "kind": "train", "nx": 65, "ny": 65, "nz": 193, "samples": 8, "batch": 8},
        # a warm start of the headline braid
        {"name": "warm_start", "kind": "warm", "nx": 65, "ny": 65, "nz": 193, "settle": 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["relax"] * 6 + ["ensemble", "row", "unet", "unet", "train", "warm"])
    if kind == "relax":
        while True:
            nx, ny, nz = _log_int(rng, 17, 140), _log_int(rng, 17, 140), _log_int(rng, 40, 400)
            if nx * ny * nz <= 6_500_000:
                break
        inertia = rng.random() < 0.15
        f64 = inertia or rng.random() < 0.4
        return {"kind": "relax", "nx": nx, "ny": ny, "nz": nz, "prec": "f64" if f64 else "f32k",
                "api": rng.choice(["step", "run", "run", "graph"]), "attempts": rng.randint(20, 60),
                "pressure": rng.random() < 0.35, "xp": rng.random() < 0.25, "yp": rng.random() < 0.25,
                "zp": rng.random() < 0.15, "eps": rng.random() < 0.25 and not inertia, "inertia": inertia}
    if kind == "ensemble":
        return {"kind": "ensemble", "members": rng.randint(2, 16), "prec": rng.choice(["f32k", "f32k", "f64"]),
                "attempts": rng.randint(10, 40)}
    if kind == "row":
        return {"kind": "row", "nx": _log_int(rng, 17, 140), "ny": _log_int(rng, 17, 140), "nz": _log_int(rng, 40, 320),
                "prec": rng.choice(["f64", "f32k"]), "pressure": rng.random() < 0.5}
    m = [4 * _log_int(rng, 3, 16) + 1, 4 * _log_int(rng, 3, 16) + 1, 4 * _log_int(rng, 8, 48) + 1]
    if kind == "unet":
        return {"kind": "unet", "nx": m[0], "ny": m[1], "nz": m[2], "part": rng.choice(["forward", "grad"])}
    if kind == "train":
        n = rng.randint(2, 8)
        return {"kind": "train", "nx": m[0], "ny": m[1], "nz": m[2], "samples": n, "batch": n}
    return {"kind": "warm", "nx": m[0], "ny": m[1], "nz": m[2], "settle": rng.randint(5, 30)}


# ------------------------------------------------------------------ inputs
def _amplitudes(seed, member=0):
    return np.random.default_rng((seed, member)).uniform(0.5, 1.5, 6)


def _braid(shape, seed, member=0, peri=(False, False, False)):
    """B0 and the uniform grid of a seeded braid, padded AoS, on the GPU:
    B0 = e_z + sum_k c_k (-(y - y_k), x - x_k, 0) exp(-r_k^2/2 - (z - z_k)^2/4)."""
    amp = _amplitudes(seed, member)
    ax = [torch.arange(-1, n + 1, dtype=torch.float64, device="cuda") * (L / (n - 1)) + O
          for n, L, O in zip(shape, BOX, ORIGIN)]
    x, y, z = ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]
    B = torch.zeros((len(ax[2]), len(ax[1]), len(ax[0]), 3), dtype=torch.float64, device="cuda")
    B[..., 2] = 1.0
    for k in range(6):
        s = 1.0 if k % 2 == 0 else -1.0
        e = torch.exp(-((x - s) ** 2) / 2) * torch.exp(-(y ** 2) / 2) * torch.exp(-((z + 20.0 - 8.0 * k) ** 2) / 4)
        e = e * (s * float(amp[k]))
        B[..., 0] -= y * e
        B[..., 1] += (x - s) * e
        del e
    for axis, on in ((0, peri[2]), (1, peri[1]), (2, peri[0])):   # ghost layers copy the opposite inner layer
        if on:
            n = B.shape[axis]
            B.narrow(axis, 0, 1).copy_(B.narrow(axis, n - 2, 1).clone())
            B.narrow(axis, n - 1, 1).copy_(B.narrow(axis, 1, 1).clone())
    X = torch.empty_like(B)
    X[..., 0], X[..., 1], X[..., 2] = x, y, z
    return B, X


def _displacement(shape, seed, member=0):
    """A smooth displacement of inner points of the size a relaxation makes
    (zero on the boundary), [nz][ny][nx][3]."""
    r = np.random.default_rng((seed, member, 7))
    u = [torch.linspace(0.0, math.pi, n, dtype=torch.float64, device="cuda") for n in shape]
    d = torch.zeros(shape[2], shape[1], shape[0], 3, dtype=torch.float64, device="cuda")
    for c in range(3):
        for _ in range(3):
            m = r.integers(1, 4, 3)
            a = float(r.normal() * (0.12, 0.12, 0.4)[c])
            d[..., c] += a * (torch.sin(float(m[2]) * u[2])[:, None, None] * torch.sin(float(m[1]) * u[1])[None, :, None]
                              * torch.sin(float(m[0]) * u[0])[None, None, :])
    return d


def _displaced(shape, seed, member=0):
    B, X = _braid(shape, seed, member)
    X[1:-1, 1:-1, 1:-1] += _displacement(shape, seed, member)
    return B, X


def _host(t):
    return t.reshape(-1).cpu().numpy()


def _params(shape, case):
    p = g.params_default()
    p.nx, p.ny, p.nz = shape
    p.Lx, p.Ly, p.Lz = BOX
    p.Ox, p.Oy, p.Oz = ORIGIN
    p.nCycle = 10 ** 8
    p.maxError = MAX_ERROR
    p.set_str("jMethod", "Stokes")
    p.set_str("pMethod", "Classic")
    p.zUpdate = True
    p.pressure = bool(case.get("pressure", False))
    p.beta = 0.1
    p.epsilonProf = bool(case.get("eps", False))
    p.xPeri, p.yPeri, p.zPeri = (bool(case.get(k, False)) for k in ("xp", "yp", "zp"))
    p.inertia = bool(case.get("inertia", False))
    p.nu = 0.5
    return g.params_derive(p)


def _prec(case):
    return g.PREC_F64 if case.get("prec") == "f64" else g.PREC_F32K


def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _fine(case):
    return tuple(2 * n - 1 for n in _shape(case))


def _peri(case):
    return tuple(bool(case.get(k, False)) for k in ("xp", "yp", "zp"))


DT0 = 0.01


def _dt0(case):
    """First time step: on the finest grids one of 0.01 leaves the range where the scheme is stable."""
    return 1e-4 if case.get("nz", 0) > 500 else DT0


def _member_shape(i):
    return ENSEMBLE_SIZES[(i * 5 + i // 3) % len(ENSEMBLE_SIZES)]


def _features(B, shape):
    """Network features of a braid: Bx, By, Bz - 1 and the coordinates
    scaled to [-1, 1]; two unused channels."""
    f = torch.zeros(shape[2], shape[1], shape[0], 8, dtype=torch.float64, device="cuda")
    f[..., :3] = B[1:-1, 1:-1, 1:-1]
    f[..., 2] -= 1.0
    for c, (n, view) in enumerate(zip(shape, ((1, 1, -1), (1, -1, 1), (-1, 1, 1)))):
        f[..., 3 + c] = torch.linspace(-1, 1, n, dtype=torch.float64, device="cuda").view(view)
    return f


def prepare(case, seed):
    kind, shape = case["kind"], _shape(case) if "nx" in case else None
    if kind == "relax":
        B, X = _braid(shape, seed, peri=_peri(case))
        return {"case": case, "ctx": g.Context(_params(shape, case), _prec(case)), "B0": _host(B), "xb": _host(X)}
    if kind == "ensemble":
        shapes = [_member_shape(i) for i in range(case["members"])]
        init = [tuple(_host(t) for t in _braid(s, seed, i)) for i, s in enumerate(shapes)]
        return {"case": case, "batch": g.Batch([_params(s, case) for s in shapes], _prec(case)), "init": init}
    if kind == "row":
        B, X = _displaced(shape, seed)
        p = _params(shape, case)
        for name in ("redB2", "redJMax", "redJxB_B2Max", "redEpsilonStar", "redErrB_1ez", "redErrXb_XbAn", "redConvex",
                     "redWedgeMin"):
            setattr(p, name, True)
        c = g.Context(p, _prec(case))
        c.upload(_host(B), _host(X), 0.0, DT0)
        return {"case": case, "ctx": c}
    if kind == "warm":
        B, X = _braid(_fine(case), seed)
        u = g.UNet(*shape)
        warmstart.load(u)
        return {"case": case, "ctx": g.Context(_params(_fine(case), case), g.PREC_F32K), "unet": u, "B0": _host(B),
                "xb": _host(X)}
    if kind == "unet":
        u = g.UNet(*shape)
        warmstart.load(u)
        B, _ = _braid(shape, seed)
        return {"case": case, "unet": u, "feat": _features(B, shape).cpu().numpy(),
                "target": _displacement(shape, seed).cpu().numpy()}
    u = g.UNet(*shape, capacity=case["samples"])
    warmstart.load(u)
    with g.Context(_params(shape, case), g.PREC_F32K) as c:
        for i in range(case["samples"]):
            B, X = _displaced(shape, seed, i)
            c.upload(_host(B), _host(X), 0.0, DT0)
            u.add_sample(c)
    return {"case": case, "unet": u}


def _f32(a):
    """FP32 quantities (weights, gradients, the head's output) that the API
    hands over in doubles."""
    return torch.from_numpy(a).float()


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "relax":
        c, n = state["ctx"], case["attempts"]
        c.upload(state["B0"], state["xb"], 0.0, _dt0(case))
        if case["api"] == "step":
            for _ in range(n):
                st = c.step()
        else:
            st = c.run(max_attempts=n, n_cycle=10 ** 9, batch=min(n, 50), use_graph=case["api"] == "graph")
        return {"xb": c.download(g.FIELD_XB), "attempts": int(st.n_attempt)}
    if kind == "ensemble":
        b, n = state["batch"], case["attempts"]
        for m, (B0, xb) in zip(b.members, state["init"]):
            m.upload(B0, xb, 0.0, DT0)
        st = b.run(max_attempts=n, n_cycle=10 ** 9, batch=n)
        return {"xb": [m.download(g.FIELD_XB) for m in b.members], "attempts": int(sum(s.n_attempt for s in st))}
    if kind == "row":
        c = state["ctx"]
        c.fields()
        r = c.reductions()
        return {k: float(getattr(r, k)) for k in ROW}
    if kind == "warm":
        c, u = state["ctx"], state["unet"]
        c.upload(state["B0"], state["xb"], 0.0, DT0)
        i = u.warm_start(c, settle=case["settle"], force=True)
        return {"xb": c.download(g.FIELD_XB), "mesh_ok": int(i.mesh_ok), "used": int(i.used)}
    u = state["unet"]
    if kind == "unet":
        if case["part"] == "forward":
            return {"y": _f32(u.forward(state["feat"]))}
        loss, grad = u.loss_grad(state["feat"], state["target"])
        return {"loss": _f32(np.array([loss])), "grad": _f32(grad)}
    loss = u.train(1, batch=case["batch"], lr=1e-4, seed=1)
    return {"loss": _f32(np.array([loss])), "params": _f32(u.get_params())}


ROW = ("B2", "JMax", "JxB_B2Max", "JxBMax_JBMax", "epsilonStar", "errB_1ez", "errXb_XbAn", "convex", "wedgeMin")


# -------------------------------------------------------------------- work
def _relax_work(points, padded, f64, attempts, pressure):
    """Bytes of six stages per attempt (positions, B0 and earlier slopes read
    once, the new slope written once; FP32 with compensation 480 B a point,
    FP64 792 B), the state up and the positions down; operations of the
    Jacobian, B, the current, the force and the stage sums."""
    per = 792.0 if f64 else 480.0
    return {"bytes": points * per * attempts + padded * 9 * 8.0,
            "flops": points * attempts * (6 * (180.0 + (150.0 if pressure else 0.0)) + 150.0)}


def _unet_macs(shape):
    p1 = shape[0] * shape[1] * shape[2]
    p2, p3 = (math.prod((n + k - 1) // k for n in shape) for k in (2, 4))
    return 27.0 * (p1 * (8 * 32 + 32 * 32 + 96 * 32 + 32 * 32 + 32 * 3) + p2 * (32 * 64 + 3 * 64 * 64 + 64 * 64 + 64 * 64)
                   + p3 * (64 * 128 + 128 * 128))


def _unet_bytes(shape):
    p1 = shape[0] * shape[1] * shape[2]
    p2, p3 = (math.prod((n + k - 1) // k for n in shape) for k in (2, 4))
    # each activation written once and read once, 16 bits a channel
    return 4.0 * (p1 * (8 + 32 + 96 + 32 + 32 + 8) + p2 * (32 + 64 + 192 + 64 + 64) + p3 * (64 + 128 + 128))


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        w = {"bytes": 0.0, "flops": 0.0}
        for i in range(case["members"]):
            s = _member_shape(i)
            one = _relax_work(math.prod(s), math.prod(n + 2 for n in s), case["prec"] == "f64", case["attempts"], False)
            w = {k: w[k] + one[k] for k in w}
        return w
    s = _shape(case)
    pts, pad = math.prod(s), math.prod(n + 2 for n in s)
    if kind == "relax":
        w = _relax_work(pts, pad, case["prec"] == "f64", case["attempts"], case["pressure"])
        if case["inertia"]:
            w["bytes"] += pts * 600.0 * case["attempts"]
        return w
    if kind == "row":
        f64 = case["prec"] == "f64"
        # positions and B0 in, B, J and the determinant (and the pressure gradient) out, and these in again
        size = 8 if f64 else 4
        return {"bytes": pts * (size * (6 if f64 else 9) + 2.0 * (size * (9 if case["pressure"] else 6) + 8)), "flops": pts * 600.0}
    if kind == "warm":
        f = _fine(case)
        w = _relax_work(math.prod(f), math.prod(n + 2 for n in f), False, case["settle"], False)
        return {"bytes": w["bytes"] + _unet_bytes(s), "flops": w["flops"] + 2 * _unet_macs(s)}
    if kind == "unet":
        n = 3 if case["part"] == "grad" else 1
        return {"bytes": n * _unet_bytes(s) + pts * 8.0 * (11 if n == 1 else 11), "flops": 2.0 * n * _unet_macs(s)}
    n = case["samples"]
    return {"bytes": 3.0 * n * _unet_bytes(s) + 1.42e6 * 4 * 7, "flops": 6.0 * n * _unet_macs(s)}


# ------------------------------------------------------------------- exact
_B = ((0.2,), (3 / 40, 9 / 40), (0.3, -0.9, 1.2), (-11 / 54, 2.5, -70 / 27, 35 / 27),
      (1631 / 55296, 175 / 512, 575 / 13824, 44275 / 110592, 253 / 4096))
_C = (37 / 378, 0.0, 250 / 621, 125 / 594, 0.0, 512 / 1771)
_CS = (2825 / 27648, 0.0, 18575 / 48384, 13525 / 55296, 277 / 14336, 0.25)


def _cross(a, b):
    return torch.stack((a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]))


def _dot(a, b):
    return (a * b).sum(0)


class _Grid:
    """Plain 64-bit evaluation on one grid; fields are [3][nz][ny][nx] with
    one ghost layer (positions two)."""

    def __init__(self, shape, peri, pressure, eps, beta=0.1):
        self.n, self.peri, self.pressure, self.beta = shape, peri, pressure, beta
        self.h = [L / (m - 1) for L, m in zip(BOX, shape)]
        self.eps = 1.0
        if eps:
            f = [1 - 4 * (i - m / 2) / m * (i + 1 - m / 2) / m
                 for i, m in ((torch.arange(m, dtype=torch.float64, device="cuda"), m) for m in shape)]
            self.eps = f[2][:, None, None] * f[1][None, :, None] * f[0][None, None, :]
        # the lattice with two ghost layers (line-tied ghosts and the points beyond them)
        ax = [torch.arange(-2, m + 2, dtype=torch.float64, device="cuda") * h + O
              for m, h, O in zip(shape, self.h, ORIGIN)]
        self.lat = torch.empty((3, len(ax[2]), len(ax[1]), len(ax[0])), dtype=torch.float64, device="cuda")
        self.lat[0], self.lat[1], self.lat[2] = ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]

    def widen(self, x):
        """Inner positions with two ghost layers: the lattice on line-tied
        axes, images shifted by the period on periodic ones."""
        e = self.lat.clone()
        e[:, 2:-2, 2:-2, 2:-2] = x
        for c, axis in ((2, 1), (1, 2), (0, 3)):
            if not self.peri[c]:
                continue
            n, per = self.n[c], BOX[c] + self.h[c]
            lo, hi = e.narrow(axis, n, 2).clone(), e.narrow(axis, 2, 2).clone()
            lo[c] -= per
            hi[c] += per
            e.narrow(axis, 0, 2).copy_(lo)
            e.narrow(axis, n + 2, 2).copy_(hi)
        return e

    @staticmethod
    def _diff(e, axis):
        """Central difference (not divided) along an axis, one layer less on every side."""
        s = [slice(None)] + [slice(1, -1)] * 3
        a, b = list(s), list(s)
        a[axis], b[axis] = slice(2, None), slice(None, -2)
        return e[tuple(a)] - e[tuple(b)]

    def fields(self, x, B0):
        """B with one ghost layer, and J, det, grad p at inner points."""
        e = self.widen(x)
        dr = [self._diff(e, axis) for axis in (3, 2, 1)]
        vol = _dot(dr[0], _cross(dr[1], dr[2]))
        det = vol / (8 * self.h[0] * self.h[1] * self.h[2])
        B = sum(dr[a] * (B0[a] / (2 * self.h[a])) for a in range(3)) / det
        for c, axis in ((0, 3), (1, 2), (2, 1)):   # the normal component is held on line-tied faces
            if not self.peri[c]:
                for side in (0, B.shape[axis] - 1):
                    B[c].narrow(axis - 1, side, 1).copy_(B0[c].narrow(axis - 1, side, 1))
        inner = (slice(None), slice(1, -1), slice(1, -1), slice(1, -1))
        dri = [d[inner] for d in dr]
        C = [_cross(dri[(a + 1) % 3], dri[(a + 2) % 3]) for a in range(3)]
        voli, deti = vol[inner[1:]], det[inner[1:]]
        J = sum(_cross(C[a], self._diff(B, axis)) for a, axis in ((0, 3), (1, 2), (2, 1))) / voli
        gp = None
        if self.pressure:
            # -beta/det sum_l C_l/vol sum_b tr-like second differences: the derivative of beta/det
            p = (slice(None), slice(2, -2), slice(2, -2), slice(2, -2))
            mid = e[p]
            ax = (3, 2, 1)

            def at(*steps):
                s = list(p)
                for a, d in steps:
                    s[ax[a]] = slice(2 + d, e.shape[ax[a]] - 2 + d)
                return e[tuple(s)]

            gp = 0
            for a in range(3):
                N = 4 * _dot(at((a, 1)) - 2 * mid + at((a, -1)), C[a])
                for b in range(3):
                    if b != a:
                        N = N + _dot(at((a, 1), (b, 1)) - at((a, 1), (b, -1)) - at((a, -1), (b, 1)) + at((a, -1), (b, -1)),
                                     C[b])
                gp = gp + N * C[a]
            gp = gp * (-self.beta / deti / voli ** 2)
        return B, J, deti, gp

    def relax(self, x, B0, attempts, dt, inertia=False, nu=0.5):
        """Adaptive Cash-Karp steps from x; the positions and the controller's state."""
        done = 0
        u = torch.zeros_like(x) if inertia else None
        while done < attempts:
            ks, us = [], []
            for n in range(6):
                w = _B[n - 1] if n else ()
                xs = x + sum(b * k for b, k in zip(w, ks)) if n else x
                B, J, det, gp = self.fields(xs, B0)
                k = _cross(J, B[:, 1:-1, 1:-1, 1:-1])
                if inertia:
                    v = u + sum(b * q for b, q in zip(w, us)) if n else u
                    k = dt * det * (k - nu * v)
                    us.append(k - dt * gp if gp is not None else k)
                    ks.append(dt * v)
                else:
                    k = k * (dt * self.eps)
                    ks.append(k - dt * gp if gp is not None else k)
            err = sum((c - cs) * k for c, cs, k in zip(_C, _CS, ks)).abs().max().item()
            if err < MAX_ERROR:
                x = x + sum(c * k for c, k in zip(_C, ks))
                if inertia:
                    u = u + sum(c * q for c, q in zip(_C, us))
            if err > 0:
                dt = dt * (0.9 * MAX_ERROR / err) ** 0.2
            done += 1
        return x

    def padded(self, x):
        return self.widen(x)[:, 1:-1, 1:-1, 1:-1].permute(1, 2, 3, 0).reshape(-1)


def _soa(t):
    return t.permute(3, 0, 1, 2).contiguous()


def _exact_relax(case, shape, B, X, attempts, inertia=False):
    G = _Grid(shape, _peri(case), bool(case.get("pressure", False)), bool(case.get("eps", False)))
    x = G.relax(_soa(X)[:, 1:-1, 1:-1, 1:-1], _soa(B), attempts, _dt0(case), inertia)
    return G.padded(x)


def _exact_row(case, seed):
    shape = _shape(case)
    B0, X = _displaced(shape, seed)
    G = _Grid(shape, (False,) * 3, False, False)
    x = _soa(X)[:, 1:-1, 1:-1, 1:-1]
    B, J, det, _ = G.fields(x, _soa(B0))
    b = B[:, 1:-1, 1:-1, 1:-1]
    jxb, b2, j = _cross(J, b).norm(dim=0), _dot(b, b), J.norm(dim=0)
    w = torch.ones_like(b2)
    for axis in range(3):
        for side in (0, w.shape[axis] - 1):
            w.narrow(axis, side, 1).mul_(0.5)
    out = {"B2": (b2 * det * w).sum() * G.h[0] * G.h[1] * G.h[2], "JMax": j.max(), "JxB_B2Max": (jxb / b2).max(),
           "JxBMax_JBMax": jxb.max() / (j * b2.sqrt()).max()}
    z = b.clone()
    z[2] -= 1.0
    out["errB_1ez"] = (_dot(z, z).sum() / b2.numel()).sqrt()
    p = g.params_default()   # the analytic map's three numbers
    o = G.lat[:, 2:-2, 2:-2, 2:-2]
    f = torch.exp(-(o[0] ** 2 + o[1] ** 2) / p.ar ** 2 - o[2] ** 2 / p.az ** 2) * p.phi1
    an = torch.stack((torch.cos(f) * o[0] + torch.sin(f) * o[1], torch.cos(f) * o[1] - torch.sin(f) * o[0], o[2]))
    out["errXb_XbAn"] = (((x - an) ** 2).sum() / b2.numel()).sqrt()
    i, k = shape[0] // 2, shape[1] // 2
    a, zc = (_dot(J, b) / b2)[:, k, i], x[2, :, k, i]
    dz = zc[:, None] - zc[None, :]
    q = math.sqrt(2.0) * ((a[:, None] - a[None, :]) / torch.where(dz == 0, torch.full_like(dz, math.inf), dz)).abs()
    out["epsilonStar"] = q.max()
    e = G.widen(x)
    p = (slice(None), slice(2, -2), slice(2, -2), slice(2, -2))

    def edge(a, d):
        s = list(p)
        s[3 - a] = slice(2 + d, e.shape[3 - a] - 2 + d)
        return e[tuple(s)] - e[p]

    wedge = torch.full_like(b2, math.inf)
    for su in (-1, 1):
        for sv in (-1, 1):
            uv = _cross(edge(0, su), edge(1, sv))
            for sw in (-1, 1):
                wedge = torch.minimum(wedge, _dot(uv, edge(2, sw)) * (su * sv * sw))
    out["wedgeMin"], out["convex"] = wedge.min(), 1.0 if float(wedge.min()) >= 0 else -1.0
    return {k: float(out[k]) for k in ROW}


_LAYERS = ((8, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128), (192, 64), (64, 64), (96, 32), (32, 32), (32, 3))


def _weights():
    with np.load(os.path.join(os.path.dirname(g.__file__), "data", "unet_braid65x65x193.npz"), allow_pickle=False) as f:
        w = (f["bf16"].astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        return torch.from_numpy(w).cuda(), float(f["scale"][0])


def _conv(a, w, b):
    """3 x 3 x 3 convolution with zero padding: [z][y][x][ci] -> [z][y][x][co]."""
    p = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1, 1, 1))
    nz, ny, nx = a.shape[:3]
    out = b.expand(nz * ny * nx, -1)
    for t in range(27):
        s = p[t // 9:t // 9 + nz, t // 3 % 3:t // 3 % 3 + ny, t % 3:t % 3 + nx].reshape(nz * ny * nx, -1)
        out = out + s @ w[:, t].t().contiguous()
    return out.reshape(nz, ny, nx, -1)


def _pool(a):
    p = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1, 1, 1))
    n = [(m + 1) // 2 for m in a.shape[:3]]
    return sum(p[z:z + 2 * n[0] - 1:2, y:y + 2 * n[1] - 1:2, x:x + 2 * n[2] - 1:2]
               for z in range(3) for y in range(3) for x in range(3)) / 27.0


def _up(a):
    for axis in range(3):
        n = a.shape[axis]
        lo, hi = a.narrow(axis, 0, n - 1), a.narrow(axis, 1, n - 1)
        both = torch.stack((lo, (lo + hi) / 2), axis + 1).flatten(axis, axis + 1)
        a = torch.cat((both, a.narrow(axis, n - 1, 1)), axis)
    return a


def _net(w, feat):
    """The head's output of the three-level network for packed parameters w."""
    at, L = 0, []
    for ci, co in _LAYERS:
        k = w[at:at + co * 27 * ci].reshape(co, 27, ci)
        L.append((k, w[at + co * 27 * ci:at + co * 27 * ci + co]))
        at += co * 27 * ci + co
    r = torch.relu
    a2 = r(_conv(r(_conv(feat, *L[0])), *L[1]))
    a4 = r(_conv(r(_conv(_pool(a2), *L[2])), *L[3]))
    a6 = r(_conv(r(_conv(_pool(a4), *L[4])), *L[5]))
    a8 = r(_conv(r(_conv(torch.cat((_up(a6), a4), 3), *L[6])), *L[7]))
    return _conv(r(_conv(r(_conv(torch.cat((_up(a8), a2), 3), *L[8])), *L[9])), *L[10])


def _loss_grad(w, scale, feat, target):
    w = w.clone().requires_grad_(True)
    loss = ((_net(w, feat) - target / scale) ** 2).mean()
    loss.backward()
    return loss.detach(), w.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        out = []
        for i in range(case["members"]):
            s = _member_shape(i)
            out.append(_exact_relax(case, s, *_braid(s, seed, i), case["attempts"]).cpu().numpy())
        return {"xb": out, "attempts": None}
    shape = _shape(case)
    if kind == "relax":
        if math.prod(shape) * case["attempts"] > 1.5e9:
            return None
        x = _exact_relax(case, shape, *_braid(shape, seed, peri=_peri(case)), case["attempts"], case["inertia"])
        return {"xb": x.cpu().numpy(), "attempts": None}
    if kind == "row":
        return _exact_row(case, seed)
    w, scale = _weights()
    if kind == "warm":
        B, X = _braid(_fine(case), seed)
        f = torch.zeros(shape[2], shape[1], shape[0], 8, dtype=torch.float64, device="cuda")
        f[..., :6] = _features(B, _fine(case))[::2, ::2, ::2, :6]
        X[1:-1, 1:-1, 1:-1] += scale * _up(_net(w, f))
        G = _Grid(_fine(case), (False,) * 3, False, False)
        valid = float(G.fields(_soa(X)[:, 1:-1, 1:-1, 1:-1], _soa(B))[2].min()) > 0   # no settling on a folded mesh
        x = _exact_relax(case, _fine(case), B, X, case["settle"] if valid else 0)
        return {"xb": x.cpu().numpy(), "mesh_ok": None, "used": None}
    if kind == "unet":
        feat = _features(_braid(shape, seed)[0], shape)
        if case["part"] == "forward":
            with torch.no_grad():
                return {"y": (scale * _net(w, feat)).cpu().numpy()}
        loss, grad = _loss_grad(w, scale, feat, _displacement(shape, seed))
        return {"loss": loss.reshape(1).cpu().numpy(), "grad": grad.cpu().numpy()}
    total, grad = 0.0, 0.0
    for i in range(case["samples"]):
        loss, q = _loss_grad(w, scale, _features(_braid(shape, seed, i)[0], shape), _displacement(shape, seed, i))
        total, grad = total + loss, grad + q / case["batch"]
    total = total / case["samples"]
    w = w - 1e-4 * grad / (grad.abs() + 1e-8)   # the first Adam step: m / sqrt(v) after their corrections
    params = torch.cat((w, torch.tensor([scale], dtype=torch.float64, device="cuda")))
    return {"loss": total.reshape(1).cpu().numpy(), "params": params.cpu().numpy()}
