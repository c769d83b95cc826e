"""Performance cases of the plane-wave Maxwell eigensolver: what a program that uses it has it
do, through the Python entry points (``solve_k``, ``solve_k_learned``, ``solve_k_batch``,
``solve_k_periodic``, ``rrule_solve_k``, ``eme.eme``, ``WarmNet.loss_grad``).

The work is mode solving: ε⁻¹ maps in, propagation constants (and, where the call gives them,
gradients and S-matrices) out.  ε⁻¹ is a host array by the interface's nature; the solver
handle (its plans, twiddles and ε⁻¹ on the device) is what a program keeps between calls, so
``prepare`` builds it.  Geometry and frequency come from the seed, spread around each
structure of the repository's benchmark: the Gaussian index bump of the reference's scaling
benchmark, the Si3N4 rectangle, the thin-film LiNbO3 rib, random ridges with rotated tensors,
the two-core coupler of the EME chain and the Bragg grating.

Solves ask for k_tol 1e-10 and eig_tol 1e-8 as the benchmark does.  Cases whose outputs depend
on the eigenvectors to first order (gradients, S-matrices) ask for eig_tol 1e-11, as a
program that differentiates or cascades would.  Eigenvectors themselves are not fetched:
their phase is set by the largest field entry, which mirror-symmetric structures have twice.
"""
import math
import os
import random  # noqa: F401  (draw takes a random.Random)
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("optimode.jl_amd"))

import omx  # noqa: E402
from omx import eme as EME  # noqa: E402
from omx import warmstart as WS  # noqa: E402

OMEGA = 1 / 1.55  # 1/um
SIO2, SIN = 2.085, 3.96
LN = (4.89, 4.57, 4.89)
CELLS = {"gauss": (6.0, 4.0), "rect": (6.0, 4.0), "rib": (8.0, 4.0), "ridge": (6.0, 4.0), "coupler": (8.0, 4.0)}
TOL = dict(k_tol=1e-10, eig_tol=1e-8, max_eigsolves=60, maxiter=300)
TIGHT = dict(k_tol=1e-12, eig_tol=1e-11, max_eigsolves=60, maxiter=300)


def listed():
    return [
        # the reference's scaling benchmark at its smallest grid: a quick look at one mode
        dict(name="gauss_32_1mode", kind="solve", shape="gauss", nx=32, ny=32, nev=1, precision="mixed"),
        # a standard single solve of a few guided modes
        dict(name="rect_128_4modes", kind="solve", shape="rect", nx=128, ny=128, nev=4, precision="mixed"),
        # a cell cut to the structure, not to a power of two
        dict(name="ridge_250x135_3modes", kind="solve", shape="ridge", nx=250, ny=135, nev=3, precision="mixed"),
        # a fine grid with factors of three, many modes, full tensors
        dict(name="ridge_384_12modes", kind="solve", shape="ridge", nx=384, ny=384, nev=12, precision="mixed"),
        # the headline solve from the plain start (any geometry)
        dict(name="rib_256_8modes", kind="solve", shape="rib", nx=256, ny=256, nev=8, precision="mixed"),
        # the headline solve from the learned start (bench.py's default)
        dict(name="rib_256_8modes_learned", kind="learned", shape="rib", nx=256, ny=256, nev=8, precision="mixed"),
        # one cold cross-section of the EME chain: the largest 2D cell and block
        dict(name="coupler_512x256_16modes", kind="solve", shape="coupler", nx=512, ny=256, nev=16, precision="mixed"),
        # a geometry sweep over uneven grids and mode counts in one call
        dict(name="batch_mixed_6", kind="batch", count=6, nmax=256, nevmax=8),
        # Bloch modes of one period of a grating, 3D cell
        dict(name="bragg_128x96x24_4modes", kind="bragg", nx=128, ny=96, nz=24, nev=4),
        # design gradient: solve and pull back cotangents on k and on the eigenvectors
        dict(name="gradient_256_8modes", kind="gradient", shape="rib", nx=256, ny=256, nev=8),
        # a stretch of the EME chain: cold first slice, warm-started ones, overlaps, S-matrix
        dict(name="eme_512x256_16modes", kind="eme", nx=512, ny=256, nev=16, slices=3),
        # one training minibatch of the warm-start network (loss and gradient)
        dict(name="network_batch16", kind="network", hw=64, nev=8, batch=16, bf16=True),
    ]


# --- drawn cases -------------------------------------------------------------------------

def _smooth(lo, hi, step=1):
    """Sizes in [lo, hi] the transforms accept (factors 2, 3 and 5), multiples of step."""
    out = []
    for n in range(lo, hi + 1):
        m = n
        for f in (2, 3, 5):
            while m % f == 0:
                m //= f
        if m == 1 and n % step == 0:
            out.append(n)
    return out


def _near(rng, lo, hi, step=1):
    """A size of _smooth spread over the logarithm of the range."""
    sizes = _smooth(lo, hi, step)
    at = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(sizes, key=lambda n: (abs(math.log(n / at)), n))


def draw(rng):
    kind = rng.choice(["solve"] * 8 + ["learned", "learned", "batch", "batch", "bragg", "bragg", "gradient", "gradient",
                                       "eme", "eme", "network", "network"])
    if kind == "solve":
        shape = rng.choice(["gauss", "rect", "rib", "ridge", "ridge", "coupler"])
        if shape == "gauss":
            n = _near(rng, 32, 256)
            return dict(kind="solve", shape=shape, nx=n, ny=n, nev=rng.choice([1, 1, 2]), precision="mixed")
        # sizes of either parity, the two sides independent within a factor of two or so
        nx = _near(rng, 48, 512)
        ny = _near(rng, max(48, nx // 2), min(384, 2 * nx))
        most = 16 if nx * ny <= 512 * 256 else 12
        fp64 = rng.random() < 0.2
        nev = rng.randint(1, 4 if fp64 else most)
        if fp64:  # the all-FP64 option, for checks: smaller cells
            nx, ny = min(nx, 192), min(ny, 192)
        return dict(kind="solve", shape=shape, nx=nx, ny=ny, nev=nev, precision="fp64" if fp64 else "mixed")
    if kind == "learned":
        return dict(kind="learned", shape="rib", nx=rng.choice([128, 192, 256, 320, 384]), ny=rng.choice([128, 192, 256]),
                    nev=rng.randint(4, 8), precision="mixed")
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(2, 8), nmax=rng.choice([128, 192, 256]), nevmax=rng.randint(4, 8))
    if kind == "bragg":
        return dict(kind="bragg", nx=_near(rng, 48, 128, 2), ny=_near(rng, 48, 96, 2), nz=_near(rng, 8, 24, 2),
                    nev=rng.randint(1, 4))
    if kind == "gradient":
        nx = _near(rng, 64, 256, 2)
        return dict(kind="gradient", shape=rng.choice(["rib", "ridge"]), nx=nx, ny=_near(rng, 64, nx, 2),
                    nev=rng.randint(1, 6))
    if kind == "eme":
        nx = _near(rng, 128, 512, 2)
        return dict(kind="eme", nx=nx, ny=_near(rng, 64, max(64, nx // 2), 2), nev=rng.randint(2, 10), slices=rng.randint(2, 4))
    return dict(kind="network", hw=rng.choice([32, 64]), nev=rng.randint(4, 16), batch=rng.randint(1, 24),
                bf16=rng.random() < 0.5)


# --- structures --------------------------------------------------------------------------

def _axes(n, d, sub):
    """Sub-sample positions of each pixel along one axis: (n, sub), pixel centres -d/2 + i d/n."""
    return -d / 2 + d / n * (np.arange(n)[:, None] + ((np.arange(sub) + 0.5) / sub - 0.5)[None, :])


def _rotated(diag, angles):
    """A symmetric tensor with the given principal values, axes turned about x, y and z."""
    R = np.eye(3)
    for axis, t in enumerate(angles):
        i, j = [(1, 2), (0, 2), (0, 1)][axis]
        Q = np.eye(3)
        Q[i, i] = Q[j, j] = math.cos(t)
        Q[i, j], Q[j, i] = -math.sin(t), math.sin(t)
        R = Q @ R
    return R @ np.diag(diag) @ R.T


def _smoothed(nx, ny, dx, dy, regions, background, sub=4):
    """ε⁻¹ (3, 3, nx, ny) of piecewise-constant tensors with averaged interface pixels: the
    mean of ε⁻¹ along the interface normal, the inverse of the mean ε across it.  regions:
    (mask function of x and y, tensor), earlier ones on top."""
    X = _axes(nx, dx, sub)[:, None, :, None]
    Y = _axes(ny, dy, sub)[None, :, None, :]
    left = np.ones((nx, ny, sub, sub), dtype=bool)
    mean_e, mean_i = np.zeros((nx, ny, 3, 3)), np.zeros((nx, ny, 3, 3))
    tr = np.zeros((nx, ny))
    for mask, eps in regions + [(None, background)]:
        here = left if mask is None else left & np.broadcast_to(mask(X, Y), left.shape)
        f = here.mean(axis=(2, 3))
        left = left & ~here
        mean_e += f[..., None, None] * eps
        mean_i += f[..., None, None] * np.linalg.inv(eps)
        tr += f * np.trace(eps)
    gx, gy = np.gradient(tr)
    gx, gy = gx * nx / dx, gy * ny / dy
    g = np.sqrt(gx * gx + gy * gy)
    n = np.stack([gx, gy, np.zeros_like(g)], -1) / np.where(g > 0, g, 1.0)[..., None]
    P = n[..., :, None] * n[..., None, :]
    B = np.linalg.inv(mean_e)
    ei = B + P @ (mean_i - B) @ P
    ei = 0.5 * (ei + np.swapaxes(ei, -1, -2))
    return np.ascontiguousarray(np.moveaxis(ei, (-2, -1), (0, 1)))


def _iso(e):
    return e * np.eye(3)


def _structure(shape, nx, ny, r):
    """ε⁻¹ of a structure on its cell, its dimensions drawn from r."""
    dx, dy = CELLS[shape]
    if shape == "gauss":
        w, h, e = r.uniform(0.9, 1.1), r.uniform(0.55, 0.65), r.uniform(4.0, 4.4)
        x, y = _axes(nx, dx, 1), _axes(ny, dy, 1)
        eps = 2.1 + (e - 2.1) * np.exp(-(x / w) ** 2 - (y.T / h) ** 2)
        return np.ascontiguousarray(np.eye(3)[:, :, None, None] / eps)
    if shape == "rect":
        w, h = r.uniform(1.5, 1.7), r.uniform(0.65, 0.75)
        core = [(lambda X, Y: (abs(X) <= w / 2) & (abs(Y) <= h / 2), _iso(SIN))]
        return _smoothed(nx, ny, dx, dy, core, _iso(SIO2))
    if shape == "coupler":
        gap, w1, w2 = r.uniform(0.3, 1.5), r.uniform(0.8, 1.0), r.uniform(1.0, 1.2)
        return _coupler(nx, ny, gap, w1, w2)
    if shape == "rib":
        top, film = r.uniform(1.0, 1.4), r.uniform(0.56, 0.64)
        slab, slope = film * r.uniform(0.45, 0.55), math.tan(math.radians(r.uniform(57.0, 65.0)))
        ln = np.diag(LN)
        regions = [(lambda X, Y: (Y >= slab) & (Y <= film) & (abs(X) <= top / 2 + (film - Y) / slope), ln),
                   (lambda X, Y: (Y >= 0) & (Y < slab) & (X == X), ln), (lambda X, Y: (Y < 0) & (X == X), _iso(SIO2))]
        return _smoothed(nx, ny, dx, dy, regions, _iso(1.0))
    # ridge: top width, height, sidewall and a core tensor with turned axes on SiO2 in air
    w, h = r.uniform(1.2, 2.2), r.uniform(0.5, 0.8)
    slope = math.tan(math.radians(r.uniform(60.0, 88.0)))
    e = r.uniform(3.9, 4.8)
    core = _rotated((e, e * r.uniform(0.94, 0.98), e), [r.uniform(-0.4, 0.4) for _ in range(3)])
    regions = [(lambda X, Y: (Y >= 0) & (Y <= h) & (abs(X) <= w / 2 + (h - Y) / slope), core),
               (lambda X, Y: (Y < 0) & (X == X), _iso(SIO2))]
    return _smoothed(nx, ny, dx, dy, regions, _iso(1.0))


def _coupler(nx, ny, gap, w1, w2):
    dx, dy = CELLS["coupler"]
    x1, x2 = -(gap + w1) / 2, (gap + w2) / 2
    cores = [(lambda X, Y: (abs(X - x1) <= w1 / 2) & (abs(Y) <= 0.4), _iso(SIN)),
             (lambda X, Y: (abs(X - x2) <= w2 / 2) & (abs(Y) <= 0.4), _iso(SIN))]
    return _smoothed(nx, ny, dx, dy, cores, _iso(SIO2))


def _problems(case, seed):
    """The eigenproblems of a case: dicts with the cell, grid, ε⁻¹, ω and mode count."""
    r = np.random.default_rng([seed, 17])
    kind = case["kind"]
    if kind in ("solve", "learned", "gradient"):
        ei = _structure(case["shape"], case["nx"], case["ny"], r)
        return [dict(cell=CELLS[case["shape"]], n=(case["nx"], case["ny"]), ei=ei, omega=OMEGA * r.uniform(0.97, 1.03),
                     nev=case["nev"])]
    if kind == "batch":
        sizes = [n for n in (128, 192, 256) if n <= case["nmax"]]
        out = []
        for i in range(case["count"]):
            n = sizes[i % len(sizes)]
            out.append(dict(cell=CELLS["ridge"], n=(n, n), ei=_structure("ridge", n, n, r), omega=r.uniform(0.6, 0.9),
                            nev=int(4 + i * (case["nevmax"] - 4) // max(1, case["count"] - 1))))
        return out
    if kind == "bragg":
        d = (4.0, 3.0, 0.45)
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        x, y, z = (_axes(m, s, 1)[:, 0] for m, s in zip((nx, ny, nz), d))
        w = r.uniform(0.9, 1.1) * (1 + r.uniform(0.4, 0.5) * np.cos(2 * np.pi * z / d[2]))
        eps = 2.1 + 1.9 * np.exp(-(x[:, None, None] / w) ** 2 - (y[None, :, None] / r.uniform(0.38, 0.44)) ** 2)
        return [dict(cell=d, n=(nx, ny, nz), ei=np.ascontiguousarray(np.eye(3)[:, :, None, None, None] / eps),
                     omega=0.5 * r.uniform(0.98, 1.02), nev=case["nev"])]
    # eme: neighbouring cross-sections of the taper
    s0 = r.uniform(0.05, 0.8)
    return [dict(cell=CELLS["coupler"], n=(case["nx"], case["ny"]), omega=OMEGA, nev=case["nev"],
                 ei=_coupler(case["nx"], case["ny"], 0.3 + 1.2 * s, 0.8 + 0.4 * s, 1.2 - 0.4 * s))
            for s in (s0 + 0.005 * i for i in range(case["slices"]))]


def _network(case, seed):
    """Parameters of a network in training and one minibatch."""
    hw, nev, B = case["hw"], case["nev"], case["batch"]
    r = np.random.default_rng([seed, 23])
    p = []
    for ci, co in ((7, 16), (16, 32), (32, 32), (64, 32), (48, 32), (32, 4 * nev)):
        p += [r.standard_normal(co * ci * 9) * math.sqrt(2 / (9 * ci)), 0.02 * r.standard_normal(co)]
    p += [r.standard_normal(nev * 32) * math.sqrt(1 / 32), 0.02 * r.standard_normal(nev)]
    x = r.standard_normal((B, 7, hw, hw))
    tf, tk = r.standard_normal((B, 4 * nev, hw, hw)), r.standard_normal((B, nev))
    return tuple(a.astype(np.float32) for a in (np.concatenate(p), x, tf, tk))


# --- the calls ---------------------------------------------------------------------------

def _grid(p):
    return omx.Grid3(*p["cell"], *p["n"]) if len(p["n"]) == 3 else omx.Grid(*p["cell"], *p["n"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "network":
        p, x, tf, tk = _network(case, seed)
        net = WS.WarmNet(case["hw"], case["nev"], bf16=case["bf16"])
        net.params = p
        return dict(kind=kind, net=net, x=x, tf=tf, tk=tk)
    ps = _problems(case, seed)
    if kind == "batch":
        return dict(kind=kind, problems=[dict(grid=_grid(p), epsinv=p["ei"], omega=p["omega"], nev=p["nev"], **TOL)
                                         for p in ps])
    solver = omx.HIPSolver(precision=case.get("precision", "mixed"))
    grid = _grid(ps[0])
    solver.handle(grid, ps[0]["ei"])
    state = dict(kind=kind, solver=solver, grid=grid, ei=ps[0]["ei"], omega=ps[0]["omega"], nev=ps[0]["nev"])
    if kind == "learned":
        state["start"] = WS.LearnedStart.load(os.path.join(WS.DATA_DIR, "warmnet_tfln256.npz"))
    elif kind == "eme":
        state["cells"] = [p["ei"] for p in ps]
    elif kind == "gradient":
        # an objective on the modes: k, and overlaps with given vectors
        r = np.random.default_rng([seed, 29])
        c = r.standard_normal((ps[0]["nev"], 4 * grid.N)).view(np.complex128)
        state["c"] = c / np.linalg.norm(c, axis=1)[:, None]
    return state


def run(state):
    kind = state["kind"]
    if kind == "network":
        loss, grad = state["net"].loss_grad(state["x"], state["tf"], state["tk"])
        return {"loss": loss, "grad": grad}
    if kind == "batch":
        return {"k": [q["kmags"] for q in omx.solve_k_batch(state["problems"])]}
    omega, ei, grid, solver, nev = (state[k] for k in ("omega", "ei", "grid", "solver", "nev"))
    if kind == "solve":
        return {"k": omx.solve_k(omega, ei, grid, solver, nev=nev, fetch_evecs=False, **TOL)[0]}
    if kind == "learned":
        return {"k": WS.solve_k_learned(omega, ei, grid, solver, state["start"], nev=nev, fetch_evecs=False, **TOL)[0]}
    if kind == "bragg":
        return {"k": omx.solve_k_periodic(omega, ei, grid.Dz, grid, solver, nev=nev, fetch_evecs=False, **TOL)[0]}
    if kind == "eme":
        cells = state["cells"]
        res = EME.eme(cells, [1.0] * len(cells), omega, grid, solver, nev=nev, **TIGHT)
        return {"k": list(res.kmags), "S": res.S.S}
    # gradient of sum_j k_j + |<c_j, ev_j>|^2 with respect to ω and ε⁻¹
    (k, ev), pullback = omx.rrule_solve_k(omega, ei, grid, solver, nev=nev, **TIGHT)
    evbar = [2 * c * np.vdot(c, v) for c, v in zip(state["c"], ev)]
    _, wbar, eibar, _, _ = pullback((np.ones(nev), evbar))
    return {"k": k, "omegabar": wbar, "epsinvbar": eibar}


def work(case):
    """Per mode: 12 applications of the operator and of its preconditioner (one eigenpair at
    its own k from a start block, to these tolerances), each reading and writing one
    single-precision vector of two components per pixel and reading ε⁻¹ once, with three
    forward and three inverse transforms; gradients add as many for the linear solve in double
    precision.  ε⁻¹ in and the results out once.  The network: its convolutions forward and
    twice backward, parameters, inputs and targets read once, the gradient written once."""
    if case["kind"] == "network":
        hw, nev, B = case["hw"], case["nev"], case["batch"]
        dims = ((7, 16, 1), (16, 32, 2), (32, 32, 4), (64, 32, 2), (48, 32, 1), (32, 4 * nev, 1))
        par = sum(ci * co * 9 + co for ci, co, _ in dims) + 33 * nev
        macs = sum(ci * co * 9 * (hw // q) ** 2 for ci, co, q in dims)
        return {"bytes": 4.0 * (2 * par + B * ((7 + 4 * nev) * hw * hw + nev)), "flops": 6.0 * B * macs}
    kind = case["kind"]
    if kind == "batch":
        sizes = [n for n in (128, 192, 256) if n <= case["nmax"]]
        todo = [(sizes[i % len(sizes)] ** 2, int(4 + i * (case["nevmax"] - 4) // max(1, case["count"] - 1)))
                for i in range(case["count"])]
    else:
        N = case["nx"] * case["ny"] * case.get("nz", 1)
        todo = [(N, case["nev"])] * (case["slices"] if kind == "eme" else 1)
    b = f = 0.0
    for N, nev in todo:
        vec = 16.0 * N
        one = 2 * (2 * vec + 24.0 * N)
        flops = 2 * 6 * 5.0 * N * math.log2(N)
        b += 12 * nev * one + 72.0 * N
        f += 12 * nev * flops
        if kind == "gradient":
            b += 12 * nev * 2 * one + 72.0 * N
            f += 12 * nev * flops
    return {"bytes": b, "flops": f}


# --- values in 64 bits, by plain torch -----------------------------------------------------

class _Curl:
    """M(k) on coefficient vectors (m, 2, *n) of the two transverse plane-wave directions:
    curl, transform, ε⁻¹, transform back, curl; and an approximate inverse by the reverse
    path with the mean permittivity."""

    def __init__(self, p, dev):
        self.dims = tuple(range(-len(p["n"]), 0))
        self.e = torch.as_tensor(p["ei"], device=dev)
        self.ave = 3.0 / (self.e[0, 0] + self.e[1, 1] + self.e[2, 2])
        g = [torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=dev) / d for n, d in zip(p["n"], p["cell"])]
        g = list(torch.meshgrid(*g, indexing="ij"))
        self.gx, self.gy, self.gz = g + [torch.zeros_like(g[0])] * (3 - len(g))

    def basis(self, k):
        wx, wy, wz = -self.gx, -self.gy, k - self.gz
        w = torch.sqrt(wx ** 2 + wy ** 2 + wz ** 2)
        rho = torch.sqrt(wx ** 2 + wy ** 2)
        safe = torch.where(rho > 0, rho, torch.ones_like(rho))
        n = torch.stack([torch.where(rho > 0, -wy / safe, 0 * rho), torch.where(rho > 0, wx / safe, 1 + 0 * rho), 0 * rho])
        m = torch.linalg.cross(n, torch.stack([wx, wy, wz]), dim=0) / w
        return n, m, w

    def M(self, k, X):
        n, m, w = self.basis(k)
        D = torch.fft.fftn((X[:, 1:] * m - X[:, :1] * n) * w, dim=self.dims)
        E = torch.fft.ifftn(torch.stack([(self.e[a] * D).sum(1) for a in range(3)], 1), dim=self.dims)
        return torch.stack([-(E * n).sum(1) * w, (E * m).sum(1) * w], 1)

    def P(self, k, X):
        n, m, w = self.basis(k)
        E = torch.fft.ifftn((X[:, :1] * n - X[:, 1:] * m) / w, dim=self.dims)
        D = torch.fft.fftn(E * self.ave, dim=self.dims)
        return torch.stack([(D * n).sum(1) / w, -(D * m).sum(1) / w], 1)


def _orth(S):
    """An orthonormal basis of the rows of S (twice, dropping what is dependent)."""
    for _ in range(2):
        S = S / torch.linalg.norm(S, dim=1, keepdim=True)
        lam, U = torch.linalg.eigh((S.conj() @ S.T).cpu())
        keep = lam > 1e-12 * lam[-1]
        T = (U[:, keep] / torch.sqrt(lam[keep])).to(S.device)
        S = T.T @ S
    return S


def _lowest(A, k, X, count, tol, rounds=400):
    """The lowest eigenpairs of M(k): a block method on [X, P R, previous step], until the
    first `count` residuals are below tol.  X (m, 2, *n) is the start and the result."""
    shape, m, old = X.shape, X.shape[0], None
    X = _orth(X.reshape(m, -1))
    for it in range(rounds):
        AX = A.M(k, X.reshape(shape)).reshape(m, -1)
        lam, U = torch.linalg.eigh((X.conj() @ AX.T).cpu())
        U = U.T.contiguous().to(X.device)
        X, AX = U @ X, U @ AX
        lam = lam.to(X.device)
        R = AX - lam[:, None] * X
        if float(torch.linalg.norm(R[:count], dim=1).max()) < tol:
            break
        W = A.P(k, R.reshape(shape)).reshape(m, -1)
        S = torch.cat([X, W] + ([old] if old is not None else []))
        new = S[m:] - (S[m:] @ X.conj().T) @ X
        Q = torch.cat([X, _orth(new - (new @ X.conj().T) @ X)])
        AQ = A.M(k, Q.reshape(-1, *shape[1:])).reshape(Q.shape)
        _, V = torch.linalg.eigh((Q.conj() @ AQ.T).cpu())
        V = V[:, :m].T.contiguous().to(Q.device)
        old = V[:, m:] @ Q[m:]
        X = V @ Q
        X = _orth(X) if it % 10 == 9 else X
    return lam, X.reshape(shape)


def _exact_k(p):
    """k of each of the nev lowest bands at ω: Newton on ω²(k) = ω² per band."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    A = _Curl(p, dev)
    w2 = p["omega"] ** 2
    k = p["omega"] * math.sqrt(1.0 / min(float(p["ei"][a, a].min()) for a in range(3)))
    g = torch.Generator().manual_seed(1)
    nev = p["nev"]
    X = torch.randn((nev + 4, 2) + tuple(p["n"]), generator=g, dtype=torch.complex128).to(dev)
    X = A.P(k, X)
    lam, X = _lowest(A, k, X, nev, 1e-4)
    out = []
    for j in range(nev):
        for step in range(20):
            lam, X = _lowest(A, k, X, j + 1, 1e-7 if step else 1e-4)
            v = X[j:j + 1]
            d = 1e-4
            up, dn = ((v.conj() * A.M(k + s, v)).sum().real for s in (d, -d))
            f, slope = float(lam[j]) - w2, float(up - dn) / (2 * d)
            if step and abs(f) < 1e-12:
                break
            k -= f / slope
        out.append(k)
    return np.array(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "network":
        return _exact_network(case, seed)
    ps = _problems(case, seed)
    if sum(int(np.prod(p["n"])) * p["nev"] for p in ps) > 300_000:
        return None  # over 20 s
    k = [_exact_k(p) for p in ps]
    if kind == "batch":
        return {"k": k}
    if kind == "eme":
        return {"k": k, "S": None}
    if kind == "gradient":
        return {"k": k[0], "omegabar": None, "epsinvbar": None}
    return {"k": k[0]}


def _exact_network(case, seed):
    p, x, tf, tk = (torch.as_tensor(a, dtype=torch.float64) for a in _network(case, seed))
    p.requires_grad_(True)
    F, at = torch.nn.functional, [0]
    nev = case["nev"]

    def take(*shape):
        n = math.prod(shape)
        at[0] += n
        return p[at[0] - n:at[0]].reshape(shape)

    def conv(v, co):
        W = take(co, v.shape[1], 3, 3)
        return F.conv2d(v, W, take(co), padding=1)

    def up(v):
        return v.repeat_interleave(2, 2).repeat_interleave(2, 3)

    a1 = torch.relu(conv(x, 16))
    a2 = torch.relu(conv(F.avg_pool2d(a1, 2), 32))
    a3 = torch.relu(conv(F.avg_pool2d(a2, 2), 32))
    a4 = torch.relu(conv(torch.cat([up(a3), a2], 1), 32))
    a5 = torch.relu(conv(torch.cat([up(a4), a1], 1), 32))
    y = conv(a5, 4 * nev)
    W = take(nev, 32)
    k = a3.mean((2, 3)) @ W.T + take(nev)
    loss = ((y - tf) ** 2).mean() + ((k - tk) ** 2).mean()
    loss.backward()
    return {"loss": loss.detach(), "grad": p.grad}
