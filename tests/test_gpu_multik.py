"""The shared-subspace FP32 phase of solve_k against the per-band form on the same problems:
grids at the edges of its tiles (odd sizes, odd pixel counts, sizes that leave partial row and
column blocks), the smallest and the widest blocks, every kind of start, and batches.

Both forms end in the same FP64 refinement with |change of w^2| <= k_tol = 1e-11, so k agrees
to k_tol / (slope k) <= 1e-11 / (2 * 0.3 * 0.3) < 6e-11; 2e-10 allows for both sides."""
import ctypes
import time

import numpy as np
import pytest

import omx
from omx import geometry as G

pytestmark = pytest.mark.gpu
W0 = 1 / 1.55
KW = dict(k_tol=1e-11, eig_tol=1e-9, max_eigsolves=60, maxiter=300, return_info=True)


def _eps(nx, ny, seed=0):
    """A ridge whose core has every tensor entry, averaged linearly at the interface."""
    r = np.random.default_rng(seed)
    a = r.uniform(-0.3, 0.3, 3)
    Q, _ = np.linalg.qr(np.eye(3) + np.array([[0, a[0], a[1]], [-a[0], 0, a[2]], [-a[1], -a[2], 0]]))
    core = Q @ np.diag([4.2, 4.0, 4.2]) @ Q.T
    g = omx.Grid(6.0, 4.0, nx, ny)
    return g, G.ridge_waveguide(g, 1.5 + 0.1 * seed, 0.6, 75.0, core, backend="gpu")


SHARED = dict(shared=1, per_band=0, redone=0)
PER_BAND = dict(shared=0, per_band=1, redone=0)
REDONE = dict(shared=0, per_band=1, redone=1)


def _solve(g, ei, nev, multik, took=None, solver=None, **kw):
    """solve_k with the option ``multik``; a solve that the shared search space does not finish
    ends in the per-band form, so what is compared with that form has to say which one it took."""
    s = omx.HIPSolver() if solver is None else solver
    s.options["multik"] = float(multik)
    res = omx.solve_k(W0, ei, g, s, nev=nev, **{**KW, **kw})
    assert omx.solve_phases() == ((SHARED if multik else PER_BAND) if took is None else took)
    return res


@pytest.mark.parametrize("nx,ny,nev", [(16, 12, 1), (12, 18, 2), (27, 25, 3), (40, 30, 6), (64, 64, 13), (135, 81, 4),
                                       (100, 48, 7), (128, 96, 16), (50, 250, 5), (256, 128, 15)])
def test_matches_the_per_band_form(nx, ny, nev):
    print(f"multik {nx}x{ny} nev {nev}", flush=True)
    g, ei = _eps(nx, ny)
    k0, ev0, i0 = _solve(g, ei, nev, 0)
    k1, ev1, i1 = _solve(g, ei, nev, 1)
    assert i0["converged"] == i1["converged"] == 1
    assert np.max(np.abs(k1 / k0 - 1)) < 2e-10
    for j in range(nev):
        # bands closer than 1e-4 share a subspace; the others match one by one
        near = [i for i in range(nev) if abs(k0[i] - k0[j]) < 1e-4]
        w = sum(abs(np.vdot(ev0[i], ev1[j])) ** 2 for i in near)
        assert w > 1 - 1e-9


def test_degenerate_bands():
    """A square core: the two lowest bands are degenerate by symmetry."""
    print("multik degenerate", flush=True)
    g = omx.Grid(4.0, 4.0, 48, 48)
    ei = G.rect_waveguide(g, w=1.0, h=1.0)
    k0, _, _ = _solve(g, ei, 4, 0)
    k1, ev, _ = _solve(g, ei, 4, 1)
    assert abs(k0[0] - k0[1]) < 1e-9
    assert np.max(np.abs(k1 / k0 - 1)) < 2e-10
    # the pair is handed over as orthogonal vectors at one k.  Split by 4e-10 in w^2, less than
    # eig_tol, the residuals alone would admit any overlap; what the refinement may turn is
    # its own Rayleigh-Ritz rounding, 1e-16 |M| over the splitting of 4e-10 with |M| of 100
    c = abs(np.vdot(ev[0], ev[1]))
    print(f"  overlap of the pair {c:.1e}", flush=True)
    assert c < 1e-4


def test_a_solve_the_shared_space_gives_up_is_done_per_band():
    """Two iterations never converge: the per-band form then has to give what it gives alone."""
    print("multik give-up", flush=True)
    g, ei = _eps(64, 48)
    s = omx.HIPSolver()
    s.options["multik_maxit"] = 2.0
    k1, _, i1 = _solve(g, ei, 4, 1, took=REDONE, solver=s)
    k0, _, i0 = _solve(g, ei, 4, 0)
    assert i0["converged"] == i1["converged"] == 1
    assert np.max(np.abs(k1 / k0 - 1)) < 2e-10


def test_a_block_that_loses_rank_ends_its_solve_only():
    """A start block of zeros on a grid too small for guard columns leaves the shared search
    space empty: its blocks have no rank.  That is not an error of the call, which then does
    what the per-band form does with such a start, and the handle goes on."""
    print("multik lost rank", flush=True)
    g, ei = _eps(5, 5)
    nev = 16  # 3 nev = 48 of 50 unknowns
    zero = np.zeros((nev, 2 * g.N), dtype=np.complex128)
    ends = []
    for multik in (0, 1):
        s = omx.HIPSolver()
        s.options["multik"] = float(multik)
        try:
            ends.append(omx.solve_k(W0, ei, g, s, nev=nev, Hguess=zero, kguess=1.0, **KW)[0])
        except omx.OmxError as e:
            ends.append(e.status)
        print(f"  multik {multik}: {ends[-1]}, {omx.solve_phases()}", flush=True)
    assert omx.solve_phases()["redone"] == 1 and omx.solve_phases()["shared"] == 0
    if isinstance(ends[0], int):
        assert ends[1] == ends[0]
    else:
        assert np.max(np.abs(ends[1] / ends[0] - 1)) < 2e-10
    k0 = _solve(g, ei, 3, 0)[0]
    assert np.max(np.abs(_solve(g, ei, 3, 1, solver=s)[0] / k0 - 1)) < 2e-10


def test_every_start_reaches_the_same_bands():
    print("multik starts", flush=True)
    g, ei = _eps(90, 64)
    nev = 4
    k0, ev, _ = _solve(g, ei, nev, 0)
    n2 = 2 * g.N
    full = np.stack(ev)
    r = np.random.default_rng(1)
    noisy = full + 0.05 * r.standard_normal((nev, 2 * n2)).view(np.complex128) / np.sqrt(n2)
    for kw in (dict(kguess=1.01 * k0[0], Hguess=noisy), dict(kguess=0.99 * k0, Hguess=noisy, band_guess=True),
               dict(Hguess=noisy[:2]), dict(kguess=k0[:1])):
        k1, _, info = _solve(g, ei, nev, 1, **kw)
        assert info["converged"] == 1
        assert np.max(np.abs(k1 / k0 - 1)) < 2e-10
    low = np.zeros((nev, 2, 16, 16), dtype=np.complex128)
    sx, sy = np.r_[0:8, 90 - 8:90], np.r_[0:8, 64 - 8:64]
    for j in range(nev):
        low[j] = full[j].reshape((2, 90, 64), order="F")[:, sx][:, :, sy]
    rows = low.transpose(0, 3, 2, 1).reshape(nev, -1)
    k1, _, _ = _solve(g, ei, nev, 1, kguess=k0[:1], Hguess=rows, guess_hw=16)
    assert np.max(np.abs(k1 / k0 - 1)) < 2e-10
    s = omx.HIPSolver(warm_start=True)
    omx.solve_k(0.99 * W0, ei, g, s, nev=nev, **KW)
    assert omx.solve_phases() == SHARED
    k1, _, _ = omx.solve_k(W0, ei, g, s, nev=nev, **KW)
    assert omx.solve_phases() == SHARED
    assert np.max(np.abs(k1 / k0 - 1)) < 2e-10


def test_batch_on_an_odd_grid():
    """Problems of one launch group with their own eps^-1, omega and mode count, on a grid whose
    pixel count is odd (the fields' strides)."""
    print("multik batch", flush=True)
    probs, refs = [], []
    for i, nev in enumerate((3, 6, 1)):
        g, ei = _eps(45, 75, seed=i)
        probs.append(dict(grid=g, epsinv=ei, omega=W0 * (1 + 0.02 * i), nev=nev, k_tol=1e-11, eig_tol=1e-9, maxiter=300))
        s = omx.HIPSolver()
        s.options["multik"] = 0.0
        refs.append(omx.solve_k(probs[-1]["omega"], ei, g, s, nev=nev, **KW)[0])
    res = omx.solve_k_batch(probs)
    assert omx.solve_phases() == dict(shared=3, per_band=0, redone=0)
    for q, k0 in zip(res, refs):
        assert q["status"] == 0
        assert np.max(np.abs(q["kmags"] / k0 - 1)) < 2e-10


def test_a_batch_redoes_only_the_problems_left_undone():
    """A problem whose top bands do not propagate at its omega converges in no form, one that
    asks for a residual below rounding not in the refinement: the others of their launch group
    keep the shared search space's results, at the cost of those alone."""
    print("multik batch with problems that fail", flush=True)
    g, ei = _eps(64, 48)
    good = [dict(grid=g, epsinv=ei, omega=W0 * f, nev=nev, k_tol=1e-10, eig_tol=1e-8, maxiter=300)
            for f, nev in ((1.0, 4), (1.05, 3), (0.95, 5))]
    refs = [omx.solve_k(q["omega"], ei, g, omx.HIPSolver(), nev=q["nev"], k_tol=1e-10, eig_tol=1e-8, maxiter=300)[0]
            for q in good]
    below = dict(good[0], omega=0.05, nev=8, max_eigsolves=8, maxiter=40)
    exact = dict(good[1], eig_tol=1e-17, max_eigsolves=8)
    for bad in ([below], [exact], [below, exact]):
        res = omx.solve_k_batch(good[:1] + bad + good[1:])
        took = omx.solve_phases()
        print(f"  {len(bad)} of them: status {[q['status'] for q in res]}, {took}", flush=True)
        assert took == dict(shared=3, per_band=len(bad), redone=len(bad))
        assert all(q["status"] == omx._lib.OMX_ERR_NOT_CONVERGED for q in res[1:1 + len(bad)])
        for q, k0 in zip(res[:1] + res[1 + len(bad):], refs):
            assert q["status"] == 0 and q["info"]["converged"] == 1
            assert np.max(np.abs(q["kmags"] / k0 - 1)) < 2e-9  # k_tol / (2 * 0.3 * 0.3), both sides


def test_a_batch_redone_whole():
    """Two iterations an eigensolve allow the shared search space sixteen, too few for either
    problem, and the per-band form two per Newton step, which it makes do with."""
    print("multik batch redone", flush=True)
    g, ei = _eps(64, 48)
    probs = [dict(grid=g, epsinv=ei, omega=W0 * f, nev=nev, k_tol=1e-10, eig_tol=1e-8, maxiter=2, max_eigsolves=60)
             for f, nev in ((1.0, 4), (1.05, 3))]
    res = omx.solve_k_batch(probs)
    assert omx.solve_phases() == dict(shared=0, per_band=2, redone=2)
    for p, q in zip(probs, res):
        k0 = omx.solve_k(p["omega"], ei, g, omx.HIPSolver(), nev=p["nev"], k_tol=1e-10, eig_tol=1e-8, maxiter=300)[0]
        assert q["status"] == 0
        assert np.max(np.abs(q["kmags"] / k0 - 1)) < 2e-9


def test_a_batch_with_both_kinds_of_results():
    """Sixteen iterations are enough for the lowest mode of a smooth guide, not for the ridges:
    one problem's result comes from the shared search space, its neighbours' from the run per
    band after it.  k and vectors of all of them against solves of their own."""
    print("multik batch of both kinds", flush=True)
    g, ridge = _eps(64, 48)
    x, y = np.arange(64)[:, None] * 6 / 64 - 3, np.arange(48)[None, :] / 12 - 2
    eps = 2.1 + 2.1 * np.exp(-x ** 2 - (y / 0.6) ** 2)
    smooth = np.ascontiguousarray(np.eye(3)[:, :, None, None] / eps)
    tol = dict(k_tol=1e-11, eig_tol=1e-9)
    probs = [dict(grid=g, epsinv=e, omega=W0 * f, nev=n, maxiter=2, max_eigsolves=60, **tol)
             for e, f, n in ((ridge, 1.0, 4), (smooth, 1.0, 1), (ridge, 1.05, 3))]
    res = omx.solve_k_batch(probs, fetch_evecs=True)
    assert omx.solve_phases() == dict(shared=1, per_band=2, redone=2)
    for p, q in zip(probs, res):
        assert q["status"] == 0 and q["info"]["converged"] == 1 and q["info"]["max_residual"] <= 1e-9
        k0, ev0 = omx.solve_k(p["omega"], p["epsinv"], g, omx.HIPSolver(), nev=p["nev"], maxiter=300, **tol)
        assert np.max(np.abs(q["kmags"] / k0 - 1)) < 2e-10
        for a, b in zip(q["evecs"], ev0):
            assert abs(abs(np.vdot(a, b)) - 1) < 1e-9


@pytest.mark.parametrize("nx,ny,nev", [(45, 45, 4), (27, 45, 12)])
def test_the_shared_space_works_again_after_a_solve_that_overflowed(nx, ny, nev):
    """Start vectors of 1e25 overflow single precision in the first iteration, the norm's
    weight 1 / k^2 at a k of 1e-9 or so in one of the first fifty, of either parity.  Whatever
    such a solve ends in, the handle's next one runs in the shared search space, on grids
    whose pixel counts leave the Gram products' last loads beyond the fields (2025 = 1 and
    1215 = 3 mod 4)."""
    print(f"multik after an overflow {nx}x{ny} nev {nev}", flush=True)
    g, ei = _eps(nx, ny)
    s = omx.HIPSolver()
    k0, ev, _ = _solve(g, ei, nev, 1, solver=s)
    H = np.stack(ev)
    for kw in [dict(Hguess=1e25 * H)] + [dict(Hguess=H, kguess=10.0 ** (0.05 * e)) for e in range(-181, -174)]:
        try:
            omx.solve_k(W0, ei, g, s, nev=nev, **{**KW, "maxiter": 20, **kw})
        except omx.OmxError:
            pass
        print(f"  kguess {kw.get('kguess')}: {omx.solve_phases()}", flush=True)
        assert np.max(np.abs(_solve(g, ei, nev, 1, solver=s)[0] / k0 - 1)) < 2e-10


def _box(d, nx=40, ny=45):
    """A guide that fills most of its cell: past the lowest pair the bands are near cut-off, the
    eleventh and twelfth below it."""
    x, y = -d / 2 + d / nx * np.arange(nx), 0.98 * (-d / 2 + d / ny * np.arange(ny))
    eps = 2.1 + 2.1 * np.exp(-(x[:, None] / 0.4) ** 2 - (y[None, :] / 0.3) ** 2)
    return omx.Grid(d, 0.98 * d, nx, ny), np.ascontiguousarray(np.eye(3)[:, :, None, None] / eps)


@pytest.mark.parametrize("d,nev", [(1.1, 10), (1.3, 10), (1.1, 8), (0.95, 4)])
def test_bands_near_cut_off(d, nev):
    """The guard columns of ten bands do not propagate at this omega, and the bands' own k
    spread over a factor of two and more: both must stay in the shared search space, in no
    more iterations than the same solve without such guards needs."""
    print(f"multik near cut-off {d} nev {nev}", flush=True)
    g, ei = _box(d)
    k0, _, _ = _solve(g, ei, nev, 0)
    k1, _, info = _solve(g, ei, nev, 1)
    print(f"  k {k1[0]:.4f} .. {k1[-1]:.4f}, {info['lobpcg_iters_fp32']} iterations over the bands", flush=True)
    assert np.max(np.abs(k1 / k0 - 1)) < 1e-11 / (2 * 0.1 * 0.1)
    assert info["lobpcg_iters_fp32"] <= 15 * nev


@pytest.mark.parametrize("why", ["evanescent bands", "below single precision"])
def test_a_hopeless_phase_ends_early(why, monkeypatch, capfd):
    """Bands with no k at this omega, and a threshold the phase's single precision cannot meet:
    the shared search space stops trying well before its cap of 200 iterations."""
    print(f"multik hopeless: {why}", flush=True)
    monkeypatch.setenv("OMX_TRACE", "1")
    g, ei = _eps(64, 48)
    s = omx.HIPSolver(fp32_tol=1e-9) if "below" in why else omx.HIPSolver()
    capfd.readouterr()
    try:
        k, _ = omx.solve_k(0.05 if "evan" in why else W0, ei, g, s, nev=8 if "evan" in why else 4, k_tol=1e-10,
                           eig_tol=1e-10, maxiter=40, max_eigsolves=8)
    except omx.OmxError as e:
        assert e.status == omx._lib.OMX_ERR_NOT_CONVERGED
    its = capfd.readouterr().err.count("[omx] multik it")
    print(f"  {its} iterations, {omx.solve_phases()}", flush=True)
    assert omx.solve_phases()["redone"] == 1
    assert its < 80


@pytest.mark.parametrize("sep", [1.2, 1.5, 1.8, 2.1, 2.4])
def test_close_bands(sep):
    """Two equal guides sep on either side of the middle: pairs of bands whose k differ by 1e-3
    down to rounding.  Pairs closer than 3e-5 take their vectors at one k, and each must still
    settle at its own."""
    print(f"multik pair at {sep}", flush=True)
    g = omx.Grid(10.0, 4.0, 100, 48)
    x, y = np.arange(100)[:, None] * 0.1 - 5.0, np.arange(48)[None, :] / 12 - 2.0
    eps = 2.1 + 2.0 * np.exp(-(y / 0.4) ** 2) * (np.exp(-((x - sep) / 0.5) ** 2) + np.exp(-((x + sep) / 0.5) ** 2))
    ei = np.ascontiguousarray(np.eye(3)[:, :, None, None] / eps)
    k0, _, _ = _solve(g, ei, 4, 0)
    k1, _, _ = _solve(g, ei, 4, 1)
    print(f"  k {k1}, splits {k1[0] / k1[1] - 1:.1e} {k1[2] / k1[3] - 1:.1e}", flush=True)
    assert np.max(np.abs(k1 / k0 - 1)) < 2e-10


def test_a_tolerance_below_rounding_costs_one_solve(monkeypatch, capfd):
    """A residual of 1e-17 is out of reach of either form.  The refinement of the shared
    space's blocks sees that it makes no progress; only the per-band form after it goes to the
    caller's limit of eigensolves."""
    print("multik tolerance below rounding", flush=True)
    monkeypatch.setenv("OMX_TRACE", "1")
    g, ei = _eps(64, 48)
    capfd.readouterr()
    with pytest.raises(omx.OmxError) as e:
        omx.solve_k(W0, ei, g, omx.HIPSolver(), nev=3, k_tol=1e-10, eig_tol=1e-17, maxiter=100, max_eigsolves=24)
    assert e.value.status == omx._lib.OMX_ERR_NOT_CONVERGED
    log = capfd.readouterr().err
    first, second = log.split("[omx] fp32 lobpcg run", 1)
    steps = [t.count("[omx] fp64 refine step") - t.count(", correction ") for t in (first, second)]
    print(f"  refinement steps {steps}, {omx.solve_phases()}", flush=True)
    assert omx.solve_phases() == REDONE
    assert steps[0] <= 8


def test_device_time_of_a_solve_done_twice():
    """device_ms is the call's: of a solve whose first run ends undone, both runs'.  On a warm
    handle the device works for all but the host's share of the wall time (a tenth of such a
    solve; the first run takes three quarters of this one)."""
    print("multik device time", flush=True)
    g, ei = _eps(128, 96)
    L, P = omx._lib.lib(), omx._lib
    h = omx.HIPSolver().handle(g, ei)
    km = np.empty(4)
    share = []
    for _ in range(4):
        info = omx.OmxInfo()
        t = time.perf_counter()
        st = L.omx_solve_k(h.h, W0, 4, 1e-10, 1e-17, 4, 100, None, None, 0, P.dptr(km), None, ctypes.byref(info))
        t = time.perf_counter() - t
        assert st == P.OMX_ERR_NOT_CONVERGED and omx.solve_phases() == REDONE
        share.append(1e-3 * info.device_ms / t)
    print(f"  device time over wall time {share}", flush=True)
    assert max(share[1:]) > 0.8


def test_kernel_stats_count_the_columns_that_ran():
    """The profile's bytes of the shared space: the operator on all m columns of every iteration
    made, the preconditioner on those that went on (all in the first, none in the last)."""
    print("multik kernel stats", flush=True)
    g, ei = _eps(64, 48)
    nev, m = 4, 6
    s = omx.HIPSolver(profile=True)
    _, _, info = _solve(g, ei, nev, 1, solver=s)
    ms, n, b = omx.kernel_stats(s, "op_fp32")
    one, per = 32.0 * g.N, 24.0 * g.N
    print(f"  {n} intervals, {ms:.3f} ms, {b / (one + per):.1f} columns", flush=True)
    assert info["lobpcg_iters_fp32"] / nev <= n <= info["lobpcg_iters_fp32"]
    assert ms > 0
    assert n * (one * m + per) + one * m + per <= b < (2 * n - 1) * (one * m + per)
