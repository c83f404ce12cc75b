"""CG loops that run in one launch with the fields on the chip (tl_chip.hip),
through the native driver.

The grids put the edges of the tiles everywhere they can be: one block and
several, partial tiles on each axis, one cell beyond a full tile, odd row
lengths, halo depths 2 and 3 (the driver primes two layers), every number of
cells per thread, the largest grids that fit and the first that do not.

The reference is the reference's CG (2d/drivers/cg_driver.c:78-99) in numpy
with exactly rounded sums, from the coefficients and the right-hand side of
the oracle's run, whose iteration count must agree.  (The oracle's own sums
add the cells one after another: at 2 x 131200 its alpha is 3e-11 off.)

Tolerance: a fixed number of iterations from the same state.  Sums in another
order move alpha and beta by some rounding errors, so p by some of its own,
and the next p.Ap by as many of |p|.|A||p|, which is up to the condition number
of A larger than p.Ap (long thin cells: 1e7).  With 64 of them per iteration
(rows of a lane, then a tree of sums) alpha is uncertain by 2^-47 of that
ratio.  A step r - alpha A p or beta p + r inherits this from its terms, which
are as large as the fields were before the step: so u and p are held to 1e-12
plus the sum of those bounds, of the largest value they had at the start or
the end, and the norm of r likewise.
"""
import math

import numpy as np
import pytest

from tealeaf_amd import deck as tdeck
from tests.numerics import apply_a

pytestmark = pytest.mark.gpu


def _text(nx, ny, nz, iters, hd, recip=False, solver=tdeck.CG, presteps=30):
    if nz:
        text = tdeck.cuboid_3d(77777, 1, solver=solver, max_iters=iters, dt=0.004,
                               presteps=presteps,
                               coefficient=tdeck.RECIP_CONDUCTIVITY if recip else tdeck.CONDUCTIVITY)
    else:
        text = tdeck.layered_2d(77777, 1, solver=solver, max_iters=iters, presteps=presteps)
    for axis, n in (("x", nx), ("y", ny), ("z", nz)):
        text = text.replace(f"{axis}_cells = 77777", f"{axis}_cells = {n}")
    return text.replace("halo_depth = 2", f"halo_depth = {hd}")


COEFS = (("kx", 8), ("ky", 9), ("kz", 10))


def _dot(a, b):
    try:
        return math.fsum((a * b).ravel())
    except (ValueError, OverflowError):        # infinities or NaN among them
        return float(np.sum(a * b))


def _reference(w, iters, h):
    """u, p, the starting r, r.r after `iters` CG iterations, on the interior,
    what other orders of summation can make of alpha (relative, summed), and
    what each iteration left of r.r (below 1% its prediction cancels and is not
    used)."""
    diag = 1.0 + sum(w[c] + np.roll(w[c], -1, axis) for c, axis in
                     zip(("kx", "ky", "kz"), range(w["u0"].ndim - 1, -1, -1)))
    inner = tuple(slice(h, n - h) for n in w["u0"].shape)
    k = (w["kx"], w["ky"], h, w.get("kz"))
    u = w["u0"][inner].copy()
    r = u - apply_a(w["u0"], *k)
    r0, p = r.copy(), np.zeros_like(w["u0"])
    p[inner] = r
    rro, slack, left = _dot(r, r), 0.0, []
    with np.errstate(all="ignore"):
        for _ in range(iters):
            q = apply_a(p, *k)
            pw = _dot(p[inner], q)
            alpha = np.float64(rro) / pw
            slack += 2.0 ** -47 * np.nan_to_num(
                np.sum(2.0 * diag[inner] * p[inner] ** 2) / np.float64(abs(pw)))
            u += alpha * p[inner]
            r = r - alpha * q
            rrn = _dot(r, r)
            left.append(rrn / np.float64(rro))
            p[inner] = np.float64(rrn) / rro * p[inner] + r
            rro = rrn
    return u, p[inner], r0, rro, slack, left


def _compare(text, dims, cancels=0, on_chip=True):
    from oracle.pyoracle import run_problem
    from tealeaf_amd.problem import Problem
    s, states = tdeck.parse_deck(text, dims)
    want = run_problem(s, states, steps=1, fields=(("u0", 4),) + COEFS[:dims])
    with Problem(s, states) as prob:
        prob.set_on_chip(on_chip)
        rep = prob.step(0)
        got = {f: prob.get(f) for f in ("u", "p")}
    h = s.halo_depth
    inner = tuple(slice(h, n - h) for n in s.shape())
    w = {f: a.reshape(s.shape()) for f, a in want["fields"].items()}
    assert rep["n_cg_steps"] == want["steps"][0]["n_cg_steps"]
    u, p, r0, rr, slack, left = _reference(w, rep["n_cg_steps"], h)
    assert sum(f < 0.01 for f in left) >= cancels
    for f, b, start in (("u", u, w["u0"][inner]), ("p", p, r0)):
        a = got[f][inner]
        scale = max(np.max(np.abs(start)), np.max(np.abs(np.nan_to_num(b))))
        # (a 1 x 1 grid starts solved: 0 / 0 there, NaN as in the reference)
        np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
        assert np.max(np.abs(np.nan_to_num(a - b))) <= (1e-12 + slack) * scale, f
    norm = rep["error"] if dims == 3 else np.sqrt(rep["error"])   # 3D reports the root
    np.testing.assert_allclose(norm, np.sqrt(rr), rtol=1e-11 + slack,
                               atol=(1e-12 + slack) * np.sqrt(np.sum(r0 * r0)))
    return left


# nx, ny, iterations, halo depth
GRIDS2 = [(1, 1, 2, 2), (16, 64, 5, 2), (17, 65, 5, 2), (48, 48, 9, 2), (64, 128, 7, 2),
          (64, 129, 7, 3), (65, 128, 7, 2), (63, 16, 5, 2), (3, 700, 5, 2), (700, 3, 5, 2),
          (511, 513, 6, 2), (520, 1029, 4, 2), (1001, 777, 4, 2), (1441, 1310, 3, 2),
          (1448, 1449, 3, 2)]


@pytest.mark.parametrize("grid", GRIDS2, ids=[f"{g[0]}x{g[1]}h{g[3]}" for g in GRIDS2])
def test_cg_2d_matches_reference(hip, oracle, grid):
    nx, ny, iters, hd = grid
    _compare(_text(nx, ny, 0, iters, hd), 2)


# nx, ny, nz, iterations, halo depth, reciprocal conductivity
GRIDS3 = [(2, 2, 2, 3, 2, False), (64, 16, 8, 5, 2, True), (65, 17, 9, 5, 2, False),
          (32, 32, 8, 5, 2, True), (33, 31, 7, 5, 3, False), (16, 65, 5, 5, 2, False),
          (5, 6, 90, 5, 2, True), (100, 61, 40, 4, 2, True), (128, 96, 64, 3, 2, False),
          (127, 128, 128, 3, 2, True), (128, 128, 129, 3, 2, True)]


@pytest.mark.parametrize("grid", GRIDS3, ids=["x".join(map(str, g[:3])) + f"h{g[4]}" for g in GRIDS3])
def test_cg_3d_matches_reference(hip, oracle, grid):
    nx, ny, nz, iters, hd, recip = grid
    _compare(_text(nx, ny, nz, iters, hd, recip), 3)


# nx, ny, nz, timestep, iterations that cancel
CANCEL = [(48, 48, 0, 4e-5, 4), (48, 48, 0, 4e-4, 2), (64, 128, 0, 4e-5, 6), (2, 2, 2, 0.004, 3),
          (32, 32, 8, 4e-5, 4), (300, 260, 0, 4e-6, 6), (512, 512, 0, 4e-6, 2),
          (33, 31, 17, 4e-5, 4)]


@pytest.mark.parametrize("case", CANCEL, ids=["x".join(map(str, c[:3])) + f"t{c[3]:g}" for c in CANCEL])
def test_cancelling_iterations_match_reference(hip, oracle, case):
    """Short timesteps: r.r falls a hundredfold within an iteration, so the
    blocks (or the one block's waves) meet a second time for the new r.r,
    straight after the first meeting."""
    nx, ny, nz, dt, cancels = case
    text = _text(nx, ny, nz, 60, 2).replace("initial_timestep = 0.004", f"initial_timestep = {dt}")
    assert f"initial_timestep = {dt}" in text
    _compare(text, 3 if nz else 2, cancels)


@pytest.mark.parametrize("size", [(40, 30, 0), (300, 260, 0), (40, 33, 21)])
def test_one_iteration_per_launch_is_the_same(hip, size):
    """The host-driven loop launches the loop for one iteration at a time:
    every launch starts from the fields in memory, and the bits must be those
    of the run in one launch, whatever the blocks' timing was."""
    from tealeaf_amd.problem import Problem
    text = _text(*size, 60, 2)
    dims = 3 if size[2] else 2
    out = []
    try:
        for resident in (1, 0):
            hip.tlhip_set_resident(resident)
            with Problem.from_deck(text, dims) as p:
                rep = p.step(0)
                out.append((rep, p.get("u"), p.get("r"), p.get("p")))
    finally:
        hip.tlhip_set_resident(1)
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        np.testing.assert_array_equal(a, b)


def _solver_run(text, dims):
    from oracle.pyoracle import run_problem
    from tealeaf_amd.problem import Problem
    s, states = tdeck.parse_deck(text, dims)
    want = run_problem(s, states, steps=1, fields=(("u", 3), ("r", 6)))
    with Problem(s, states) as p:
        rep = p.step(0)
        got = {f: p.get(f) for f in ("u", "r")}
    return s, rep, want["steps"][0], got, {f: a.reshape(s.shape()) for f, a in want["fields"].items()}


@pytest.mark.parametrize("sweeps", [1, 51, 53])
@pytest.mark.parametrize("size", [(40, 30, 0), (65, 129, 0), (517, 200, 0), (1301, 777, 0),
                                  (33, 32, 9), (127, 90, 60)],
                         ids=lambda n: "x".join(map(str, n)))
def test_jacobi_bits(hip, oracle, size, sweeps):
    """No sum feeds back into a sweep, so u and r (the last sweep's input, or
    the residual of every 50th iteration) are the oracle's bits."""
    iters = sweeps if size[0] * size[1] < 300000 else min(sweeps, 3)
    dims = 3 if size[2] else 2
    text = _text(*size, iters, 2, solver=tdeck.JACOBI).replace("check_result\n", "")
    s, rep, orep, got, want = _solver_run(text, dims)
    assert rep["n_jacobi"] == orep["n_jacobi"]
    np.testing.assert_array_equal(got["u"], want["u"])
    np.testing.assert_array_equal(got["r"], want["r"])
    np.testing.assert_allclose(rep["error"], orep["error"], rtol=1e-9)


@pytest.mark.parametrize("size,iters", [((40, 30, 0), 70), ((65, 129, 0), 90), ((517, 203, 0), 90),
                                        ((1301, 777, 0), 45), ((41, 32, 9), 60),
                                        ((127, 90, 61), 45)],
                         ids=lambda n: str(n).replace(" ", ""))
def test_chebyshev_matches_oracle(hip, oracle, size, iters):
    """From the switch on, Chebyshev iterations have no sums in them; what the
    two runs differ by is the eigenvalue estimate of the CG steps before, an
    extreme eigenvalue of a 21 x 21 matrix of their alphas and betas, which
    moves by no more than they do (1e-12): u to 1e-10."""
    dims = 3 if size[2] else 2
    text = _text(*size, iters, 2, solver=tdeck.CHEBY, presteps=20).replace(
        "epslim = 0.0001", "epslim = 1e30\nerrswitch").replace(
        "initial_timestep = 0.004", "initial_timestep = 0.4")    # not solved by the CG steps
    s, rep, orep, got, want = _solver_run(text, dims)
    assert rep["n_cheby_steps"] == orep["n_cheby_steps"] > 0
    h = s.halo_depth
    inner = tuple(slice(h, n - h) for n in s.shape())
    a, b = got["u"][inner], want["u"][inner]
    assert np.max(np.abs(a - b)) <= 1e-10 * np.max(np.abs(b))


def test_late_report_is_not_the_next_launchs(hip):
    """A wait limit that runs out while a launch is still at work (it ends by
    itself a few ms later): the step fails, and the next problem's step gets
    its own report, not the late one."""
    from tealeaf_amd.abi import TealeafError
    from tealeaf_amd.problem import Problem
    slow = _text(1000, 1000, 0, 4000, 2, solver=tdeck.JACOBI)          # 20 ms or more
    quick = _text(40, 30, 0, 7, 2, solver=tdeck.JACOBI).replace("check_result\n", "")
    with Problem.from_deck(quick, 2) as q:
        want = q.step(0), q.get("u")
    with Problem.from_deck(slow, 2) as p, Problem.from_deck(quick, 2) as q:
        hip.tlhip_set_wait_limit(1e-4)
        try:
            with pytest.raises(TealeafError, match="no report"):
                p.step(0)
        finally:
            hip.tlhip_set_wait_limit(0.0)
        got = q.step(0), q.get("u")
    assert want[0]["n_jacobi"] == 7
    assert got[0] == want[0]
    np.testing.assert_array_equal(got[1], want[1])


REFUSED = [("2d-cg", _text(64, 50, 0, 400, 2), 2, 1),
           ("2d-cg-odd", _text(63, 50, 0, 400, 2), 2, 1),
           ("2d-cheby", _text(64, 50, 0, 400, 2, solver=tdeck.CHEBY), 2, 1),
           ("2d-cheby-late", _text(64, 50, 0, 400, 2, solver=tdeck.CHEBY), 2, 0),
           ("2d-cheby-odd-late", _text(63, 50, 0, 400, 2, solver=tdeck.CHEBY), 2, 0),
           ("2d-ppcg", _text(64, 50, 0, 400, 2, solver=tdeck.PPCG), 2, 1),
           ("2d-jacobi", _text(64, 50, 0, 60, 2, solver=tdeck.JACOBI), 2, 1),
           ("3d-cg", _text(20, 18, 16, 400, 2), 3, 1),
           ("3d-cheby-late", _text(20, 18, 16, 400, 2, solver=tdeck.CHEBY, presteps=10), 3, 0),
           ("3d-jacobi", _text(20, 18, 16, 60, 2, solver=tdeck.JACOBI), 3, 1)]


@pytest.mark.parametrize("resident", [1, 0])
@pytest.mark.parametrize("name,text,dims,cond", REFUSED, ids=[c[0] for c in REFUSED])
def test_refused_launch_goes_on_launch_by_launch(hip, name, text, dims, cond, resident):
    """A launch that the runtime refuses (here: taken for refused) changes
    nothing, and the solve runs as one that never tried: the same bits over two
    steps.  Without the cond passes CG does not run on the chip, so the first
    launch refused is Chebyshev's."""
    from tealeaf_amd.problem import Problem
    out = []
    hip.tlhip_set_resident(resident)
    hip.tlhip_set_cg_cond(cond)
    try:
        for on in (0, 2):
            with Problem.from_deck(text, dims) as p:
                p.set_on_chip(on)
                out.append(([p.step(t) for t in range(2)], [p.get(f) for f in ("u", "r", "energy")]))
    finally:
        hip.tlhip_set_resident(1)
        hip.tlhip_set_cg_cond(1)
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1], out[1][1]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("variable", ["HSA_CU_MASK", "ROC_GLOBAL_CU_MASK"])
def test_masked_cus_keep_off_the_chip(hip, monkeypatch, variable):
    """An environment that masks CUs (read here when a problem is created; the
    runtime has read its own long before) leaves no plan for the chip."""
    import ctypes
    from tealeaf_amd.problem import Problem
    monkeypatch.setenv(variable, "0x1")
    ms, n = ctypes.c_double(), ctypes.c_long()
    with Problem.from_deck(_text(64, 50, 0, 400, 2), 2) as p:
        hip.tlhip_kernel_timer_start(b"tl_chip_cg")
        try:
            rep = p.step(0)
        finally:
            hip.tlhip_kernel_timer_read(ctypes.addressof(ms), ctypes.addressof(n))
    assert n.value == 0 and rep["n_cg_steps"] > 0
