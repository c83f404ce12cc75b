"""CG loops that run in one launch with the fields on the chip (tl_chip.hip),
through the native driver, against the CPU oracle's driver.

The grids put the edges of the tiles everywhere they can be: one block and
several, partial tiles on each axis, one cell beyond a full tile, odd row
lengths, halo depths 2 and 3 (the driver primes two layers), every number of
cells per thread, the largest grids that fit and the first that do not.

Tolerance: a fixed number of iterations from the same state.  The two runs
round their dot products differently (at most ~n eps relative, n the cells
summed one after another by the oracle, in practice below 1e-13) and each
iteration's vector updates inherit that through alpha and beta, so after the
few iterations run here fields agree to 1e-12 of their largest value and the
residual norm to 1e-11.  That holds while r is more than rounding noise of
the right-hand side; a system of a handful of cells is solved before (each
iteration removes one of its few distinct eigenvalues), and its r and p are
then noise, of the oracle's size: there the prediction of r.r cancels, and
the loop has to sum the new r.r instead.
"""
import numpy as np
import pytest

from tealeaf_amd import deck as tdeck
from tests.problem_helpers import oracle_run

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


def _compare(text, dims):
    from oracle.pyoracle import run_problem
    from tealeaf_amd.problem import Problem
    s, states = tdeck.parse_deck(text, dims)
    want = run_problem(s, states, steps=1, fields=(("u", 3), ("u0", 4), ("p", 5)))
    with Problem(s, states) as p:
        rep = p.step(0)
        got = {f: p.get(f) for f in ("u", "p")}
    orep = want["steps"][0]
    assert rep["n_cg_steps"] == orep["n_cg_steps"]
    h = s.halo_depth
    inner = tuple(slice(h, n - h) for n in s.shape())
    u0 = want["fields"]["u0"]
    rr = orep["error"] ** 2 if dims == 3 else orep["error"]      # 3D reports the root
    solved = rr <= 2.0 ** -106 * np.sum(u0 * u0)
    for f, a in got.items():
        b = want["fields"][f].reshape(s.shape())[inner]
        # (a 1 x 1 grid starts solved: 0 / 0 there, NaN as in the reference)
        np.testing.assert_array_equal(np.isnan(a[inner]), np.isnan(b))
        d, m = np.nan_to_num(a[inner] - b), np.nan_to_num(b)
        if solved and f == "p":
            assert np.max(np.abs(a[inner])) <= 100 * np.max(np.abs(b))
        else:
            assert np.max(np.abs(d)) <= 1e-12 * np.max(np.abs(m)), f
    if solved:
        assert rep["error"] <= 1e4 * orep["error"]
    else:
        np.testing.assert_allclose(rep["error"], orep["error"], rtol=1e-11)
    return rep


# nx, ny, iterations, halo depth
GRIDS2 = [(1, 1, 2, 2), (16, 64, 5, 2), (17, 65, 5, 2), (48, 48, 9, 2), (64, 128, 7, 2),
          (64, 129, 7, 3), (65, 128, 7, 2), (63, 16, 5, 2), (3, 700, 5, 2), (700, 3, 5, 2),
          (511, 513, 6, 2), (520, 1029, 4, 2), (1001, 777, 4, 2), (1441, 1310, 3, 2),
          (1448, 1449, 3, 2)]


@pytest.mark.parametrize("grid", GRIDS2, ids=[f"{g[0]}x{g[1]}h{g[3]}" for g in GRIDS2])
def test_cg_2d_matches_oracle(hip, oracle, grid):
    nx, ny, iters, hd = grid
    _compare(_text(nx, ny, 0, iters, hd), 2)


# nx, ny, nz, iterations, halo depth, reciprocal conductivity
GRIDS3 = [(2, 2, 2, 3, 2, False), (64, 16, 8, 5, 2, True), (65, 17, 9, 5, 2, False),
          (32, 32, 8, 5, 2, True), (33, 31, 7, 5, 3, False), (16, 65, 5, 5, 2, False),
          (5, 6, 90, 5, 2, True), (100, 61, 40, 4, 2, True), (128, 96, 64, 3, 2, False),
          (127, 128, 128, 3, 2, True), (128, 128, 129, 3, 2, True)]


@pytest.mark.parametrize("grid", GRIDS3, ids=["x".join(map(str, g[:3])) + f"h{g[4]}" for g in GRIDS3])
def test_cg_3d_matches_oracle(hip, oracle, grid):
    nx, ny, nz, iters, hd, recip = grid
    _compare(_text(nx, ny, nz, iters, hd, recip), 3)


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
