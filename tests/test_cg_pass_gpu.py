"""CG iterations as one pass over memory (tl_cg_pass.hip), which the native
driver runs on 2D grids that do not fit the chip.

Long and flat or narrow and tall grids do not fit either, so the edges of
strips (124 columns) and of tiles (as many rows as give two waves per SIMD, one
to thirteen here) are reached with few cells; tiles of set heights too.  The
reference and the tolerance are those of test_chip_gpu.py.
"""
import numpy as np
import pytest

from tealeaf_amd import deck as tdeck
from tests.test_chip_gpu import _compare, _text

pytestmark = pytest.mark.gpu

# nx, ny, iterations, halo depth
GRIDS = [(16500, 1, 3, 2), (16500, 2, 3, 2), (16502, 3, 3, 3), (17000, 31, 4, 2),
         (16800, 32, 4, 2), (16644, 33, 4, 3), (16500, 65, 4, 2), (2, 131200, 3, 2),
         (122, 16500, 4, 2), (124, 16500, 4, 3), (126, 16600, 4, 2), (250, 8300, 4, 2),
         (1502, 1500, 4, 2), (2048, 1100, 4, 2)]


@pytest.mark.parametrize("recip", [False, True], ids=["density", "reciprocal"])
@pytest.mark.parametrize("grid", GRIDS, ids=[f"{g[0]}x{g[1]}h{g[3]}" for g in GRIDS])
def test_pass_matches_reference(hip, oracle, grid, recip):
    nx, ny, iters, hd = grid
    text = _text(nx, ny, 0, iters, hd)
    if recip:
        text = text.replace("*endtea", "coefficient_inverse_density\n*endtea")
    _compare(text, 2)


@pytest.mark.parametrize("solver", [tdeck.CG, tdeck.CHEBY, tdeck.PPCG])
def test_host_driven_is_the_same(hip, solver):
    """alpha and beta formed on the host after every pass: the same bits."""
    from tealeaf_amd.problem import Problem
    text = _text(17000, 20, 0, 90, 2, solver=solver, presteps=25)
    out = []
    try:
        for resident in (1, 0):
            hip.tlhip_set_resident(resident)
            with Problem.from_deck(text, 2) as p:
                rep = p.step(0)
                out.append((rep, p.get("u"), p.get("r"), p.get("p")))
    finally:
        hip.tlhip_set_resident(1)
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        np.testing.assert_array_equal(a, b)


# nx, ny, rows per tile: one row, the last tile full, one row in it, one missing
@pytest.mark.parametrize("grid", [(17000, 31, 1), (16800, 32, 8), (16644, 33, 8), (16500, 31, 8),
                                  (122, 16500, 75), (250, 8300, 69)],
                         ids=lambda g: "x".join(map(str, g)))
def test_tile_heights_match_reference(hip, oracle, grid):
    nx, ny, rows = grid
    hip.tlhip_set_tile_rows(rows)
    try:
        _compare(_text(nx, ny, 0, 4, 2), 2)
    finally:
        hip.tlhip_set_tile_rows(-1)


def _short(nx, ny, dt, solver=tdeck.CG, iters=60, presteps=30):
    text = _text(nx, ny, 0, iters, 2, solver=solver, presteps=presteps)
    assert "initial_timestep = 0.004" in text
    return text.replace("initial_timestep = 0.004", f"initial_timestep = {dt}")


def _passes(left):
    """Pass launches of the host-driven loop: two sums an iteration until r.r
    falls to no less than 1%, then the sums in hand and a pass per iteration
    until one would cancel."""
    n, k = 0, 0
    while k < len(left) and left[k] < 0.01:
        k += 1
    k += 1
    if k < len(left):
        n += 1
        while k < len(left) and left[k] >= 0.01:
            n, k = n + 1, k + 1
    return n


# nx, ny, timestep, whether passes run, whether one cancels
TURNS = [(48, 48, 4e-5, False, False), (48, 48, 4e-4, True, True), (300, 260, 4e-6, False, False),
         (512, 512, 4e-6, True, False), (96, 80, 4e-3, True, False)]


def _launches(hip, name, run):
    import ctypes
    ms, n = ctypes.c_double(), ctypes.c_long()
    hip.tlhip_kernel_timer_start(name)
    try:
        out = run()
    finally:
        hip.tlhip_kernel_timer_read(ctypes.addressof(ms), ctypes.addressof(n))
    return out, n.value


@pytest.mark.parametrize("resident", [1, 0])
@pytest.mark.parametrize("case", TURNS, ids=[f"{c[0]}x{c[1]}t{c[2]:g}" for c in TURNS])
def test_turns_between_two_sums_and_passes(hip, oracle, case, resident):
    """Fast iterations run with two sums, slow ones as passes: from the pair
    to passes, and back where a prediction cancels, from the launch counts of
    the host-driven loop.  Fields as the reference's on each way."""
    nx, ny, dt, passes, cancels = case
    hip.tlhip_set_resident(resident)
    try:
        left, n = _launches(hip, b"tl_cg_pass2d",
                            lambda: _compare(_short(nx, ny, dt), 2, on_chip=False))
    finally:
        hip.tlhip_set_resident(1)
    assert (n > 0) == passes
    want = _passes(left)
    assert resident or n == want
    assert (0 < want < len(left) - left.index(next(f for f in left if f >= 0.01)) if cancels
            else True)


@pytest.mark.parametrize("graphs", [0, 1])
@pytest.mark.parametrize("rel", [0.0, 1e-9])
@pytest.mark.parametrize("solver,presteps", [(tdeck.CG, 30), (tdeck.CHEBY, 4), (tdeck.CHEBY, 7),
                                             (tdeck.PPCG, 4), (tdeck.PPCG, 7)])
@pytest.mark.parametrize("dt", [4e-5, 4e-4, 4e-3])
def test_turns_resident_is_host_driven(hip, solver, presteps, dt, rel, graphs):
    """Runs that turn, cut by a switch of solvers before, at and after the
    turns: the same bits from the device's decisions and from the host's."""
    from tealeaf_amd.problem import Problem
    out = []
    hip.tlhip_set_graphs(graphs)
    try:
        for resident in (1, 0):
            hip.tlhip_set_resident(resident)
            with Problem.from_deck(_short(48, 48, dt, solver, 90, presteps), 2) as p:
                p.set_on_chip(False)
                p.set_solve(0, rel)
                out.append((p.step(0), p.step(1), p.get("u"), p.get("r"), p.get("p")))
    finally:
        hip.tlhip_set_resident(1)
        hip.tlhip_set_graphs(0)
    assert out[0][:2] == out[1][:2]
    for a, b in zip(out[0][2:], out[1][2:]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("nx,fits", [(65536 * 124, True), (65536 * 124 + 2, False)])
def test_widest_grids(hip, nx, fits):
    """A strip of columns needs a block of its own and a place for its partial
    sums: one strip more than there are places keeps the pair of passes.  The
    same u as from kx and ky (a timestep that makes the operator well
    conditioned along x)."""
    import ctypes
    from tealeaf_amd.problem import Problem
    text = _text(nx, 1, 0, 3, 2).replace("initial_timestep = 0.004", "initial_timestep = 1.5e-12")
    assert "1.5e-12" in text
    out, ms, n = [], ctypes.c_double(), ctypes.c_long()
    try:
        for cond in (1, 0):
            hip.tlhip_set_cg_cond(cond)
            with Problem.from_deck(text, 2) as p:
                hip.tlhip_kernel_timer_start(b"tl_cg_pass2d")
                rep = p.step(0)
                hip.tlhip_kernel_timer_read(ctypes.addressof(ms), ctypes.addressof(n))
                assert rep["n_cg_steps"] == 3
                assert (n.value > 0) == (fits and cond == 1)
                out.append(p.get("u"))
    finally:
        hip.tlhip_set_cg_cond(1)
    assert np.max(np.abs(out[0] - out[1])) <= 1e-12 * np.max(np.abs(out[1]))
