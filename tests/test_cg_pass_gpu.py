"""CG iterations as one pass over memory (tl_cg_pass.hip), which the native
driver runs on 2D grids that do not fit the chip.

Long and flat or narrow and tall grids do not fit either, so the edges of
strips (124 columns) and tiles (32 rows) are reached with few cells.  The reference
and the tolerance are those of test_chip_gpu.py.
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


@pytest.mark.parametrize("nx,fits", [(65536 * 124, True), (65536 * 124 + 2, False)])
def test_widest_grids(hip, nx, fits):
    """A strip of columns needs a block of its own and a place for its partial
    sums: one strip more than there are places takes the passes over kx and
    ky.  The same u either way (a timestep that makes the operator well
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
