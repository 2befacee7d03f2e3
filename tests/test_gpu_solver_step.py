"""FP64 solves whose iteration ends in one pass (the shadow product taken from the
operator's output): vector lengths that do not fill their blocks, right-hand sides
past a wavefront, columns that converge at different iterations and one that starts
converged.  The iterated residual is tested at 1e-20 |b|^2 and the true one differs
from it by rounding (1e-27 |b|^2), so the solution solves the oracle's equation to
1.1e-20; the separate passes of the lagged solve follow the same recurrence up to
rounding, so its iteration count lies within 10 % + 3."""
import numpy as np
import pytest

from conftest import rand_spinor

pytestmark = pytest.mark.gpu
BC = (1.0, 0.2, 0.0, -0.3)


@pytest.mark.parametrize("her", [False, True])
@pytest.mark.parametrize("dims,nrhs", [((3, 5, 4, 6), 1), ((4, 3, 5, 7), 7), ((4, 4, 6, 2), 12), ((2, 3, 3, 5), 70),
                                       ((10, 12, 12, 12), 12)])
def test_fp64_solve(chip, orc, dims, nrhs, her):
    print(f"solve {dims} nrhs={nrhs} her={her}", flush=True)
    g = chip.gauge_random(dims, 8, 0.3)
    ctx = chip.Context(dims, 0.14, 0.05, BC, gauge=g)
    L = orc.Lattice(dims, 0.14, 0.05, BC)
    b = rand_spinor(np.random.default_rng(nrhs), L.V, nrhs)
    if nrhs > 2:
        b[1] = 0.                     # solved at the start
        b[2, 1:] = 0.                 # a point-like source
        b[nrhs - 1] *= 1e-30
    solve = ctx.invert_Qtm_her if her else ctx.invert_Qtm
    _, x, st = solve(b, 1e-20, 2000)
    _, _, lag = solve(b, 1e-20, 2000, lagged=True)
    assert st["converged"] == lag["converged"] == nrhs
    assert abs(st["iterations"] - lag["iterations"]) <= 0.1 * lag["iterations"] + 3
    for r in sorted({0, min(2, nrhs - 1), nrhs - 1}):
        res = L.Q_phi(g, x[r]) - b[r]
        assert L.dot_re(res, res) <= 1.1e-20 * L.dot_re(b[r], b[r]), r
    if nrhs > 2:
        assert not x[1].any()
