"""Whole sources on both sides of the size up to which one solve takes the five
12-column sources: the propagators of a source solve the oracle's equations,
and the 12-column solves of the same sources give the same columns.  The solves
stop at |r|^2 <= 1e-24 |b|^2 and |D^-1| < 10 here, so two solutions differ by
less than 2e-11 of a unit source, and a column's true residual^2 is below 1e-22."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BC = (1.0, 0.0, 0.0, 0.0)


@pytest.mark.parametrize("dims,eo,prec", [((4, 4, 4, 6), False, 0), ((4, 6, 4, 8), True, 2), ((6, 4, 4, 4), True, 1),
                                          ((34, 16, 16, 16), True, 2)])
def test_sources_solve_the_equations(chip, orc, dims, eo, prec):
    print(f"sources {dims} eo={eo} prec={prec}", flush=True)
    g = chip.gauge_random(dims, 21, 0.3)
    ctx = chip.Context(dims, 0.163, 0.01, BC, gauge=g)
    ctx.set_solver_flags(chip.SOLVE_EO if eo else 0)
    src = (1, 2, 0, 3)
    delta = {0: 0.1, 1: 0.001, 2: 0.02}[prec]
    props, st = ctx.cvc_propagators(src, 1e-24, 20000, prec, delta)
    assert st["converged"] == 120 and st["iterations"] > 10
    L = {0: orc.Lattice(dims, 0.163, 0.01, BC), 1: orc.Lattice(dims, 0.163, -0.01, BC)}
    V = int(np.prod(dims))
    for fl, s, k in ((0, 4, 0), (0, 1, 7), (1, 0, 11), (1, 3, 5)):
        y = [(src[m] + (m == s)) % dims[m] for m in range(4)]
        site = ((y[0] * dims[1] + y[1]) * dims[2] + y[2]) * dims[3] + y[3]
        b = chip.point_source(V, site, k // 3, k % 3)
        r = L[fl].Q_phi(g, props[60 * fl + 12 * s + k]) - b
        assert L[fl].dot_re(r, r) < 1e-22, (fl, s, k)
    b = np.stack([chip.point_source(V, ((src[0] * dims[1] + src[1]) * dims[2] + src[2]) * dims[3] + src[3], a // 3, a % 3)
                  for a in range(12)])
    _, x, _ = ctx.invert_Qtm_her(b, 1e-24, 20000, prec=prec, delta=delta)
    assert np.max(np.abs(x - props[48:60])) < 2e-11
