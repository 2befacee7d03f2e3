"""The operator of fewer than eight right-hand sides (links from memory), whose kernel
depends on the precision and on whether there are one, two or more: odd and even
extents, blocks that do not fill a wave.  Tolerances as in the operator tests: FP64
1e-13, FP32 2e-6, FP16 2e-3 of the largest entry; even/odd solves to 1e-20 give below
1e-18 on the lattice (|A| / |M| < 10)."""
import numpy as np
import pytest

from conftest import rand_spinor, rel_err

pytestmark = pytest.mark.gpu
BC = (1.0, 0.2, 0.0, -0.3)


@pytest.mark.parametrize("nrhs", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("dims", [(3, 5, 7, 2), (8, 6, 5, 9)])
def test_operator(chip, orc, dims, nrhs):
    print(f"operator {dims} nrhs={nrhs}", flush=True)
    g = chip.gauge_random(dims, 5, 0.3)
    ctx = chip.Context(dims, 0.15, 0.02, BC, gauge=g)
    L = orc.Lattice(dims, 0.15, 0.02, BC)
    phi = rand_spinor(np.random.default_rng(nrhs), L.V, nrhs)
    want = [L.Q_phi(g, phi[r]) for r in range(nrhs)]
    fin = ctx.field(nrhs)
    fin.upload(phi)
    for prec, tol in [(chip.PREC_F64, 1e-13), (chip.PREC_F32, 2e-6), (chip.PREC_F16, 2e-3)]:
        a, b, back = ctx.field(nrhs, prec), ctx.field(nrhs, prec), ctx.field(nrhs)
        a.copy_from(fin)
        ctx.dslash(b, a)
        back.copy_from(b)
        got = back.download()
        for r in range(nrhs):
            assert rel_err(got[r], want[r]) < tol, (prec, r)


@pytest.mark.parametrize("nrhs", [1, 2, 3])
def test_even_odd(chip, orc, nrhs):
    dims = (4, 6, 2, 6)
    print(f"even/odd {dims} nrhs={nrhs}", flush=True)
    g = chip.gauge_random(dims, 6, 0.3)
    ctx = chip.Context(dims, 0.163, 0.01, BC, gauge=g)
    L = orc.Lattice(dims, 0.163, 0.01, BC)
    b = rand_spinor(np.random.default_rng(nrhs), L.V, nrhs)
    for prec, delta in [(chip.PREC_F64, 0.1), (chip.PREC_F32, 0.01), (chip.PREC_F16, 0.02)]:
        _, x, st = ctx.invert_Qtm_her(b, 1e-20, 5000, prec=prec, delta=delta, eo=True)
        assert st["converged"] == nrhs
        for a in range(nrhs):
            res = L.Q_phi(g, x[a]) - b[a]
            assert L.dot_re(res, res) / L.dot_re(b[a], b[a]) < 1e-18, (prec, a)
