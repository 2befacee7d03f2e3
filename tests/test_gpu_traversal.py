"""The automatic traversal and block sizes of the multi-rhs operator on lattices
where they can go wrong: columns that do not divide by the eight XCDs, runs that
do not fill their blocks, prime and odd extents, right-hand-side counts on both
sides of the links-in-LDS threshold and whose blocks cannot be 128-byte aligned,
a chip's worth of blocks and fewer blocks than XCDs.  The tolerances are those of
the operator tests: FP64 1e-13, FP32 2e-6, FP16 2e-3 of the largest entry."""
import numpy as np
import pytest

from conftest import rand_spinor, rel_err

pytestmark = pytest.mark.gpu
BC = (1.0, 0.2, 0.0, -0.3)


@pytest.mark.parametrize("dims,nrhs", [((5, 7, 3, 11), 12), ((2, 2, 2, 2), 12), ((3, 10, 6, 10), 7), ((3, 5, 4, 6), 8),
                                       ((4, 6, 10, 14), 9), ((2, 9, 5, 4), 60), ((6, 4, 14, 8), 48), ((2, 3, 2, 6), 256),
                                       ((3, 4, 4, 2), 85), ((10, 20, 5, 5), 16)])
def test_operator_shapes(chip, orc, dims, nrhs):
    print(f"operator {dims} nrhs={nrhs}", flush=True)
    g = chip.gauge_random(dims, 5, 0.3)
    ctx = chip.Context(dims, 0.15, 0.02, BC, gauge=g)
    L = orc.Lattice(dims, 0.15, 0.02, BC)
    phi = rand_spinor(np.random.default_rng(nrhs), L.V, nrhs)
    cols = sorted({0, nrhs // 2, nrhs - 1})
    want = {r: L.Q_phi(g, phi[r]) for r in cols}
    fin, fout = ctx.field(nrhs), ctx.field(nrhs)
    fin.upload(phi)
    ctx.dslash(fout, fin)
    got = fout.download()
    for r in cols:
        assert rel_err(got[r], want[r]) < 1e-13, r
    for prec, tol in [(chip.PREC_F32, 2e-6), (chip.PREC_F16, 2e-3)]:
        a, b, back = ctx.field(nrhs, prec), ctx.field(nrhs, prec), ctx.field(nrhs)
        a.copy_from(fin)
        ctx.dslash(b, a)
        back.copy_from(b)
        lo = back.download()
        for r in cols:
            assert rel_err(lo[r], want[r]) < tol, (prec, r)


@pytest.mark.parametrize("dims,nrhs", [((4, 6, 10, 14), 12), ((2, 2, 4, 2), 12), ((6, 10, 6, 4), 17), ((4, 4, 6, 6), 3)])
def test_even_odd_shapes(chip, orc, dims, nrhs):
    """Even/odd solves on such lattices solve the oracle's equation, in every precision:
    |D x - b|^2 <= 1e-20 |b|^2 on the odd system gives below 1e-18 on the lattice
    (|A| / |M| < 10)."""
    print(f"even/odd {dims} nrhs={nrhs}", flush=True)
    g = chip.gauge_random(dims, 6, 0.3)
    ctx = chip.Context(dims, 0.163, 0.01, BC, gauge=g)
    L = orc.Lattice(dims, 0.163, 0.01, BC)
    b = rand_spinor(np.random.default_rng(nrhs), L.V, nrhs)
    for prec, delta in [(chip.PREC_F64, 0.1), (chip.PREC_F32, 0.01), (chip.PREC_F16, 0.02)]:
        rc, x, st = ctx.invert_Qtm_her(b, 1e-20, 5000, prec=prec, delta=delta, eo=True)
        assert st["converged"] == nrhs
        for a in (0, nrhs - 1):
            res = L.Q_phi(g, x[a]) - b[a]
            assert L.dot_re(res, res) / L.dot_re(b[a], b[a]) < 1e-18, (prec, a)
