"""The FP32 operator where it marches in t by itself: the fewest and the most right-hand
sides, a time extent that four slices do not divide, chunks that do not fill a patch.
The tolerance is that of the FP32 operator tests, 2e-6 of the largest entry."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
BC = (1.0, 0.2, 0.0, -0.3)


@pytest.mark.parametrize("dims,nrhs", [((32, 32, 16, 22), 8), ((32, 32, 16, 16), 12), ((18, 16, 32, 18), 20)])
def test_fp32_march(chip, orc, dims, nrhs):
    print(f"FP32 march {dims} nrhs={nrhs}", flush=True)
    g = chip.gauge_random(dims, 9, 0.3)
    ctx = chip.Context(dims, 0.15, 0.02, BC, gauge=g)
    L = orc.Lattice(dims, 0.15, 0.02, BC)
    f64, a, b = ctx.field(nrhs), ctx.field(nrhs, chip.PREC_F32), ctx.field(nrhs, chip.PREC_F32)
    f64.fill_random(3)
    cols = (0, nrhs - 1)
    want = [L.Q_phi(g, f64.download(r, 1)[0]) for r in cols]
    a.copy_from(f64)
    ctx.dslash(b, a)
    f64.copy_from(b)
    for r, w in zip(cols, want):
        assert rel_err(f64.download(r, 1)[0], w) < 2e-6, r
