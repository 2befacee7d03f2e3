"""The two-point kernel at the edges of its split against the oracle: 256-site
chunks of a time slice (whole, one site over, ragged), 4, 8 and 12 columns, odd
extents, and a lattice whose extents exceed the phase tables.  Sums of n random
terms in FP64: |error| <= a few n eps |terms| with n <= 2.4e4, below 1e-12 of
the largest correlator entry times sqrt(n), hence the factor 10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BC = (1.0, 0.0, 0.0, 0.0)


@pytest.mark.parametrize("dims,n_c", [((3, 4, 8, 8), 3), ((2, 257, 2, 2), 1), ((5, 3, 7, 5), 2), ((2, 13, 9, 11), 3),
                                      ((2, 2046, 2, 2), 1), ((2, 2, 2, 2), 3)])
def test_twopoint_split(chip, orc, dims, n_c):
    print(f"two-point {dims} n_c={n_c}", flush=True)
    ctx = chip.Context(dims, 0.15, 0.01, BC)
    L = orc.Lattice(dims, 0.15, 0.01, BC)
    rng = np.random.default_rng(sum(dims))
    N = 4 * n_c
    chi, phi = rng.standard_normal((N, L.V, 24)), rng.standard_normal((N, L.V, 24))
    src = tuple(d // 2 for d in dims)
    fc, fp = ctx.field(N), ctx.field(N)
    fc.upload(chi)
    fp.upload(phi)
    for gs, gk, mom in ((5, 5, None), (0, 11, (1, 0, 1)), (13, 2, (0, 1, 1))):
        want = L.contract_twopoint(gs, gk, list(chi), list(phi), n_c, mom, src)
        got = ctx.field_contract_twopoint(gs, gk, fc, fp, n_c, mom, src)
        assert np.max(np.abs(got - want)) < 1e-11 * np.max(np.abs(want)), (gs, gk, mom)
