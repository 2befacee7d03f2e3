"""The contraction at the edges of its slabs and blocks against the oracle: one
slab, a last slab of one slice, slices larger than a slab, sites that do not
fill the 16- and 20-site blocks, the smallest extents.  conn sums 16 terms of
12 x 12 products, each of up to 100 roundings: below 1e-12 of the largest entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BC = (1.0, 0.3, -0.2, 0.5)


@pytest.mark.parametrize("dims,src", [((2, 2, 2, 2), (1, 1, 0, 1)), ((3, 5, 3, 7), (2, 4, 1, 6)), ((4, 2, 5, 6), (0, 1, 4, 0)),
                                      ((5, 10, 10, 20), (4, 3, 9, 19)), ((2, 30, 17, 16), (1, 29, 16, 2))])
def test_contract_slabs(chip, orc, dims, src):
    print(f"contraction slabs {dims}", flush=True)
    g = chip.gauge_random(dims, 11, 0.3)
    ctx = chip.Context(dims, 0.15, 0.02, BC, gauge=g)
    L = orc.Lattice(dims, 0.15, 0.02, BC)
    props = np.random.default_rng(sum(dims)).standard_normal((120, L.V, 24))
    want, ct = L.cvc_contract(g, list(props), src)
    got, ct_got = ctx.cvc_contract(list(props), src)
    want = np.asarray(want).reshape(got.shape)
    assert np.max(np.abs(got - want)) < 1e-12 * np.max(np.abs(want))
    assert np.max(np.abs(ct_got - ct)) < 1e-12 * np.max(np.abs(ct))
