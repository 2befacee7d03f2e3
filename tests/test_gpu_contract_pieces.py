"""The contraction on lattices of several slabs against the oracle: slabs of one and of
two slices, a shorter last slab, a slab of all slices but one, two slices, conn in more
pieces than there are slots and in pieces larger than a slot.  Gauge field and
propagators repeat a small cell, and the boundary phases per link are those of the
cell, so conn repeats the oracle's conn of the cell.  It sums 16 terms of 12 x 12
products, each of up to 100 roundings: below 1e-12 of the largest entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BC = (1.0, 0.3, -0.2, 0.5)


def repeat(a, cell, dims):
    """a[..., V(cell), k] -> [..., V(dims), k], periodic in every direction"""
    lead = a.shape[:-2]
    a = a.reshape(*lead, *cell, a.shape[-1])
    a = np.tile(a, (1,) * len(lead) + tuple(d // c for d, c in zip(dims, cell)) + (1,))
    return np.ascontiguousarray(a.reshape(*lead, int(np.prod(dims)), a.shape[-1]))


@pytest.mark.parametrize("dims,cell,src", [((10, 40, 40, 20), (5, 4, 5, 4), (9, 3, 11, 19)),
                                           ((3, 48, 45, 32), (3, 4, 3, 4), (1, 47, 0, 2)),
                                           ((5, 20, 40, 20), (5, 4, 5, 4), (4, 1, 39, 0)),
                                           ((5, 20, 20, 20), (5, 4, 5, 4), (0, 19, 7, 5)),
                                           ((2, 40, 40, 24), (2, 4, 5, 4), (1, 2, 3, 23))])
def test_contract_pieces(chip, orc, dims, cell, src):
    print(f"contraction pieces {dims}", flush=True)
    V, Vc = int(np.prod(dims)), int(np.prod(cell))
    g = chip.gauge_random(cell, 12, 0.3)
    props = np.random.default_rng(sum(dims)).standard_normal((120, Vc, 24))
    L = orc.Lattice(cell, 0.15, 0.02, tuple(b * c / d for b, c, d in zip(BC, cell, dims)))
    want, ct = L.cvc_contract(g, list(props), tuple(s % c for s, c in zip(src, cell)))
    ctx = chip.Context(dims, 0.15, 0.02, BC, gauge=repeat(g.reshape(Vc, 72), cell, dims))
    up, dn = ctx.field(60), ctx.field(60)
    for k in range(0, 120, 12):
        (up if k < 60 else dn).upload(repeat(props[k:k + 12], cell, dims), k % 60)
    got, ct_got = ctx.field_cvc_contract(up, dn, src)
    want = repeat(np.asarray(want).reshape(Vc, 32), cell, dims)
    assert np.max(np.abs(got.reshape(V, 32) - want)) < 1e-12 * np.max(np.abs(want))
    assert np.max(np.abs(ct_got - ct)) < 1e-12 * np.max(np.abs(ct))
