"""The link-force kernels on lattices whose sites do not fill their four- and
eight-site blocks: dL/dmu and tr(T F) on random link directions against central
finite differences of the value (h = 1e-5), which costs h^2 ~ 1e-10 of curvature
and 1e-15 / h ~ 1e-10 of rounding beside the solves' 1e-12: 1e-6 relative, as in
the gradient test."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BC = (1.0, 0.0, 0.0, 0.0)


def value(chip, dims, kappa, mu, gauge, src):
    ctx = chip.Context(dims, kappa, mu, BC, gauge=gauge)
    return ctx.cvc_gradient(src, sp=1e-27, force=False)[0]


@pytest.mark.parametrize("dims", [(3, 2, 5, 3), (2, 3, 3, 5)])
def test_force_on_ragged_lattices(chip, dims):
    print(f"gradient {dims}", flush=True)
    kappa, mu, src, h = 0.14, 0.05, (1, 0, 2, 1), 1e-5
    g = chip.gauge_random(dims, 8, 0.3)
    ctx = chip.Context(dims, kappa, mu, BC, gauge=g)
    _, dmu, F, _ = ctx.cvc_gradient(src, sp=1e-27)
    fd = (value(chip, dims, kappa, mu + h, g, src) - value(chip, dims, kappa, mu - h, g, src)) / (2 * h)
    assert abs(fd - dmu) < 1e-6 * max(1., abs(dmu))
    rng = np.random.default_rng(2)
    V = int(np.prod(dims))
    U = (g[..., 0::2] + 1j * g[..., 1::2]).reshape(V, 4, 3, 3)
    for site, rho in ((V - 1, 0), (V - 1, 3), (V // 2, 1), (0, 2)):
        A = rng.standard_normal((3, 3)) + 1j * rng.standard_normal((3, 3))
        T = (A + A.conj().T) / 2
        T -= np.trace(T) / 3 * np.eye(3)
        w, v = np.linalg.eigh(T)
        vals = []
        for s in (1, -1):
            W = U.copy()
            W[site, rho] = (v * np.exp(1j * s * h * w)) @ v.conj().T @ U[site, rho]
            gg = np.empty_like(g)
            gg[..., 0::2] = W.reshape(V, 4, 9).real
            gg[..., 1::2] = W.reshape(V, 4, 9).imag
            vals.append(value(chip, dims, kappa, mu, gg, src))
        fd, an = (vals[0] - vals[1]) / (2 * h), np.trace(T @ F[site, rho]).real
        assert abs(fd - an) < 1e-6 * max(1., abs(an)), (site, rho, fd, an)
