"""Workloads of the propagator-and-contraction library as its programs run them.

The library's work is, in the order of the time that programs spend in it: batched
solves for propagators (twisted-mass Wilson operator inside), the operator by itself,
the contraction of a source's 120 propagators to Pi_{mu nu}(x), whole sources, meson
two-point functions, the adjoint gradient, and single operator applications and solves
on a program's own host arrays (the drop-in functions).  Lattices run from 4^4 to
64 x 32^3, right-hand sides from 1 to 48; links are exp(i 0.3 H), time is antiperiodic.

`exact` is a restatement in plain torch, 64 bits: the operator as shifts and 3x3 colour
products, solutions by conjugate gradients on the normal equations, the contraction from
its definition, the gradient by automatic differentiation of that definition.
"""
import ctypes
import math

import numpy as np
import torch

import cvc_amd

BC = (1.0, 0.0, 0.0, 0.0)
PREC = {"f64": cvc_amd.PREC_F64, "f32": cvc_amd.PREC_F32, "f16": cvc_amd.PREC_F16}
DIMS = ("T", "LX", "LY", "LZ")


def _case(name, kind, dims, **more):
    c = {"name": name, "kind": kind, **dict(zip(DIMS, dims)), "kappa": 0.1632, "mu": 0.004}
    c.update(more)
    return c


def listed():
    return [
        # a reference program calling Q_phi_tbc on its own arrays, on a test-size lattice: latency
        _case("operator_host_8x8x8x8", "operator_host", (8, 8, 8, 8)),
        # one solution checked or one column propagated on resident fields
        _case("operator_1rhs_48x24", "operator", (48, 24, 24, 24), nrhs=1, prec="f64"),
        # the benchmark's operator: the 12 spin-colour columns of a point source
        _case("operator_12rhs_64x32", "operator", (64, 32, 32, 32), nrhs=12, prec="f64"),
        # the drop-in invert_Qtm: one column on host arrays, a small lattice far from criticality
        _case("solve_host_8x8x8x8", "solve_host", (8, 8, 8, 8), kappa=0.14, mu=0.01, iters=25),
        # the reference's own algorithm on a propagator's 12 columns, FP64 throughout
        _case("solve_f64_32x16", "solve", (32, 16, 16, 16), nrhs=12, prec="f64", eo=False, iters=150),
        # the same with FP32 inside and even/odd preconditioning, a lattice of no powers of two
        _case("solve_f32_eo_28x18x14x20", "solve", (28, 18, 14, 20), nrhs=12, prec="f32", eo=True, iters=50),
        # the production setting: FP16 inside, even/odd
        _case("solve_f16_eo_40x20", "solve", (40, 20, 20, 20), nrhs=12, prec="f16", eo=True, iters=50),
        # four source positions batched in one call, FP32 inside
        _case("solve_f32_eo_48rhs_24x14", "solve", (24, 14, 14, 16), nrhs=48, prec="f32", eo=True, iters=50),
        # 120 resident propagators to Pi_{mu nu}(x) and the contact term
        _case("contract_40x20", "contract", (40, 20, 20, 20)),
        # a meson correlator with sink momentum from two resident propagators
        _case("twopoint_64x32", "twopoint", (64, 32, 32, 32), idsource=5, idsink=5),
        # a whole source: 120 solves and the contraction, production setting
        _case("source_16x8", "source", (16, 8, 8, 8), prec="f16", eo=True, kappa=0.163, mu=0.01, iters=50),
        # value and gradient (mass and every link) of the vacuum polarisation: forward and adjoint solves
        _case("gradient_8x8x8x8", "gradient", (8, 8, 8, 8), prec="f64", eo=True, kappa=0.163, mu=0.01, iters=50),
    ]


# most sites x right-hand sides a drawn case of each kind has
LARGEST = {"operator_host": 1 << 20, "operator": 64 * 32**3 * 12, "solve_host": 1 << 15, "solve": 24 * 14 * 14 * 16 * 48,
           "contract": 40 * 20**3, "twopoint": 64 * 32**3, "source": 16 * 8**3, "gradient": 8**4}


def draw(rng):
    kind = rng.choice(("operator_host", "operator", "operator", "solve_host", "solve", "solve", "solve", "contract",
                       "twopoint", "source", "gradient"))
    c = {"kind": kind, "kappa": 0.163, "mu": 0.01}
    if kind == "solve_host":
        c["kappa"] = 0.14
    if kind == "operator":
        c.update(nrhs=rng.choice((1, 2, 3, 4, 6, 8, 12, 12, 16, 24, 48)), prec=rng.choice(("f64", "f64", "f32")))
    elif kind == "solve":
        c.update(nrhs=rng.choice((1, 4, 12, 12, 12, 24)), prec=rng.choice(("f64", "f64", "f32", "f16")))
        c["eo"] = c["prec"] != "f64" or rng.random() < 0.4     # FP32 and FP16 inside go with even/odd
    elif kind == "twopoint":
        c.update(idsource=rng.randrange(16), idsink=rng.randrange(16))
    elif kind in ("source", "gradient"):
        c.update(prec=rng.choice(("f64", "f32", "f16")) if kind == "source" else "f64", eo=True)
    most = LARGEST[kind] // c.get("nrhs", 1)
    if kind == "twopoint":
        c["idsink"] = c["idsource"]
    while True:
        edge = math.exp(rng.uniform(math.log(256), math.log(most))) ** 0.25
        dims = [max(4, round(edge * math.exp(rng.uniform(-0.35, 0.35)))) for _ in DIMS]
        if c.get("eo"):
            dims = [L + L % 2 for L in dims]     # the parities alternate around the torus
        if math.prod(dims) <= most and max(dims) <= 64:
            break
    c.update(zip(DIMS, dims))
    if kind in ("solve", "solve_host", "source", "gradient"):
        c["iters"] = 25 if kind == "solve_host" else 50 if c["eo"] else 150
    return c


def _dims(case):
    return tuple(case[d] for d in DIMS)


class _SetHead(ctypes.Structure):
    """The head of a resident set (struct cvchip_field): size, precision, sites, device address."""
    _fields_ = [("nrhs", ctypes.c_int), ("prec", ctypes.c_int), ("V", ctypes.c_int64), ("data", ctypes.c_void_p)]


class _DeviceArray:
    def __init__(self, address, shape, typestr):
        self.__cuda_array_interface__ = {"data": (address, False), "shape": shape, "typestr": typestr, "version": 2}


def _view(field):
    """A set's device memory as a tensor, in the library's layout: [12][V][nrhs] complex in FP64,
    [6][V][nrhs] pairs of complex in FP32 (component 3 spin + colour).  The tensor keeps the set
    (and, through it, its context) alive: the memory goes back when the set does."""
    h = _SetHead.from_address(field._h.value)
    shape, kind = ((12, h.V, h.nrhs, 2), "<f8") if h.prec == cvc_amd.PREC_F64 else ((6, h.V, h.nrhs, 2, 2), "<f4")
    t = torch.as_tensor(_DeviceArray(h.data, shape, kind), device="cuda")
    assert t.data_ptr() == h.data, "a copy, not a view"
    t.owner = field
    return t


def _source_point(case, seed):
    rng = np.random.default_rng([seed, 7])
    return tuple(int(rng.integers(0, L)) for L in _dims(case))


def _source_points(case, seed, n):
    rng = np.random.default_rng([seed, 7])
    return [tuple(int(rng.integers(0, L)) for L in _dims(case)) for _ in range(n)]


def prepare(case, seed):
    kind, dims = case["kind"], _dims(case)
    V = math.prod(dims)
    torch.cuda.init()
    gauge = None if kind == "twopoint" else cvc_amd.gauge_random(dims, seed, 0.3)
    ctx = cvc_amd.Context(dims, case["kappa"], case["mu"], BC, gauge=gauge)
    st = {"kind": kind, "ctx": ctx, "case": case}
    if kind == "operator_host":
        st["gauge"], st["phi"] = gauge, np.random.default_rng(seed).standard_normal((V, 24))
        st["xi"] = np.zeros((V, 24))
    elif kind == "operator":
        start = ctx.field(case["nrhs"])
        start.fill_random(seed)
        st["in"], st["out"] = start, ctx.field(case["nrhs"], PREC[case["prec"]])
        if case["prec"] != "f64":
            st["in"] = ctx.field(case["nrhs"], PREC[case["prec"]])
            st["in"].copy_from(start)
        st["view"], st["in_view"] = _view(st["out"]), _view(st["in"])
    elif kind == "solve_host":
        t, x, y, z = _source_point(case, seed)
        site = ((t * dims[1] + x) * dims[2] + y) * dims[3] + z
        st["b"] = cvc_amd.point_source(V, site, seed % 4, seed % 3)
    elif kind == "solve":
        n = case["nrhs"]
        points = _source_points(case, seed, -(-n // 12))
        st["x"], st["b"] = ctx.field(n), ctx.field(n)
        whole = ctx.field(12 * len(points))
        whole.point_sources(points)
        st["b"].copy_columns(0, whole, 0, n)
        st["view"], st["b_view"] = _view(st["x"]), _view(st["b"])
    elif kind == "contract":
        st["up"], st["dn"], st["src"] = ctx.field(60), ctx.field(60), _source_point(case, seed)
        st["up"].fill_random(2 * seed)
        st["dn"].fill_random(2 * seed + 1)
    elif kind == "twopoint":
        st["chi"], st["phi"], st["src"] = ctx.field(12), ctx.field(12), _source_point(case, seed)
        st["chi"].fill_random(2 * seed)
        st["phi"].fill_random(2 * seed + 1)
        _view(st["phi"]).mul_(0.5).add_(_view(st["chi"]))     # two columns of one correlated ensemble
        torch.cuda.synchronize()
        st["mom"] = tuple(int(v) for v in np.random.default_rng([seed, 9]).integers(0, 2, 3))
    else:
        st["src"] = _source_point(case, seed)
        ctx.set_solver_flags(cvc_amd.SOLVE_EO if case["eo"] else 0)
    return st


def _delta(case):
    return {"f64": 0.1, "f32": 0.001, "f16": 0.02 if case["eo"] else 0.1}[case["prec"]]


TOL = 1e-24     # squared relative residual


def run(st):
    kind, ctx, case = st["kind"], st["ctx"], st["case"]
    if kind == "operator_host":
        return ctx.Q_phi(st["phi"], out=st["xi"])
    if kind == "operator":
        ctx.dslash(st["out"], st["in"])
        return st["view"]
    if kind == "solve_host":
        return ctx.invert_Qtm(st["b"], TOL, 2000)[1]
    if kind == "solve":
        st["x"].zero()
        ctx.invert_her(st["x"], st["b"], TOL, 20000, prec=PREC[case["prec"]], delta=_delta(case), eo=case["eo"])
        return st["view"]
    if kind == "contract":
        return ctx.field_cvc_contract(st["up"], st["dn"], st["src"])
    if kind == "twopoint":
        return ctx.field_contract_twopoint(case["idsource"], case["idsink"], st["chi"], st["phi"], snk_mom=st["mom"],
                                           src=st["src"])
    if kind == "source":
        return ctx.cvc_source(st["src"], TOL, 20000, PREC[case["prec"]], _delta(case))[:2]
    value, dmu, force, _ = ctx.cvc_gradient(st["src"], sp=TOL, niter_max=20000, prec=PREC[case["prec"]],
                                            delta=_delta(case))
    return value, dmu, force


COMPLEX_BYTES = {"f64": 16, "f32": 8, "f16": 4 + 4 / 12}     # a stored spinor component (FP16: and its share of the scale)


def _operator_work(V, N, prec):
    return V * (24 * N * COMPLEX_BYTES[prec] + (576 if prec == "f64" else 192)), V * N * 1416


def _solve_work(case, V, N):
    """`iters` BiCGStab iterations on gamma5 D gamma5 D: four operator applications (on the even/odd
    system four of half the sites each way), and p, r, s, t, Ap, x, r^ once read or written in each of
    the three vector updates (13 passes)."""
    b, f = _operator_work(V, N, case["prec"])
    sites = V / 2 if case["eo"] else V
    per_it = 4 * b + 13 * 12 * sites * N * COMPLEX_BYTES[case["prec"]]
    return case["iters"] * per_it, case["iters"] * (4 * f + 6 * 96 * sites * N)


def work(case):
    kind, V = case["kind"], math.prod(_dims(case))
    if kind == "operator_host":
        b, f = _operator_work(V, 1, "f64")
    elif kind == "operator":
        b, f = _operator_work(V, case["nrhs"], case["prec"])
    elif kind == "solve_host":
        b, f = (case["iters"] * v for v in (2 * _operator_work(V, 1, "f64")[0] + 13 * 192 * V, 3500 * V))
    elif kind == "solve":
        b, f = _solve_work(case, V, case["nrhs"])
    else:
        # 120 columns, links and conn once; per (mu, nu) 2 x 24 products of a link, a vertex and a dot product
        contract = V * (120 * 192 + 576 + 256), V * 16 * 48 * (264 + 144 + 96)
        if kind == "twopoint":
            b, f = V * 2 * 12 * 192, V * 12 * 12 * 14
        elif kind == "contract":
            b, f = contract
        else:
            solve = _solve_work(case, V, 120)
            b, f = contract[0] + solve[0], contract[1] + solve[1]
            if kind == "gradient":
                b, f = 2 * b, 2 * f
    return {"bytes": b, "flops": f}


# --------------------------------------------------------------- plain torch, 64 bits

_I = 1j
_G = [[(2, -1), (3, -1), (0, -1), (1, -1)], [(3, -_I), (2, -_I), (1, _I), (0, _I)],
      [(3, -1), (2, 1), (1, 1), (0, -1)], [(2, -_I), (3, _I), (0, _I), (1, -_I)]]     # (column, value) of each row


def _gamma(mu):
    g = torch.zeros(4, 4, dtype=torch.complex128)
    for a, (col, v) in enumerate(_G[mu]):
        g[a, col] = v
    return g


_G5 = torch.diag(torch.tensor([1, 1, -1, -1], dtype=torch.complex128))
_ONE = torch.eye(4, dtype=torch.complex128)


def _links(case, seed, dev):
    """Links with the boundary phase, [4][3][3][T][LX][LY][LZ]."""
    dims = _dims(case)
    g = torch.from_numpy(cvc_amd.gauge_random(dims, seed, 0.3)).to(dev)
    u = torch.view_as_complex(g.view(*dims, 4, 3, 3, 2)).permute(4, 5, 6, 0, 1, 2, 3).contiguous()
    ph = torch.tensor([complex(math.cos(math.pi * b / L), math.sin(math.pi * b / L)) for b, L in zip(BC, dims)],
                      dtype=torch.complex128)
    return u * ph.to(dev).view(4, 1, 1, 1, 1, 1, 1)


def _colour(u, h, dag=False):
    """u h (dag: u^+ h) on colour: u [3][3][sites], h [spin][3][sites][columns]."""
    w = u.conj().transpose(0, 1) if dag else u
    return torch.stack([sum(w[i, j].unsqueeze(-1) * h[:, j] for j in range(3)) for i in range(3)], 1)


def _shift(f, mu, step, first):
    """f(x + step mu); `first` is the index of the time axis."""
    return torch.roll(f, -step, first + mu)


def _operator(u, psi, kappa, mu):
    """D psi, psi [4][3][T][LX][LY][LZ][columns]."""
    hop = torch.zeros_like(psi)
    for m in range(4):
        for sign, dag in ((-1, False), (1, True)):
            h = torch.stack([psi[a] + sign * _G[m][a][1] * psi[_G[m][a][0]] for a in (0, 1)])
            if dag:
                w = _shift(_colour(u[m], h, True), m, -1, 2)
            else:
                w = _colour(u[m], _shift(h, m, 1, 2))
            hop[:2] += w
            for a in (2, 3):
                hop[a] += sign * _G[m][a][1] * w[_G[m][a][0]]
    out = psi / (2 * kappa) - 0.5 * hop
    out[:2] += 1j * mu * psi[:2]
    out[2:] -= 1j * mu * psi[2:]
    return out


def _g5(psi):
    return torch.cat((psi[:2], -psi[2:]))


def _solve(u, b, kappa, mu, tol=1e-28):
    """D x = b by conjugate gradients on D^+ D, all columns at once."""
    normal = lambda v: _g5(_operator(u, _g5(_operator(u, v, kappa, mu)), kappa, -mu))  # noqa: E731
    dot = lambda v: torch.view_as_real(v).square().sum(-1).flatten(0, -2).sum(0)  # noqa: E731
    x, r = torch.zeros_like(b), _g5(_operator(u, _g5(b), kappa, -mu))
    p, rr = r.clone(), dot(r)
    stop = tol * rr
    for _ in range(5000):
        q = normal(p)
        a = rr / (p.conj() * q).real.flatten(0, -2).sum(0)
        a = torch.where(rr > 0, a, torch.zeros_like(a))
        x += a * p
        r -= a * q
        new = dot(r)
        if bool((new <= stop).all()):
            break
        p = r + torch.where(rr > 0, new / rr, torch.zeros_like(rr)) * p
        rr = new
    return x


def _unpack(view, dims):
    """A set's layout as complex128 [4][3][T][LX][LY][LZ][columns]."""
    if view.dtype == torch.float32:
        view = view.permute(0, 3, 1, 2, 4).reshape(12, view.shape[1], view.shape[2], 2)
    return torch.view_as_complex(view.double().contiguous()).view(4, 3, *dims, -1)


def _pack(psi, like_f32):
    v = torch.view_as_real(psi.reshape(12, -1, psi.shape[-1]))
    return v.view(6, 2, *v.shape[1:]).permute(0, 2, 3, 1, 4).contiguous() if like_f32 else v


def _points(dims, src, dev):
    """Point sources at y + 0^, .., y + 3^ and y, [4][3][sites][60]."""
    b = torch.zeros(12, *dims, 60, dtype=torch.complex128, device=dev)
    for s in range(5):
        x = [(c + (1 if s == m else 0)) % L for m, (c, L) in enumerate(zip(src, dims))]
        for k in range(12):
            b[k, x[0], x[1], x[2], x[3], 12 * s + k] = 1
    return b.view(4, 3, *dims, 60)


def _spin(g, v):
    return torch.einsum("ab,b...->a...", g.to(v.device), v)


def _contract(u, up, dn, src):
    """conn [sites][4 mu + nu] and the contact term [4] of columns up, dn [4][3][sites][60]."""
    dims, dev = up.shape[2:6], up.device
    y = tuple(src)
    conn, contact = [[None] * 4 for _ in range(4)], []
    for nu in range(4):
        us = u[(nu, slice(None), slice(None)) + y]
        yn = tuple((c + (m == nu)) % L for m, (c, L) in enumerate(zip(y, dims)))
        g = _gamma(nu) @ _G5
        g1 = torch.kron((g - _G5).to(dev), us.contiguous())
        g2 = torch.kron((g + _G5).to(dev), us.conj().transpose(0, 1).contiguous())
        own, far = slice(48, 60), slice(12 * nu, 12 * nu + 12)
        psi = torch.cat((dn[..., far] @ g1.conj().T, dn[..., own] @ g2.conj().T), -1)
        phi = torch.cat((up[..., own], up[..., far]), -1)
        for mu in range(4):
            m, p = _G5 @ (_gamma(mu) - _ONE), _G5 @ (_gamma(mu) + _ONE)
            t = (psi.conj() * _spin(m, _colour(u[mu], _shift(phi, mu, 1, 2)))).sum((0, 1, -1))
            t = t + (_shift(psi, mu, 1, 2).conj() * _spin(p, _colour(u[mu], phi, True))).sum((0, 1, -1))
            conn[mu][nu] = -0.25 * t.reshape(-1)
        a = torch.kron((_gamma(nu) - _ONE).to(dev), us.contiguous()) @ up[(slice(None), slice(None)) + yn].reshape(12, 60)[:, own]
        b = torch.kron((_gamma(nu) + _ONE).to(dev), us.conj().transpose(0, 1).contiguous()) @ up[(slice(None), slice(None)) + y].reshape(12, 60)[:, far]
        contact.append(-0.5 * torch.trace(a) + 0.5 * torch.trace(b))
    return torch.stack([conn[mu][nu] for mu in range(4) for nu in range(4)], -1), torch.stack(contact)


def _polarisation(conn, contact, dims, src, qmax=2.0):
    """sum over mu and |q| <= qmax of Re Pi_{mu mu}(q)."""
    n = torch.meshgrid(*[torch.arange(-((L - 1) // 2), L // 2 + 1, dtype=torch.float64) * (2 * math.pi / L)
                         for L in dims], indexing="ij")
    q = torch.stack([v.reshape(-1) for v in n], -1)
    q = q[q.square().sum(-1) <= qmax * qmax + 1e-12].to(conn.device)
    x = torch.meshgrid(*[torch.arange(L, dtype=torch.float64, device=conn.device) - c for L, c in zip(dims, src)],
                       indexing="ij")
    w = sum(torch.cos(torch.stack([v.reshape(-1) for v in x], -1) @ k) for k in q)
    return (w * conn[:, ::5].real.sum(-1)).sum() - len(q) * contact.real.sum()


def _gradient(u, case, src, dev):
    """Value, d/dmu and the traceless Hermitian F of dL = tr(T F) for U -> exp(i eps T) U.  Columns are
    implicit functions of the links: with G = dL/dS, dL = -Re <Lambda, dD S>, Lambda = D^{-+} G."""
    dims, kappa, mu = _dims(case), case["kappa"], case["mu"]
    b = _points(dims, src, dev)
    cols = [_solve(u, b, kappa, s * mu).requires_grad_() for s in (1, -1)]
    u = u.clone().requires_grad_()
    m = torch.tensor(mu, dtype=torch.float64, device=dev, requires_grad=True)
    conn, contact = _contract(u, cols[0], cols[1], src)
    value = _polarisation(conn, contact, dims, src)
    value.backward()
    for s, c in zip((1, -1), cols):
        lam = _g5(_solve(u.detach(), _g5(c.grad), kappa, -s * mu))
        for part in range(0, 60, 12):
            k = slice(part, part + 12)
            psi = c.detach()[..., k]
            d = torch.zeros_like(psi)
            for n in range(4):
                fwd = _colour(u[n], _shift(psi, n, 1, 2))
                bwd = _shift(_colour(u[n], psi, True), n, -1, 2)
                d = d - 0.5 * (fwd - _spin(_gamma(n), fwd) + bwd + _spin(_gamma(n), bwd))
            d = d + 1j * s * m * _g5(psi)
            (-(lam[..., k].conj() * d).real.sum()).backward()
    k = u.detach().permute(3, 4, 5, 6, 0, 1, 2).reshape(-1, 4, 3, 3)
    g = u.grad.permute(3, 4, 5, 6, 0, 1, 2).reshape(-1, 4, 3, 3)
    f = 1j * (k @ g.conj().transpose(-1, -2))                 # dL = Re tr(g^+ i T u) = Re tr(T f)
    f = 0.5 * (f + f.conj().transpose(-1, -2))
    f = f - torch.diagonal(f, dim1=-2, dim2=-1).sum(-1)[..., None, None] / 3 * torch.eye(3, device=dev)
    return float(value.detach()), float(m.grad), f


_GAMMAS = [_gamma(m) for m in range(4)] + [_ONE, _G5] + [_gamma(m) @ _G5 for m in range(4)]
_GAMMAS += [_gamma(a) @ _gamma(b) for a, b in ((0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3))]


def _twopoint(case, chi, phi, mom, src):
    """C(t) = sum_x e^{i p (x - y)} tr[(g5 G_src)^~ chi^+ g5 G_snk phi], signs as contract_twopoint's: an
    imaginary source gamma enters by its entries' imaginary parts and a factor -i."""
    dims, dev = _dims(case), chi.device
    gs = _GAMMAS[case["idsource"]]
    imag = bool(gs[0].imag.abs().sum() > 0)
    snk = _spin(_G5 @ _GAMMAS[case["idsink"]], phi)
    total = torch.zeros(dims, dtype=torch.complex128, device=dev)
    for m in range(4):
        col = int(gs[m].abs().argmax())
        s = complex(gs[m, col])
        s = (-s.imag if imag else s.real) * (1 if col < 2 else -1)
        total += s * (chi[..., 3 * col:3 * col + 3].conj() * snk[..., 3 * m:3 * m + 3]).sum((0, 1, -1))
    ang = [2 * math.pi * p / L * (torch.arange(L, dtype=torch.float64, device=dev) - c)
           for p, L, c in zip(mom, dims[1:], src[1:])]
    ph = torch.exp(1j * (ang[0][:, None, None] + ang[1][:, None] + ang[2]))
    c = (total * ph).sum((1, 2, 3))
    return -1j * c if imag else c


def exact(case, seed):
    kind, dims = case["kind"], _dims(case)
    dev = torch.device("cuda")
    kappa, mu = case["kappa"], case["mu"]
    if kind == "solve" and math.prod(dims) * case["nrhs"] > 40 * 20**3 * 12:
        return None
    st = prepare(case, seed)
    if kind == "twopoint":
        chi, phi = (_unpack(_view(st[k]), dims) for k in ("chi", "phi"))
        return _twopoint(case, chi, phi, st["mom"], st["src"])
    u = _links(case, seed, dev)
    if kind in ("operator_host", "solve_host"):
        v = torch.from_numpy(st["phi"] if kind == "operator_host" else st["b"]).to(dev)
        psi = torch.view_as_complex(v.view(-1, 12, 2)).T.reshape(4, 3, *dims, 1)
        out = _operator(u, psi, kappa, mu) if kind == "operator_host" else _solve(u, psi, kappa, mu)
        v = torch.view_as_real(out.reshape(12, -1).T.contiguous()).reshape(-1, 24)
        return v if kind == "operator_host" else v.unsqueeze(0)
    if kind == "operator":
        f32, v = case["prec"] == "f32", st["in_view"]
        parts = []
        for r in range(0, case["nrhs"], 4):     # four columns at a time: the shifts hold several copies
            parts.append(_pack(_operator(u, _unpack(v[:, :, r:r + 4], dims), kappa, mu), f32))
        return torch.cat(parts, 2)
    if kind == "solve":
        return _pack(_solve(u, _unpack(st["b_view"], dims), kappa, mu), False)
    if kind == "gradient":
        return _gradient(u, case, st["src"], dev)
    if kind == "contract":
        up, dn = (_unpack(_view(st[k]), dims) for k in ("up", "dn"))
    else:
        b = _points(dims, st["src"], dev)
        up, dn = (_solve(u, b, kappa, s * mu) for s in (1, -1))
    conn, contact = _contract(u, up, dn, st["src"])
    return torch.view_as_real(conn), contact
