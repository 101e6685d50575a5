"""What a program built on this package spends its time on, as single calls.

Each case is one call (or one short sequence of calls) through the public
entry points of `lmx`: operator applications in the library layout and in the
reference's padded storage, the refresh after a link update, the reverse
rules, the fermion force, the FP64 solver, the mixed multi-RHS solver and the
generation of sources.  Sizes are those of this repository's configurations
(16^4, 24^3 x 48, 32^4, 48^3 x 96), of its tests (8^3 x 16, 16^3 x 32) and odd,
ragged ones of the same range.  Boundary phases are (1, 1, 1, -1) throughout.

`exact` restates the operators on torch tensors in 64 bits (dense gamma
matrices, rolls along the axes), without the package.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "latticematrices.jl_amd"))

import lmx  # noqa: E402

PHASES = (1, 1, 1, -1)


def listed():
    return [
        # smallest call: one D psi on a lattice of 8192 sites (thermalisation and debugging runs)
        dict(name="apply_8x8x8x16", kind="apply", dims="8x8x8x16", dtype="f64", dagger=False, csw=0.0, nrhs=1),
        # one FP64 D psi at the benchmark's lattice: measurements, residual checks
        dict(name="apply_32x32x32x32", kind="apply", dims="32x32x32x32", dtype="f64", dagger=False, csw=0.0, nrhs=1),
        # ComplexF32 fields on a lattice with no power of two in it, four sources at once
        dict(name="apply_f32_18x20x22x30", kind="apply", dims="18x20x22x30", dtype="f32", dagger=True, csw=0.0, nrhs=4),
        # the largest volume: D^dagger D with the clover term
        dict(name="ddagd_clover_48x48x48x96", kind="ddagd", dims="48x48x48x96", dtype="f64", csw=1.0, nrhs=1),
        # D psi in place on the arrays of a host program in the reference's storage
        dict(name="padded_24x24x24x48", kind="padded", dims="24x24x24x48", dtype="f64", dagger=False, csw=0.0, nrhs=1),
        # molecular dynamics: the links have changed, the next D psi refreshes the clover term first
        dict(name="refresh_clover_24x24x24x48", kind="refresh", dims="24x24x24x48", csw=1.0),
        # forward and backward of D(U) psi with the clover term
        dict(name="grad_clover_16x16x16x32", kind="grad", dims="16x16x16x32", csw=1.0, nrhs=1),
        # fermion force of one molecular-dynamics step (solve, reverse rule, projection)
        dict(name="force_16x16x16x16", kind="force", dims="16x16x16x16", links="haar", kappa=0.125, csw=0.0),
        # FP64 solve on a small lattice
        dict(name="solve_f64_8x8x8x16", kind="solve", dims="8x8x8x16", precision="f64", kappa=0.122, nrhs=1, tune=False),
        # the benchmark: twelve sources, 16-bit inner vectors, launch shape tuned beforehand
        dict(name="solve_h16_32x32x32x32_x12", kind="solve", dims="32x32x32x32", precision="h16", kappa=0.124, nrhs=12,
             tune=True),
        # a batch of four sources with FP32 inner vectors, without tuning
        dict(name="solve_f16_24x24x24x48_x4", kind="solve", dims="24x24x24x48", precision="f16", kappa=0.1235, nrhs=4,
             tune=False),
        # the twelve Gaussian sources of such a solve
        dict(name="sources_32x32x32x32_x12", kind="sources", dims="32x32x32x32", nrhs=12),
    ]


def _draw_dims(rng, lo, hi):
    """Extents with a volume between lo and hi (log-uniform): half of them multiples of four, half any integers."""
    for _ in range(1000):
        V = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        step = rng.choice((1, 4))
        d = [max(4, step * round(V ** 0.25 * math.exp(rng.uniform(-0.25, 0.25)) / step)) for _ in range(3)]
        d.append(max(4, step * round(V / (d[0] * d[1] * d[2]) / step)))
        if lo <= math.prod(d) <= hi and d[3] <= 8 * d[0]:
            return "x".join(map(str, d))
    return "12x12x12x24"


def draw(rng):
    kind = rng.choice(("apply", "apply", "ddagd", "padded", "refresh", "grad", "force", "solve", "solve", "sources"))
    csw = rng.choice((0.0, 1.0))
    if kind == "apply":
        nrhs = rng.choice((1, 1, 2, 3, 4, 12))
        return dict(kind=kind, dims=_draw_dims(rng, 4096, 4000000 // nrhs), dtype=rng.choice(("f64", "f32")),
                    dagger=rng.random() < 0.5, csw=csw, nrhs=nrhs)
    if kind == "ddagd":
        return dict(kind=kind, dims=_draw_dims(rng, 4096, 10000000), dtype="f64", csw=csw, nrhs=1)
    if kind == "padded":
        return dict(kind=kind, dims=_draw_dims(rng, 4096, 3000000), dtype=rng.choice(("f64", "f32")),
                    dagger=rng.random() < 0.5, csw=csw, nrhs=rng.choice((1, 1, 2)))
    if kind == "refresh":
        return dict(kind=kind, dims=_draw_dims(rng, 4096, 2000000), csw=1.0)
    if kind == "grad":
        return dict(kind=kind, dims=_draw_dims(rng, 4096, 1000000), csw=csw, nrhs=rng.choice((1, 2)))
    if kind == "force":
        links = rng.choice(("haar", "weak"))
        return dict(kind=kind, dims=_draw_dims(rng, 4096, 300000), links=links,
                    kappa=round(rng.uniform(0.115, 0.123), 4), csw=csw if links == "weak" else 0.0)
    if kind == "sources":
        nrhs = rng.choice((1, 4, 12))
        return dict(kind=kind, dims=_draw_dims(rng, 4096, 12000000 // nrhs), nrhs=nrhs)
    precision = rng.choice(("f64", "h16", "h16", "f16", "f32"))
    nrhs = 1 if precision == "f64" else rng.choice((1, 2, 4, 5, 12))
    return dict(kind=kind, dims=_draw_dims(rng, 4096, 300000 if precision == "f64" else 3000000 // nrhs),
                precision=precision, kappa=round(rng.uniform(0.115, 0.1235), 4), nrhs=nrhs, tune=False)


def _dims(case):
    return tuple(int(v) for v in case["dims"].split("x"))


def _kappa(case):
    return case.get("kappa", 0.124)


def _device():
    return torch.device("cuda", torch.cuda.current_device())


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _mm(a, b):
    """Products of 3 x 3 matrices, the matrix indices first."""
    return torch.stack([torch.stack([a[i, 0] * b[0, j] + a[i, 1] * b[1, j] + a[i, 2] * b[2, j] for j in range(3)])
                        for i in range(3)])


def _weak(n, eps, g):
    """n links exp(i eps H), H = sum_a h_a lambda_a / 2 with h_a ~ N(0, 1): complex [3, 3, n]."""
    h = torch.randn((8, n), dtype=torch.float64, device=_device(), generator=g) * (0.5 * eps * 0.5)  # half the exponent
    o = torch.zeros_like(h[0])
    s = h[7] / math.sqrt(3.0)
    re = torch.stack([torch.stack([h[2] + s, h[0], h[3]]), torch.stack([h[0], s - h[2], h[5]]),
                      torch.stack([h[3], h[5], -2.0 * s])])
    im = torch.stack([torch.stack([o, -h[1], -h[4]]), torch.stack([h[1], o, -h[6]]), torch.stack([h[4], h[6], o])])
    a = torch.complex(-im, re)
    one = torch.eye(3, dtype=a.dtype, device=a.device)[:, :, None]
    u = one + a / 12
    for k in range(11, 0, -1):
        u = one + _mm(a, u) / k
    return _mm(u, u)


def _haar(n, g):
    """n Haar-random SU(3) matrices (Gram-Schmidt of Gaussian rows, the third the conjugate cross product)."""
    z = torch.randn((2, 3, n, 2), dtype=torch.float64, device=_device(), generator=g)
    z = torch.view_as_complex(z)
    a = z[0] / z[0].abs().square().sum(0).sqrt()
    b = z[1] - a * (a.conj() * z[1]).sum(0)
    b = b / b.abs().square().sum(0).sqrt()
    c = torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]).conj()
    return torch.stack([a, b, c])


def _links(case, seed):
    """Links as complex [4, 3, 3, V], sites x-fastest."""
    V = math.prod(_dims(case))
    g = _gen(1000003 * seed + 1)
    u = torch.empty((4, 3, 3, V), dtype=torch.complex128, device=_device())
    for mu in range(4):
        for s in range(0, V, 1 << 21):
            n = min(1 << 21, V - s)
            u[mu, :, :, s:s + n] = _haar(n, g) if case.get("links") == "haar" else _weak(n, 0.2, g)
    return u


def _spinors(case, seed, n, which=0):
    """Gaussian spinors, sigma = sqrt(1/2): complex [n, 12, V]."""
    V = math.prod(_dims(case))
    z = torch.randn((n, 12, V, 2), dtype=torch.float64, device=_device(), generator=_gen(1000003 * seed + 2 + which))
    return torch.view_as_complex(z.mul_(math.sqrt(0.5)))


def _gauge(lat, u):
    return lmx.GaugeField(lat, torch.view_as_real(u.reshape(4, 9, lat.V)).contiguous())


def _spinor(lat, z):
    return lmx.SpinorField(lat, z.shape[0], torch.view_as_real(z).contiguous())


def _core(case, z):
    """Spinors [n, 12, V] as core arrays in the reference's order, C order [n, L4, L3, L2, L1, 4, 3]."""
    return z.movedim(1, -1).reshape((z.shape[0],) + tuple(reversed(_dims(case))) + (4, 3)).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    lat = lmx.Lattice(_dims(case), PHASES)
    s = dict(case=case, lat=lat)
    if kind == "sources":
        s["keys"] = [lmx.RNGStreamKey(seed + 1 + r) for r in range(case["nrhs"])]
        s["x"] = lat.spinor(case["nrhs"])
        return s
    csw = case.get("csw", 0.0)
    U = s["U"] = _gauge(lat, _links(case, seed))
    D = s["D"] = lmx.WilsonDiracOperator4D(U, _kappa(case), csw)
    n = case.get("nrhs", 1)
    z = _spinors(case, seed, n)
    if kind == "padded":
        z = z if case["dtype"] == "f64" else z.to(torch.complex64)
        s["psi"] = torch.stack([lmx.lattice_matrix(lat, c.contiguous(), nw=1) for c in _core(case, z)])
        s["out"] = torch.zeros_like(s["psi"])
    elif kind == "apply" and case["dtype"] == "f32":
        s["psi"] = torch.view_as_real(z.to(torch.complex64)).contiguous()
        s["out"] = lmx.spinor_f32(lat, n)
    else:
        s["psi"], s["out"] = _spinor(lat, z), lat.spinor(n)
    if kind in ("apply", "padded"):
        s["A"] = lmx.adjoint(D) if case["dagger"] else D
        if case["dtype"] == "f32":
            # the single-precision copies of the links are built on the first use of the operator
            (lmx.mul_f32_(s["out"], s["A"], s["psi"]) if kind == "apply" else
             lmx.mul_padded_(s["out"], s["A"], s["psi"], nw=1))
    elif kind == "ddagd":
        s["A"] = lmx.DdagDOp(D, lat.spinor(n))
    elif kind == "grad":
        s["cot"] = torch.view_as_real(_spinors(case, seed, n, 1)).contiguous()
        U.data.requires_grad_(True)
        s["psi"].data.requires_grad_(True)
    elif kind == "force":
        s["phi"] = lat.spinor()
        lmx.mul_(s["phi"], lmx.adjoint(D), s["psi"])
        s["G"], s["F"] = lmx.GaugeField(lat), lmx.GaugeField(lat)
    elif kind == "solve":
        s["x"], s["b"] = s.pop("out"), s.pop("psi")
        if case["precision"] == "f64":
            s["work"] = [lat.spinor() for _ in range(3)]
            s["A"] = lmx.DdagDOp(D, lat.spinor())
        elif case["tune"]:
            lmx.autotune(D, case["precision"], n)
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "apply":
        if case["dtype"] == "f32":
            return lmx.mul_f32_(s["out"], s["A"], s["psi"])
        return lmx.mul_(s["out"], s["A"], s["psi"]).data
    if kind == "ddagd":
        return lmx.mul_(s["out"], s["A"], s["psi"]).data
    if kind == "padded":
        return lmx.mul_padded_(s["out"], s["A"], s["psi"], nw=1)
    if kind == "refresh":
        s["U"].mark_halo_dirty_()
        return lmx.mul_cached_clover_(s["out"], s["D"], s["U"], s["psi"]).data
    if kind == "grad":
        out = lmx.wilson_apply_ad(s["D"], s["psi"])
        dlinks, dpsi = torch.autograd.grad(out, (s["U"].data, s["psi"].data), s["cot"])
        return out, dlinks, dpsi
    if kind == "force":
        res, eta, chi = lmx.dSFdU(s["G"], s["D"], s["phi"], force=s["F"])
        return s["G"].data, s["F"].data, eta.data, chi.data
    if kind == "sources":
        return lmx.randomize_gaussian_matrix_(s["x"], s["keys"], sigma=math.sqrt(0.5)).data
    lmx.clear_matrix_(s["x"])
    if case["precision"] == "f64":
        lmx.solve_(s["x"], s["A"], s["b"], *s["work"])
    else:
        lmx.cg_batched_(s["x"], s["D"], s["b"], precision=case["precision"], use_graph=True)
    return s["x"].data


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _iterations(case):
    """About how many iterations conjugate gradients needs to 1e-10: the condition number of D from kappa, the links'
    disorder and the antiperiodic direction."""
    k = _kappa(case)
    lost = 0.47 if case.get("links") == "haar" else 0.053
    low = 1 - 8 * k * (1 - lost) + k * (math.pi / _dims(case)[3]) ** 2
    return 0.5 * math.log(2e10) * (1 + 8 * k) / max(low, 0.02)


def work(case):
    V = math.prod(_dims(case))
    kind, n = case["kind"], case.get("nrhs", 1)
    clover = case.get("csw", 0.0) != 0.0
    e = 8 if case.get("dtype") == "f32" else 16  # bytes of a complex number
    apply_b = V * (36 * e + 24 * e * n + (27 * e if clover else 0))
    apply_f = V * n * (1368 + (600 if clover else 0))
    if kind in ("apply", "padded"):
        return {"bytes": apply_b, "flops": apply_f}
    if kind == "ddagd":
        return {"bytes": 2 * apply_b, "flops": 2 * apply_f}
    build_f = V * 6 * 4 * 3 * 216  # four leaves of three products in each of six planes
    if kind == "refresh":
        return {"bytes": V * 16 * (36 + 27 + 24), "flops": build_f + apply_f}
    if kind == "grad":
        # forward: links, psi, out; backward: the cotangent and psi in, both gradients out
        return {"bytes": V * 16 * (36 + 24 * n + 24 * n + 36 + 12 * n),
                "flops": 2 * apply_f + V * n * 1200 + (2 * build_f if clover else 0)}
    if kind == "sources":
        return {"bytes": V * 192 * n, "flops": V * n * 12 * 60}
    its = _iterations(case)
    if kind == "force" or case["precision"] == "f64":
        # an iteration: D and D^dagger, the updates of x, r and p
        return {"bytes": its * (2 * apply_b + V * 192 * 9), "flops": its * (2 * apply_f + V * 12 * 24)}
    # an iteration of the mixed solver: D and D^dagger on the inner vectors, x, r, p and t read and written
    sp, lk = (52 if case["precision"] == "h16" else 96), (288 if case["precision"] == "f32" else 144)
    return {"bytes": its * V * (2 * lk + n * 8 * sp), "flops": its * n * V * (2 * 1368 + 12 * 24)}


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
# gamma_mu of the chiral basis: (column, value) of the one entry in each row
_GAMMA = (((3, -1j), (2, -1j), (1, 1j), (0, 1j)), ((3, -1), (2, 1), (1, 1), (0, -1)),
          ((2, -1j), (3, 1j), (0, 1j), (1, -1j)), ((2, -1), (3, -1), (0, -1), (1, -1)))


def _gamma(mu, psi):
    """gamma_mu psi, psi [n, 4, 3, T, Z, Y, X]."""
    return torch.stack([v * psi[:, c] for c, v in _GAMMA[mu]], 1)


def _fwd(f, mu):
    return torch.roll(f, -1, -1 - mu)


def _bwd(f, mu):
    return torch.roll(f, 1, -1 - mu)


def _phase(f, mu, edge):
    """The antiperiodic direction's sign on the slice that wrapped."""
    if PHASES[mu] == 1:
        return f
    sign = torch.ones(f.shape[-1 - mu], dtype=torch.float64, device=f.device)
    sign[edge] = PHASES[mu]
    return f * sign.reshape((-1,) + (1,) * mu)


def _mv(u, psi, dagger=False):
    """u psi or u^dagger psi on the colour index; u [3, 3, sites], psi [n, 4, 3, sites]."""
    pick = (lambda i, j: u[j, i].conj()) if dagger else (lambda i, j: u[i, j])
    return torch.stack([pick(i, 0) * psi[:, :, 0] + pick(i, 1) * psi[:, :, 1] + pick(i, 2) * psi[:, :, 2]
                        for i in range(3)], 2)


def _dag(a):
    return a.transpose(0, 1).conj()


def _planes(u):
    """F_mu,nu = (Q - Q^dagger) / 8 of the four leaves, by (mu, nu)."""
    out = {}
    for mu in range(4):
        for nu in range(mu + 1, 4):
            a, b = u[mu], u[nu]
            am, bm = _bwd(a, mu), _bwd(b, nu)  # links that end at x
            # x -> x+mu -> x+mu+nu -> x+nu -> x
            q = _mm(_mm(a, _fwd(b, mu)), _mm(_dag(_fwd(a, nu)), _dag(b)))
            # x -> x+nu -> x+nu-mu -> x-mu -> x
            q = q + _mm(_mm(b, _dag(_bwd(_fwd(a, nu), mu))), _mm(_dag(_bwd(b, mu)), am))
            # x -> x-mu -> x-mu-nu -> x-nu -> x
            q = q + _mm(_mm(_dag(am), _dag(_bwd(bm, mu))), _mm(_bwd(_bwd(a, mu), nu), bm))
            # x -> x-nu -> x-nu+mu -> x+mu -> x
            q = q + _mm(_mm(_dag(bm), _bwd(a, nu)), _mm(_bwd(_fwd(b, mu), nu), _dag(a)))
            out[mu, nu] = (q - _dag(q)) / 8
    return out


def _wilson(u, psi, kappa, dagger=False, planes=None, csw=0.0):
    """D psi or D^dagger psi; u [4, 3, 3, T, Z, Y, X], psi [n, 4, 3, T, Z, Y, X]."""
    hop = None
    for mu in range(4):
        f = _phase(_fwd(psi, mu), mu, -1)
        b = _phase(_bwd(psi, mu), mu, 0)
        gf, gb = _gamma(mu, f), _gamma(mu, b)
        term = _mv(u[mu], f + gf if dagger else f - gf) + _mv(_bwd(u[mu], mu), b - gb if dagger else b + gb, True)
        hop = term if hop is None else hop + term
    out = psi - kappa * hop
    if planes is not None:
        for (mu, nu), f in planes.items():
            out = out - (kappa * csw) * _gamma(mu, _gamma(nu, _mv(f, psi)))
    return out


def _operator(case, u):
    planes = _planes(u) if case.get("csw", 0.0) else None
    return lambda psi, dagger=False: _wilson(u, psi, _kappa(case), dagger, planes, case.get("csw", 0.0))


def _solution(D, b, most):
    """(D^dagger D)^-1 b by conjugate gradients far beyond the tolerance of the calls."""
    x, r = torch.zeros_like(b), b.clone()
    p, rr = r.clone(), r.abs().square().sum()
    for k in range(most):
        ap = D(D(p), True)
        alpha = rr / (p.conj() * ap).sum().real
        x, r = x + alpha * p, r - alpha * ap
        new = r.abs().square().sum()
        if k % 16 == 15 and float(new) < 1e-29 * float(b.abs().square().sum()):
            break
        p, rr = r + (new / rr) * p, new
    return x


def _flat(z):
    """[n, 4, 3, T, Z, Y, X] as the library's [n, 12, V, 2]."""
    return torch.view_as_real(z.reshape(z.shape[0], 12, -1))


def exact(case, seed):
    kind, n = case["kind"], case.get("nrhs", 1)
    V, its = math.prod(_dims(case)), _iterations(case)
    if kind == "sources" or (kind in ("solve", "force") and its * V * n > 1.5e8):
        return None
    sites = tuple(reversed(_dims(case)))
    u = _links(case, seed).reshape((4, 3, 3) + sites)
    z = _spinors(case, seed, n)
    if case.get("dtype") == "f32":
        z = z.to(torch.complex64).to(torch.complex128)
    psi = z.reshape((n, 4, 3) + sites)
    if kind == "grad":
        u.requires_grad_(True)
        psi.requires_grad_(True)
        out = _operator(case, u)(psi)
        cot = _spinors(case, seed, n, 1).reshape(out.shape)
        du, dpsi = torch.autograd.grad(out, (u, psi), cot)
        return _flat(out.detach()), torch.view_as_real(du.reshape(4, 9, V)), _flat(dpsi)
    D = _operator(case, u)
    if kind in ("apply", "refresh"):
        return _flat(D(psi, case.get("dagger", False)))
    if kind == "ddagd":
        return _flat(D(D(psi), True))
    if kind == "padded":
        out = torch.zeros((n,) + tuple(v + 2 for v in sites) + (4, 3), dtype=torch.complex128, device=u.device)
        out[:, 1:-1, 1:-1, 1:-1, 1:-1] = _core(case, D(psi, case["dagger"]).reshape(n, 12, V))
        return out
    if kind == "solve":
        return _flat(_solution(D, psi, int(6 * its)))
    eta = _solution(D, D(psi, True), int(6 * its))
    chi = D(eta)
    # dS = -2 Re <chi, dD eta>: the gradient of that functional of the links
    v = u.clone().requires_grad_(True)
    s = -2.0 * (chi.conj() * _operator(case, v)(eta)).sum().real
    (g,) = torch.autograd.grad(s, v)
    f = torch.empty_like(u)
    one = torch.eye(3, dtype=u.dtype, device=u.device).reshape((3, 3, 1, 1, 1, 1))
    for mu in range(4):
        m = _mm(u[mu], _dag(g[mu]))
        m = 0.5 * (m - _dag(m))
        f[mu] = m - one * ((m[0, 0] + m[1, 1] + m[2, 2]) / 3)
    return (torch.view_as_real(g.reshape(4, 9, V)), torch.view_as_real(f.reshape(4, 9, V)), _flat(eta), _flat(chi))
