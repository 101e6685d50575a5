"""The eight-wavefront stencil (FP64, one field or clover fields) against the
oracle, bit for bit, at the sizes where its blocks can go wrong: fewer sites
than a block, a last block cut by the lattice, slabs that divide the slice and
that do not, slices that end inside a block, complex phases; and the p.Ap sums
that it leaves per 64 sites through whole CG solves."""
import numpy as np
import pytest
import torch

import oracle as orc
import lmx
from lmx import generators as gen

pytestmark = pytest.mark.gpu

ANTI = (1, 1, 1, -1)
SHAPES = [
    ((2, 2, 2, 2), ANTI),                          # 16 sites: one block, 48 idle lanes
    ((3, 5, 3, 3), ANTI),                          # 135 sites: a cut last block, lattice order
    ((8, 8, 4, 3), ANTI),                          # slices of 4 whole blocks, no slabs
    ((8, 8, 8, 4), ANTI),                          # 8 blocks a slice: slabs of one block
    ((8, 8, 9, 4), ANTI),                          # 9 blocks: slabs of two and a tail slab of one
    ((13, 13, 13, 3), ANTI),                       # 2197 sites a slice: slices end inside a block, tail slab
    ((13, 13, 13, 2), (np.exp(0.3j), 1, -1j, -1)),  # the same with complex phases
]


@pytest.mark.parametrize("L,phases", SHAPES)
@pytest.mark.parametrize("flags", [0, 1, 2, 3])
def test_wilson(gpu, L, phases, flags):
    print(f"blocks L={L} flags={flags}", flush=True)
    U = gen.links(L, "haar", 31)
    psi = gen.gaussian_spinor(L, 32)
    lat = lmx.Lattice(L, phases)
    Ug = lat.gauge_from_numpy(U)
    A = lmx.WilsonDiracOperator4D_Donly(Ug) if flags & 2 else lmx.WilsonDiracOperator4D(Ug, 0.117)
    y = lat.spinor()
    lmx.mul_(y, lmx.adjoint(A) if flags & 1 else A, lat.spinor_from_numpy(psi))
    ref = orc.wilson(U, psi, L, 0.117, phases, dagger=bool(flags & 1), donly=bool(flags & 2))
    assert np.array_equal(y.to_numpy(), ref)


@pytest.mark.parametrize("nrhs", [2, 3, 13])  # even and odd numbers in turn; a second group of one
@pytest.mark.parametrize("donly", [False, True])
def test_fields_that_take_turns_in_a_workgroup(gpu, nrhs, donly):
    # from 512 blocks of 64 sites on, up to twelve fields share a workgroup; one field alone is the kernel above
    L = (9, 9, 13, 32)
    print(f"fields in turn L={L} nrhs={nrhs} donly={donly}", flush=True)
    lat = lmx.Lattice(L, ANTI)
    Ug = lat.gauge_from_numpy(gen.links(L, "haar", 45))
    A = lmx.WilsonDiracOperator4D_Donly(Ug) if donly else lmx.WilsonDiracOperator4D(Ug, 0.117)
    psi = lat.spinor(nrhs)
    lmx.randomize_gaussian_matrix_(psi, [lmx.RNGStreamKey(46 + r) for r in range(nrhs)])
    one, y, z = lat.spinor(), lat.spinor(nrhs), lat.spinor()
    p32 = psi.data.to(torch.float32)
    y32, z32 = lmx.spinor_f32(lat, nrhs), lmx.spinor_f32(lat, 1)
    lmx.mul_(y, A, psi)
    lmx.mul_f32_(y32, A, p32)
    for r in range(nrhs):
        one.data.copy_(psi.data[r:r + 1])
        lmx.mul_(z, A, one)
        assert torch.equal(y.data[r], z.data[0])
        lmx.mul_f32_(z32, A, p32[r:r + 1].contiguous())
        assert torch.equal(y32[r], z32[0])


@pytest.mark.parametrize("L,csw,donly,nrhs", [
    ((16, 16, 16, 16), 1.0, False, 13),   # whole rows of a z-plane; a second launch of one field
    ((24, 24, 24, 13), 1.0, False, 3),    # blocks that cut rows; one slice a workgroup
    ((24, 24, 24, 20), 0.0, False, 4),    # four slices a workgroup
    ((24, 24, 24, 18), 1.0, False, 12),   # six slices a workgroup
    ((32, 16, 16, 32), 0.0, False, 4),
    ((32, 16, 16, 32), 0.0, True, 4),
])
@pytest.mark.parametrize("dagger", [False, True])
def test_fp32_fields_staged_in_lds(gpu, L, csw, donly, nrhs, dagger):
    # enough FP32 fields on a streaming lattice take the LDS-staged stencil; one alone is the kernel above
    print(f"FP32 LDS L={L} csw={csw} donly={donly} nrhs={nrhs} dagger={dagger}", flush=True)
    lat = lmx.Lattice(L, ANTI)
    Ug = lat.gauge_from_numpy(gen.links(L, "weak", 47, eps=0.15))
    D = lmx.WilsonDiracOperator4D_Donly(Ug) if donly else lmx.WilsonDiracOperator4D(Ug, 0.117, csw)
    A = lmx.adjoint(D) if dagger else D
    psi = lat.spinor(nrhs)
    lmx.randomize_gaussian_matrix_(psi, [lmx.RNGStreamKey(48 + r) for r in range(nrhs)])
    p32 = psi.data.to(torch.float32)
    y, z = lmx.spinor_f32(lat, nrhs), lmx.spinor_f32(lat, 1)
    lmx.mul_f32_(y, A, p32)
    for r in range(nrhs):
        lmx.mul_f32_(z, A, p32[r:r + 1].contiguous())
        assert torch.equal(y[r], z[0])


@pytest.mark.parametrize("L", [(3, 5, 3, 3), (8, 8, 9, 4), (13, 13, 13, 3)])
@pytest.mark.parametrize("dagger", [False, True])
def test_clover_three_fields(gpu, L, dagger):
    print(f"clover blocks L={L} dagger={dagger}", flush=True)
    U = gen.links(L, "weak", 33, eps=0.15)
    psi = gen.gaussian_spinor(L, 34, nrhs=3)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracCloverOperator4D(lat.gauge_from_numpy(U), 0.1235, 1.0)
    y = lat.spinor(3)
    lmx.mul_(y, lmx.adjoint(D) if dagger else D, lat.spinor_from_numpy(psi))
    F = orc.clover_field_strength(U, L)
    got = y.to_numpy()
    for r in range(3):
        assert np.array_equal(got[r], orc.wilson_clover(U, F, psi[r], L, 0.1235, 1.0, dagger=dagger))


@pytest.mark.parametrize("L", [(2, 2, 2, 2), (3, 5, 3, 3), (8, 8, 9, 4), (13, 13, 13, 3)])
def test_cg(gpu, L):
    print(f"CG blocks L={L}", flush=True)
    U = gen.links(L, "haar", 35)
    b = gen.gaussian_spinor(L, 36)
    xo, ro = orc.cg(orc.NormalOp(orc.OP_DDAGD_WILSON, L, U=U, kappa=0.12), b, rtol=1e-10, order=1)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracOperator4D(lat.gauge_from_numpy(U), 0.12)
    x, r, p, Ap, tmp = (lat.spinor() for _ in range(5))
    res = lmx.cg_(x, lmx.DdagDOp(D, tmp), lat.spinor_from_numpy(b), r, p, Ap, rtol=1e-10)
    assert res.converged and res.iterations == ro.iterations
    assert np.array_equal(x.to_numpy(), xo)
    assert res.residual_norm == ro.residual_norm


@pytest.mark.parametrize("L", [(2, 2, 2, 2), (3, 5, 3, 3), (1, 4, 5, 3), (8, 8, 4, 2)])
def test_clover_link_pullback(gpu, L):
    # blocks of 64 sites, a wavefront per link direction: fewer sites than a
    # block, a cut last block, an extent of one (a neighbour is the site itself)
    print(f"clover pullback L={L}", flush=True)
    U = gen.links(L, "haar", 37)
    psi, w = gen.gaussian_spinor(L, 38), gen.gaussian_spinor(L, 39)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracCloverOperator4D(lat.gauge_from_numpy(U), 0.12, 1.3)
    dU = lmx.GaugeField(lat)
    for _ in range(2):  # the second call adds to the first, and finds its scratch written
        lmx.wilson_pullback_(dU, D, lat.spinor_from_numpy(w), lat.spinor_from_numpy(psi), -0.12)
    ref = orc.clover_pullback(U, w, psi, L, -0.12, 1.3)
    ref = orc.clover_pullback(U, w, psi, L, -0.12, 1.3, dU=ref)
    assert np.array_equal(dU.to_numpy(), ref)


@pytest.mark.parametrize("L", [(2, 2, 2, 2), (3, 5, 3, 3), (1, 4, 5, 3), (8, 8, 9, 4), (13, 13, 13, 3)])
def test_field_strength(gpu, L):
    # a wavefront per plane over the same blocks and slabs as the stencil
    print(f"field strength L={L}", flush=True)
    U = gen.links(L, "haar", 40)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracCloverOperator4D(lat.gauge_from_numpy(U), 0.12, 1.0)
    assert np.array_equal(D.clover_planes(), orc.clover_field_strength(U, L))


@pytest.mark.parametrize("L", [(4, 4, 4, 4), (16, 16, 16, 17)])  # the small-lattice iteration and the general one
@pytest.mark.parametrize("maxiter", [0, 1, 17])  # none, one, and one into the second batch of launches
def test_cg_stops_at_maxiter(gpu, L, maxiter):
    print(f"CG maxiter L={L} maxiter={maxiter}", flush=True)
    U = gen.links(L, "weak", 41)
    b, x0 = gen.gaussian_spinor(L, 42), gen.gaussian_spinor(L, 43)
    xo, ro = orc.cg(orc.NormalOp(orc.OP_DDAGD_WILSON, L, U=U, kappa=0.12), b, x0=x0, rtol=1e-10, maxiter=maxiter,
                    order=1)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracOperator4D(lat.gauge_from_numpy(U), 0.12)
    r, p, Ap, tmp = (lat.spinor() for _ in range(4))
    x = lat.spinor_from_numpy(x0)
    res = lmx.cg_(x, lmx.DdagDOp(D, tmp), lat.spinor_from_numpy(b), r, p, Ap, rtol=1e-10, maxiter=maxiter)
    assert not res.converged and res.reason == ro.reason and res.iterations == ro.iterations == maxiter
    assert np.array_equal(x.to_numpy(), xo)
    assert res.residual_norm == ro.residual_norm


@pytest.mark.parametrize("L", [(4, 4, 4, 4), (16, 16, 16, 17)])
def test_cg_first_iteration_converges(gpu, L):
    # zero links: D = 1, so the solve ends in the iteration whose x update is still to come
    print(f"CG one iteration L={L}", flush=True)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracOperator4D(lmx.GaugeField(lat), 0.12)
    b = lat.spinor_from_numpy(gen.gaussian_spinor(L, 44))
    x, r, p, Ap, tmp = (lat.spinor() for _ in range(5))
    res = lmx.cg_(x, lmx.DdagDOp(D, tmp), b, r, p, Ap, rtol=1e-10)
    assert res.converged and res.iterations == 1 and res.residual_norm == 0.0
    assert np.array_equal(x.to_numpy(), b.to_numpy())


def _padded(L, nw, nrhs, rng):
    P = [d + 2 * nw for d in L]
    shape = (nrhs, P[3], P[2], P[1], P[0], 4, 3)
    a = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)  # the halo: garbage
    core = (slice(None),) + tuple(slice(nw, nw + d) for d in reversed(L)) + (slice(None), slice(None))
    return a, core


@pytest.mark.parametrize("L,nw,phases", [((2, 2, 2, 2), 1, ANTI), ((3, 5, 3, 3), 0, ANTI), ((3, 5, 3, 3), 2, (-1, 1j, 1, -1)),
                                         ((8, 8, 9, 4), 1, ANTI), ((13, 13, 13, 2), 1, ANTI)])
@pytest.mark.parametrize("csw", [0.0, 1.0])
@pytest.mark.parametrize("dt", [torch.complex128, torch.complex64])
@pytest.mark.parametrize("offset", [0, 1])  # in elements: at 1 a complex64 array is not 16-byte aligned
def test_reference_storage(gpu, L, nw, phases, csw, dt, offset):
    print(f"padded blocks L={L} nw={nw} csw={csw} {dt} offset={offset}", flush=True)
    U = gen.links(L, "haar", 49)
    a, core = _padded(L, nw, 2, np.random.default_rng(50))
    lat = lmx.Lattice(L, phases)
    D = lmx.WilsonDiracOperator4D(lat.gauge_from_numpy(U), 0.117, csw)
    store = torch.empty(a.size + offset, dtype=dt, device="cuda")
    psi = store[offset:].view(a.shape).copy_(torch.from_numpy(a))
    C = torch.full((a.size + offset,), 3.0, dtype=dt, device="cuda")[offset:].view(a.shape)
    lmx.mul_padded_(C, lmx.adjoint(D), psi, nw=nw)
    got = C.cpu().numpy()
    outside = np.ones(a.shape, dtype=bool)
    outside[core] = False
    assert np.all(got[outside] == 3.0)  # only core sites are written
    F = orc.clover_field_strength(U, L) if csw else None
    for r in range(2):
        p = np.ascontiguousarray(a[core][r]).reshape(-1, 4, 3)
        ref = (orc.wilson_clover(U, F, p, L, 0.117, csw, phases, dagger=True) if csw
               else orc.wilson(U, p, L, 0.117, phases, dagger=True))
        mine = got[core][r].reshape(-1, 4, 3)
        if dt == torch.complex128:
            assert np.array_equal(mine, ref)
        else:  # a few dozen roundings of 6e-8 on values of order one
            assert np.max(np.abs(mine - ref)) <= 64 * 6e-8 * np.max(np.abs(ref))
