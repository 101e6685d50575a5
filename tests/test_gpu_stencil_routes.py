"""Which stencil a FP64 apply takes: the streaming kernel on the lattices where
the eight-wavefront one is measured to be slower, that one elsewhere."""
import pytest

import lmx
from kernel_names import count, launched

pytestmark = pytest.mark.gpu

ANTI = (1, 1, 1, -1)


@pytest.mark.parametrize("L,csw,nrhs,stream", [
    ((16, 16, 16, 32), 0.0, 1, False),
    ((32, 32, 32, 16), 0.0, 1, True),    # one full round of workgroups
    ((32, 32, 32, 12), 0.0, 1, False),
    ((32, 32, 32, 12), 0.0, 2, True),    # two to six fields on large slices, a shallow walk
    ((32, 32, 32, 12), 0.0, 4, True),
    ((32, 32, 32, 12), 0.0, 6, False),
    ((24, 24, 24, 32), 0.0, 2, True),
    ((24, 24, 24, 24), 0.0, 2, False),   # the last round of workgroups too empty
    ((16, 16, 16, 96), 0.0, 2, False),   # small slices
    ((32, 32, 32, 4), 1.0, 2, True),
    ((32, 32, 32, 4), 1.0, 1, False),
    ((64, 64, 64, 4), 0.0, 1, True),     # the largest slices
    ((64, 64, 64, 4), 1.0, 1, True),
    ((128, 64, 32, 4), 0.0, 1, False),
])
def test_route(gpu, L, csw, nrhs, stream):
    print(f"route L={L} csw={csw} nrhs={nrhs}", flush=True)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracOperator4D(lmx.GaugeField(lat), 0.12, csw)  # zero links do
    x, y = lat.spinor(nrhs), lat.spinor(nrhs)
    names = launched(lambda: lmx.mul_(y, D, x))
    assert count(names, "k_stream") == (1 if stream else 0)
    assert count(names, "k_hops") == (0 if stream else 1)


@pytest.mark.parametrize("csw", [0.0, 1.0])
def test_forced_shape_in_the_solver(gpu, monkeypatch, csw):
    # D^dagger with the fused p.Ap follows a forced streaming shape on small lattices too
    print(f"forced shape CG csw={csw}", flush=True)
    monkeypatch.setenv("LMX_STREAM_TL", "4")
    monkeypatch.setenv("LMX_STREAM_ZS", "2")
    lat = lmx.Lattice((16, 8, 4, 8), ANTI)
    D = lmx.WilsonDiracOperator4D(lmx.GaugeField(lat), 0.12, csw)
    b = lat.spinor()
    b.data.fill_(1.0)
    x, r, p, Ap, tmp = (lat.spinor() for _ in range(5))
    names = launched(lambda: lmx.cg_(x, lmx.DdagDOp(D, tmp), b, r, p, Ap, rtol=0.0, maxiter=8, check_every=8))
    assert count(names, "k_hops") == 0 and count(names, "k_cg_small") == 0
    assert count(names, "k_stream") >= 16
