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
