"""Several FP64 fields on the streaming kernel, two to a work item (Wilson, an
odd count leaves the last one alone) or one (clover), against the oracle bit
for bit.  The shape is forced, as these lattices are too small to be given it."""
import numpy as np
import pytest

import oracle as orc
import lmx
from kernel_names import count, launched
from lmx import generators as gen

pytestmark = pytest.mark.gpu

ANTI = (1, 1, 1, -1)
KAPPA = 0.117


def _lattice(monkeypatch, L, TL, phases=ANTI):
    monkeypatch.setenv("LMX_STREAM_TL", str(TL))
    monkeypatch.setenv("LMX_STREAM_ZS", "1")
    return lmx.Lattice(L, phases)


@pytest.mark.parametrize("L,TL,phases", [((8, 8, 4, 16), 4, ANTI), ((8, 8, 8, 6), 3, (-1, 1, -1, -1)),
                                         ((16, 16, 8, 4), 4, ANTI)])
@pytest.mark.parametrize("nrhs", [2, 3, 4])
@pytest.mark.parametrize("flags", [0, 1, 2, 3])
def test_wilson(gpu, monkeypatch, L, TL, phases, nrhs, flags):
    print(f"streamed fields L={L} TL={TL} nrhs={nrhs} flags={flags}", flush=True)
    lat = _lattice(monkeypatch, L, TL, phases)
    U = gen.links(L, "haar", 71)
    psi = gen.gaussian_spinor(L, 72, nrhs=nrhs)
    Ug = lat.gauge_from_numpy(U)
    A = lmx.WilsonDiracOperator4D_Donly(Ug) if flags & 2 else lmx.WilsonDiracOperator4D(Ug, KAPPA)
    A = lmx.adjoint(A) if flags & 1 else A
    x, y = lat.spinor_from_numpy(psi), lat.spinor(nrhs)
    lmx.mul_(y, A, x)
    got = y.to_numpy()
    for r in range(nrhs):
        ref = orc.wilson(U, psi[r], L, KAPPA, phases, dagger=bool(flags & 1), donly=bool(flags & 2))
        assert np.array_equal(got[r], ref), r


@pytest.mark.parametrize("nrhs", [2, 3, 4])
@pytest.mark.parametrize("dagger", [False, True])
def test_clover(gpu, monkeypatch, nrhs, dagger):
    L = (8, 8, 4, 16)
    print(f"streamed clover fields nrhs={nrhs} dagger={dagger}", flush=True)
    lat = _lattice(monkeypatch, L, 4)
    U = gen.links(L, "weak", 73, eps=0.3)
    psi = gen.gaussian_spinor(L, 74, nrhs=nrhs)
    D = lmx.WilsonDiracCloverOperator4D(lat.gauge_from_numpy(U), KAPPA, 1.2)
    x, y = lat.spinor_from_numpy(psi), lat.spinor(nrhs)
    lmx.mul_(y, lmx.adjoint(D) if dagger else D, x)
    F = orc.clover_field_strength(U, L)
    got = y.to_numpy()
    for r in range(nrhs):
        assert np.array_equal(got[r], orc.wilson_clover(U, F, psi[r], L, KAPPA, 1.2, dagger=dagger)), r


@pytest.mark.parametrize("csw,nrhs", [(0.0, 1), (0.0, 2), (0.0, 3), (1.0, 3)])
def test_takes_the_streaming_kernel(gpu, monkeypatch, csw, nrhs):
    print(f"streamed fields route csw={csw} nrhs={nrhs}", flush=True)
    lat = _lattice(monkeypatch, (8, 8, 4, 16), 4)
    D = lmx.WilsonDiracOperator4D(lmx.GaugeField(lat), KAPPA, csw)
    x, y = lat.spinor(nrhs), lat.spinor(nrhs)
    names = launched(lambda: lmx.mul_(y, D, x))
    assert count(names, "k_stream<") == 1 and count(names, "k_hops") == 0
