"""Overflow in the clover link pullback: wherever the oracle's cotangent is not
finite, the device's is not."""
import numpy as np
import pytest

import oracle as orc
import lmx
from lmx import generators as gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spin", range(4))
@pytest.mark.parametrize("value", [1e200, 1e200j, np.inf])
def test_overflowing_cotangent(gpu, spin, value):
    # one spin of one site: in some planes the product's real part alone overflows, which leaves the anti-Hermitian
    # part's diagonal without a value (inf - inf)
    L = (6, 6, 6, 6)
    print(f"non-finite clover cotangent spin={spin} value={value}", flush=True)
    U = gen.links(L, "haar", 81)
    psi, w = gen.gaussian_spinor(L, 82), gen.gaussian_spinor(L, 83)
    site = 2 + 6 * (3 + 6 * (2 + 6 * 3))
    psi[site] = 0.0
    w[site] = 0.0
    psi[site, spin, 1] = value
    w[site, spin // 2 * 2, 1] = 1e200  # gamma_mu gamma_nu keeps the two halves apart
    lat = lmx.Lattice(L, (1, 1, 1, -1))
    D = lmx.WilsonDiracCloverOperator4D(lat.gauge_from_numpy(U), 0.12, 1.3)
    dU = lmx.GaugeField(lat)
    lmx.wilson_pullback_(dU, D, lat.spinor_from_numpy(w), lat.spinor_from_numpy(psi), -0.12)
    with np.errstate(all="ignore"):
        ref = orc.clover_pullback(U, w, psi, L, -0.12, 1.3)
    got = dU.to_numpy()
    bad = ~np.isfinite(ref)
    assert bad.any() and not bad.all()
    assert np.array_equal(np.isfinite(got), ~bad)
    assert np.array_equal(got[~bad], ref[~bad])
