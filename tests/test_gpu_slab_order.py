"""The order of 64-site blocks (slab_order) over the kernels that take it: the
stencil in both precisions and both storages, the field strength and the two
link pullbacks.  A block that no workgroup takes, or that two take, leaves a
wrong result; the pullbacks add to their output, so a block taken twice shows
there too."""
import numpy as np
import pytest
import torch

import oracle as orc
import lmx
from lmx import generators as gen

pytestmark = pytest.mark.gpu

ANTI = (1, 1, 1, -1)
SHAPES = [
    (8, 8, 8, 2), (8, 8, 9, 4), (13, 13, 13, 2),  # 8, 9 and 35 blocks a slice: lattice order, the last with a cut block
    (15, 16, 16, 2),   # 60 blocks: the largest slice in lattice order by a little
    (16, 16, 16, 2),   # 64 blocks: slabs of eight
    (16, 16, 17, 3),   # 68: slabs of nine and a tail slab of five
    (17, 17, 17, 2),   # 77, the last one cut: slabs of ten and a tail of seven
    (64, 64, 33, 1),   # 2112: slabs of 256 blocks, the most in FP64, and a tail of 64
]


@pytest.mark.parametrize("L", SHAPES)
def test_clover_link_pullback(gpu, L):
    print(f"slab order pullback L={L}", flush=True)
    U = gen.links(L, "weak", 61)
    psi, w = gen.gaussian_spinor(L, 62), gen.gaussian_spinor(L, 63)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracCloverOperator4D(lat.gauge_from_numpy(U), 0.12, 1.3)
    dU = lmx.GaugeField(lat)
    lmx.wilson_pullback_(dU, D, lat.spinor_from_numpy(w), lat.spinor_from_numpy(psi), -0.12)
    assert np.array_equal(dU.to_numpy(), orc.clover_pullback(U, w, psi, L, -0.12, 1.3))


@pytest.mark.parametrize("L", SHAPES)
def test_stencil_and_field_strength(gpu, L):
    print(f"slab order stencil L={L}", flush=True)
    U = gen.links(L, "weak", 64)
    psi = gen.gaussian_spinor(L, 65)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracCloverOperator4D(lat.gauge_from_numpy(U), 0.12, 1.0)
    F = orc.clover_field_strength(U, L)
    assert np.array_equal(D.clover_planes(), F)
    ref = orc.wilson_clover(U, F, psi, L, 0.12, 1.0)
    x, y = lat.spinor_from_numpy(psi), lat.spinor()
    lmx.mul_(y, D, x)
    assert np.array_equal(y.to_numpy(), ref)
    P = lmx.lattice_matrix(lat, torch.from_numpy(psi.reshape(tuple(reversed(L)) + (4, 3)).copy()).cuda(), nw=1)
    C = torch.zeros_like(P)
    lmx.mul_padded_(C, D, P, nw=1)
    assert np.array_equal(lmx.gather_matrix(lat, C, nw=1).cpu().numpy().reshape(-1, 4, 3), ref)


@pytest.mark.parametrize("L", SHAPES + [(64, 64, 65, 1)])  # 4160 blocks: slabs of 512, the most in FP32
def test_fp32_storages_agree(gpu, L):
    # one FP32 field: the library layout and the padded one by the same arithmetic
    print(f"slab order FP32 L={L}", flush=True)
    lat = lmx.Lattice(L, ANTI)
    D = lmx.WilsonDiracOperator4D(lat.gauge_from_numpy(gen.links(L, "weak", 66)), 0.12)
    psi = gen.gaussian_spinor(L, 67).astype(np.complex64)
    y = lmx.spinor_f32(lat, 1)
    lmx.mul_f32_(y, D, lmx.spinor_f32_from_numpy(lat, psi))
    P = lmx.lattice_matrix(lat, torch.from_numpy(psi.reshape(tuple(reversed(L)) + (4, 3)).copy()).cuda(), nw=1)
    C = torch.zeros_like(P)
    lmx.mul_padded_(C, D, P, nw=1)
    got = lmx.gather_matrix(lat, C, nw=1).cpu().numpy().reshape(-1, 4, 3)
    assert np.array_equal(got, lmx.spinor_f32_to_numpy(y)[0])
    full = lat.spinor_from_numpy(psi.astype(np.complex128))
    z = lat.spinor()
    lmx.mul_(z, D, full)  # a few dozen roundings of 6e-8 on values of order one
    assert np.max(np.abs(got - z.to_numpy())) <= 64 * 6e-8 * np.max(np.abs(got))
