"""Fields that share a fill launch, and large uniform ones that do not: the
launches, and each field the same as by itself."""
import pytest
import torch

import lmx
from kernel_names import count, launched

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,n,uniform,gauss", [((16, 16, 16, 16), 3, 1, 1), ((20, 20, 20, 124), 2, 1, 1),
                                                  ((20, 20, 20, 125), 2, 2, 1)])  # 992000 and 1000000 sites
def test_launches(gpu, dims, n, uniform, gauss):
    print(f"fill launches {dims} x {n}", flush=True)
    lat = lmx.Lattice(dims)
    keys = [lmx.RNGStreamKey(5 + r, r) for r in range(n)]
    psi, one = lat.spinor(n), lat.spinor(1)
    for f, want in ((lmx.randomize_matrix_, uniform), (lmx.randomize_gaussian_matrix_, gauss)):
        assert count(launched(lambda: f(psi, keys)), "k_rng_fill_spinor") == want
        for r in range(n):
            f(one, keys[r])
            assert torch.equal(psi.data[r], one.data[0]), r
