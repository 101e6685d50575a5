"""How many iterations and updates the mixed solver launches for those that run:
groups of four with one gated update where updates are rare, the update after
each iteration where they are dense.  The host's polls and graphs do not change
what runs, nor a bit of the solution."""
import numpy as np
import pytest

import lmx
from kernel_names import count, launched
from lmx import generators as gen

pytestmark = pytest.mark.gpu

L = (4, 4, 4, 8)


def _solve(kappa, delta, precision="h16", **kw):
    lat = lmx.Lattice(L, (1, 1, 1, -1))
    D = lmx.WilsonDiracOperator4D(lat.gauge_from_numpy(gen.links(L, "weak", 91, eps=0.2)), kappa)
    b, x = lat.spinor_from_numpy(gen.gaussian_spinor(L, 92, nrhs=2)), lat.spinor(2)
    res = []
    names = launched(lambda: res.extend(lmx.cg_batched_(x, D, b, precision=precision, reliable_delta=delta, **kw)))
    assert all(r.converged for r in res)
    # the two right-hand sides stop apart; what runs is the longer one's iterations
    return x.to_numpy(), res, max(r.iterations for r in res), count(names, "k_mx_fin<1>"), count(names, "k_mx_fin<3>") - 1


@pytest.mark.parametrize("kappa,delta", [(0.05, 0.5), (0.05, 0.3), (0.12, 0.9)])
def test_dense_updates_do_not_idle(gpu, kappa, delta):
    print(f"dense updates kappa={kappa} delta={delta}", flush=True)
    for every in (1, 3, 10):
        _, res, ran, iterations, _ = _solve(kappa, delta, check_every=every)
        assert ran <= 3 * max(r.reliable_updates for r in res)  # dense indeed
        assert iterations <= ran + every  # the last batch may run past the end


def test_sparse_updates_are_gated_by_group(gpu):
    print("sparse updates", flush=True)
    for every in (1, 10):
        _, res, ran, iterations, updates = _solve(0.1235, 0.1, check_every=every)
        asked = max(r.reliable_updates for r in res)
        assert ran >= 6 * asked
        assert updates <= iterations // 4 + asked + 1
        assert iterations <= ran + every + 3 * asked


@pytest.mark.parametrize("precision", ["f32", "f16", "h16"])
@pytest.mark.parametrize("kappa,delta", [(0.05, 0.5), (0.12, 0.3), (0.12, 0.9), (0.1235, 0.1)])
def test_same_bits_by_any_batching(gpu, precision, kappa, delta):
    print(f"batching {precision} kappa={kappa} delta={delta}", flush=True)
    first = None
    for kw in (dict(check_every=1), dict(check_every=3), dict(check_every=10), dict(use_graph=True),
               dict(use_graph=True, check_every=40)):
        x, res, *_ = _solve(kappa, delta, precision, **kw)
        got = [(r.iterations, r.reliable_updates) for r in res]
        if first is None:
            first = (x, got)
        assert got == first[1] and np.array_equal(x, first[0])
