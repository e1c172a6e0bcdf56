"""Baskets on both sides of the path count up to which four waves share 64 paths: the larger run's estimates are
the weighted mean of the smaller run's and those of the one path more, which the few-paths kernel also
gives by itself.

Tolerance: the same operations per path and f64 sums; in f64 a rounding apart (1e-11 of the largest of a
kind is 1e5 of them), in f32 the paths may differ by a few 6e-8 per step where products are fused
differently: 9 steps, 1e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("assets", range(1, 9))
@pytest.mark.parametrize("precision,tol", [("f64", 1e-11), ("f32", 1e-5)])
@pytest.mark.parametrize("adjoint", [True, False])
def test_both_kernels_agree(assets, precision, tol, adjoint):
    from sde_sim_rs.adjoint import Basket, basket_config
    A, N, seed = assets, 9, 23
    few = 2 * 64 * torch.cuda.get_device_properties(0).multi_processor_count
    c = basket_config(seed, assets=A)
    print("case: basket of %d assets %s, %d and %d paths" % (A, precision, few, few + 1), flush=True)
    r = [Basket(A, N, S, seed=s, precision=precision).evaluate(c["x0"], c["mu"], c["sigma"], c["rho"], adjoint=adjoint)
         for S, s in ((few, seed), (1, seed + few), (few + 1, seed))]
    for name in ("price",) + (("x0", "mu", "sigma", "chol") if adjoint else ()):
        small, one, large = (np.asarray(x[name]) for x in r)
        want = (few * small + one) / (few + 1)
        np.testing.assert_allclose(large, want, rtol=0, atol=tol * float(np.max(np.abs(want))), err_msg=name)
