"""FP32 basket gradients of every width against the sums of the same paths in float64, in both kernels.

Tolerance, relative to the sum of the magnitudes of the paths' terms: 12 steps round an asset's growth 3 times each
(6e-8), and a draw is off by at most 4.8e-7, times sigma sqrt(dt) <= 0.12: 12 * (3 * 6e-8 + 0.6e-7) = 3e-6 of X, hence
3e-6 * 150 / 20 = 2.2e-5 of the payoff's slope at a width of 20, and the same again for the product of the
growths and the sums of 1 / g and eps / g: 5e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("assets", range(1, 9))
@pytest.mark.parametrize("many", [False, True])
def test_f32_gradients(oracle, assets, many):
    from sde_sim_rs.adjoint import Basket, basket_config
    few = 2 * 64 * torch.cuda.get_device_properties(0).multi_processor_count
    A, N, seed, width = assets, 12, 29, 20.0
    S = few + 1 if many else 300
    print("case: f32 gradients A=%d S=%d" % (A, S), flush=True)
    c = basket_config(seed, assets=A)
    r = Basket(A, N, S, seed=seed, width=width, precision="f32").evaluate(c["x0"], c["mu"], c["sigma"], c["rho"])
    if many:  # the f64 kernel, which the other tests compare with autodiff
        f = Basket(A, N, S, seed=seed, width=width, precision="f64").evaluate(c["x0"], c["mu"], c["sigma"], c["rho"])
        for k in ("price", "x0", "mu", "sigma", "chol"):
            # Sums of magnitudes: X0 times the slope for mu and X0, and |eps| <= 6 of it for the others.
            scale = {"price": abs(f["price"]), "x0": 1.0, "mu": 150.0, "sigma": 300.0, "chol": 60.0}[k]
            np.testing.assert_allclose(r[k], f[k], rtol=0, atol=5e-5 * scale, err_msg=k)
        return
    u = np.stack([oracle.pseudo_f64(seed + s, N * A) for s in range(S)])
    eps = np.vectorize(oracle.inv_normal)(u).reshape(S, N, A)
    L, dt = np.linalg.cholesky(c["rho"]), 1.0 / N
    z = eps @ L.T
    g = 1.0 + c["mu"] * dt + c["sigma"] * np.sqrt(dt) * z
    X = c["x0"] * g.prod(1)
    y = (X.mean(1) - 100.0) / width
    m = (1.0 / (1.0 + np.exp(-y)))[:, None] / A * X
    terms = {"x0": m / c["x0"], "mu": m * dt * (1.0 / g).sum(1), "sigma": m * np.sqrt(dt) * (z / g).sum(1),
             "chol": np.einsum("si,sni,snk->sik", m * c["sigma"] * np.sqrt(dt), 1.0 / g, eps)}
    size = {"x0": m / c["x0"], "mu": m * dt * (1.0 / g).sum(1), "sigma": m * np.sqrt(dt) * np.abs(z / g).sum(1),
            "chol": np.einsum("si,sni,snk->sik", m * c["sigma"] * np.sqrt(dt), 1.0 / g, np.abs(eps))}
    price = (width * np.logaddexp(y, 0.0)).mean()
    assert abs(r["price"] - price) <= 5e-5 * price
    for k, t in terms.items():
        want, bound = t.mean(0), 5e-5 * size[k].mean(0)
        if k == "chol":
            want, bound = np.tril(want), np.tril(bound)
        assert np.all(np.abs(r[k] - want) <= bound), (k, r[k], want)
