"""Baskets of every width against torch: price and gradients of the same paths by reverse-mode autodiff in
float64, with step counts around the 1 to 8 steps that fill whole ChaCha blocks and path counts
around a wave and a block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("assets", range(1, 9))
@pytest.mark.parametrize("paths,steps", [(1, 1), (65, 7), (257, 17)])
def test_basket_width_matches_autodiff(oracle, assets, paths, steps):
    from sde_sim_rs.adjoint import Basket, basket_config
    A, S, N, seed = assets, paths, steps, 41
    c = basket_config(seed, assets=A)
    print("case: basket of %d assets, %d paths x %d steps" % (A, S, N), flush=True)
    u = np.stack([oracle.pseudo_f64(seed + s, N * A) for s in range(S)])
    eps = torch.tensor(np.vectorize(oracle.inv_normal)(u)).reshape(S, N, A)
    x0, mu, sg = (torch.tensor(c[k], requires_grad=True) for k in ("x0", "mu", "sigma"))
    L = torch.tensor(np.linalg.cholesky(c["rho"]), requires_grad=True)
    dt = 1.0 / N
    X = x0.expand(S, A)
    for n in range(N):
        X = X + X * (mu * dt + sg * np.sqrt(dt) * (eps[:, n] @ L.T))
    y = (X.mean(1) - 100.0) / 0.5
    pay = 0.5 * torch.logaddexp(y, torch.zeros_like(y))  # torch's softplus is linear above 20
    pay.mean().backward()
    price = float(pay.detach().mean())
    b = Basket(A, N, S, seed=seed, precision="f64", storage="tape")
    r = b.evaluate(c["x0"], c["mu"], c["sigma"], c["rho"])
    p = b.evaluate(c["x0"], c["mu"], c["sigma"], c["rho"], adjoint=False)
    assert p["price"] == r["price"] and p["variance"] == r["variance"]
    assert abs(r["price"] - price) <= 1e-12 * abs(price)
    for name, g in (("x0", x0.grad), ("mu", mu.grad), ("sigma", sg.grad), ("chol", torch.tril(L.grad))):
        scale = float(g.abs().max())
        np.testing.assert_allclose(r[name], g.numpy(), rtol=1e-9, atol=1e-9 * scale + 1e-300, err_msg=name)
    f = Basket(A, N, S, seed=seed, precision="f32", storage="tape").evaluate(c["x0"], c["mu"], c["sigma"], c["rho"])
    assert abs(f["price"] - price) <= 1e-4 * abs(price) + 1e-4
