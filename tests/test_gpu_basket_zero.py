"""Baskets in which an asset's growth factor over a step is exactly 0: price and gradients stay finite and
are those of the path product, whichever step it falls on and however many do.

With mu dt = -1 and sigma sqrt(dt) a few units in the last place of 1, the growth g = 1 + (-1 + sigma
sqrt(dt) eps) is a small multiple of such a unit, 0 for a third of the draws. sigma sqrt(dt) is a power of
two, so the rounded sum is known from eps: the reference forms g in the kernel's precision and everything
else in f64. Tolerance: each path's terms are products of 4 factors, summed in f64, against the sum of their
magnitudes: 16 roundings are 2e-6 in f32 (2e-5 leaves room for its normals, 5e-7 each in the other assets) and 2e-15
in f64 (1e-11 is what the other tests of the gradients allow)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _few():
    return 2 * 64 * torch.cuda.get_device_properties(0).multi_processor_count


def _normals(oracle, S, N, A, seed):
    u = np.stack([oracle.pseudo_f64(seed + s, N * A) for s in range(S)])
    return np.vectorize(oracle.inv_normal)(u).reshape(S, N, A)


def _reference(eps, x0, mu, sg, L, w, K, width, real):
    """Price and (gradients, sums of magnitudes) for dt = 1 with growth factors in `real`."""
    S, N, A = eps.shape
    scl = np.tril(sg[:, None] * L)
    c = mu + eps @ scl.T
    g = (1.0 + c.astype(real)).astype(np.float64)
    X = x0 * np.prod(g, axis=1)
    y = (X @ w - K) / width
    pay = width * np.logaddexp(y, 0.0)
    m = (1.0 / (1.0 + np.exp(-y)))[:, None] * w * x0  # times the product of the growths but one: d/dg
    others = np.stack([np.prod(np.delete(g, n, axis=1), axis=1) for n in range(N)], axis=1)
    dg = m[:, None, :] * others  # [S][N][A]
    z = eps @ np.tril(L).T
    terms = {"x0": m * np.prod(g, axis=1) / x0, "mu": dg.sum(1), "sigma": (dg * z).sum(1),
             "chol": np.einsum("sni,snk->sik", dg * sg, eps)}
    size = {"x0": np.abs(terms["x0"]), "mu": np.abs(dg).sum(1), "sigma": np.abs(dg * z).sum(1),
            "chol": np.einsum("sni,snk->sik", np.abs(dg * sg), np.abs(eps))}
    return pay.mean(), {k: (v.mean(0), size[k].mean(0)) for k, v in terms.items()}, g


@pytest.mark.parametrize("precision,real,unit,tol", [("f32", np.float32, 2.0 ** -23, 2e-5), ("f64", np.float64, 2.0 ** -52, 1e-11)])
@pytest.mark.parametrize("A,N", [(1, 1), (1, 3), (3, 2), (5, 3), (8, 4)])
@pytest.mark.parametrize("many", [False, True])
def test_zero_growth(oracle, precision, real, unit, tol, A, N, many):
    from sde_sim_rs.adjoint import Basket
    seed, S = 11, _few() + 1 if many else 130
    print("case: zero growth %s A=%d N=%d S=%d" % (precision, A, N, S), flush=True)
    eps = _normals(oracle, S, N, A, seed)
    x0, w = np.full(A, 64.0), np.full(A, 1.0 / A)
    mu, sg = np.full(A, 0.05), np.full(A, 0.25)
    mu[0], sg[0] = -1.0, unit
    rho = np.full((A, A), 0.25) + 0.75 * np.eye(A)
    L = np.linalg.cholesky(rho)
    K = 0.0 if A == 1 else 40.0
    price, grads, g = _reference(eps, x0, mu, sg, L, w, K, 4.0, real)
    zeros = (g[:, :, 0] == 0.0).sum(1)
    assert (zeros > 0).any() and (zeros == 0).any() and (N == 1 or (zeros > 1).any())
    b = Basket(A, N, S, horizon=float(N), strike=K, width=4.0, seed=seed, precision=precision)
    r = b.evaluate(x0, mu, sg, rho, w)
    assert abs(r["price"] - price) <= tol * price
    assert b.evaluate(x0, mu, sg, rho, w, adjoint=False)["price"] == r["price"]
    for name, (want, size) in grads.items():
        if name == "chol":
            want, size = np.tril(want), np.tril(size)
        assert np.all(np.abs(r[name] - want) <= tol * size), (name, r[name], want)


@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("many", [False, True])
def test_certain_zero(precision, many):
    """sigma = 0 and mu dt = -1: every path's asset ends at 0 after one step, with d/dX0 = 0 and d/dmu =
    weight X0 dt times the payoff's slope, 1 here to f32's last place."""
    from sde_sim_rs.adjoint import Basket
    S = _few() + 1 if many else 65
    print("case: certain zero growth %s S=%d" % (precision, S), flush=True)
    r = Basket(2, 1, S, strike=1.0, width=0.5, seed=3, precision=precision).evaluate(
        [80.0, 100.0], [-1.0, 0.0], [0.0, 0.01], np.eye(2), [0.5, 0.5])
    assert r["x0"][0] == 0.0
    assert abs(r["mu"][0] - 40.0) <= 40.0 * 2.0 ** -23
    assert all(np.all(np.isfinite(r[k])) for k in ("x0", "mu", "sigma", "chol", "rho"))
