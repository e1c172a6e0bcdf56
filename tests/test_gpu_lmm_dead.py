"""Forward 0 has fixed before the first step of every run: its sensitivity is that of the numeraire's factor
1 + tau L_0 alone, finite for a forward of 0 as for any other.

Tolerance: one f64 quotient per path on the same path values, so the ratio to the price is exact to rounding,
1e-13 for f64 sums; in f32 L_0 is rounded once (6e-8 of tau L_0) and the price's sum is the same: 1e-7."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("precision,tol", [("f64", 1e-13), ("f32", 1e-7)])
@pytest.mark.parametrize("storage", ["tape", "checkpoints"])
@pytest.mark.parametrize("first", [0.0, -0.0, 1e-12, 0.03, -0.01])
def test_fixed_forward(precision, tol, storage, first):
    from sde_sim_rs.lmm import ForwardRateModel, forward_rate_config
    c, tau = forward_rate_config(seed=5), 0.25
    print("case: fixed forward %s %s %g" % (precision, storage, first), flush=True)
    L0 = c["L0"].copy()
    L0[0] = first
    r = ForwardRateModel(steps=9, paths=321, expiry_index=3, strike=0.05, precision=precision,
                         storage=storage).evaluate(L0, c["vol"], c["loadings"])
    assert r["price"] > 0.0 and np.all(np.isfinite(r["dL0"]))
    want = -r["price"] * tau / (1.0 + tau * first)
    assert abs(r["dL0"][0] - want) <= tol * abs(want)


@pytest.mark.parametrize("precision,tol", [("f64", 1e-10), ("f32", 1e-4)])
@pytest.mark.parametrize("storage", ["tape", "checkpoints"])
def test_forwards_of_zero(oracle, precision, tol, storage):
    """Alive forwards of 0 stay there and have the sensitivities that autodiff of the same paths gives (tolerances of
    test_gpu_lmm_steps.py)."""
    from sde_sim_rs.lmm import ForwardRateModel, forward_rate_config
    from test_gpu_lmm import _sobol_normals
    from test_gpu_lmm_steps import _reference
    c, e, spp, S, K = forward_rate_config(seed=5), 3, 3, 130, 0.05
    c["L0"] = c["L0"].copy()
    c["L0"][[0, 1, 4, 20, 39]] = 0.0
    print("case: forwards of 0 %s %s" % (precision, storage), flush=True)
    price, grad = _reference(c, torch.tensor(_sobol_normals(oracle, S, e * spp, 5)), e, spp, K)
    r = ForwardRateModel(steps=e * spp, paths=S, expiry_index=e, strike=K, scramble_seed=5, precision=precision,
                         storage=storage).evaluate(c["L0"], c["vol"], c["loadings"])
    assert abs(r["price"] - price) <= tol * price
    np.testing.assert_allclose(r["dL0"], grad, rtol=0, atol=tol * np.max(np.abs(grad)))


def test_f32_price_has_no_drift(oracle):
    """The f32 price against f64 on the same points: nothing that rounds at every step is common to the paths, so what is
    left is an exponential's mean error (2.4e-9) once per forward and the rounded parameters (3e-8 of each of 36
    forwards' volatilities and levels, to which a price at the money has an elasticity of about 5, averaging
    over the forwards): 1e-7. The same steps as products of exponentials were 2.1e-7 off over 40 and 6.1e-7 over 160."""
    from sde_sim_rs.lmm import ForwardRateModel, forward_rate_config
    c = forward_rate_config(seed=5)
    for steps in (40, 160):
        print("case: f32 price drift %d steps" % steps, flush=True)
        p = [ForwardRateModel(steps=steps, paths=1 << 16, precision=x).evaluate(c["L0"], c["vol"], c["loadings"], adjoint=False)
             ["price"] for x in ("f32", "f64")]
        assert abs(p[0] - p[1]) <= 1e-7 * p[1]
