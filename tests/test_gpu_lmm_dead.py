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
