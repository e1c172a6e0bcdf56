"""f64 plans of few paths, which several waves step together (sde_team_kernel): against the oracle at the
edges of 64 paths, of a unit of steps and of the buffer's rounds, and which plans take that kernel.

Tolerance: a step's rounding error is a few ulp (2.2e-16) of the path's scale, and 130 of them stay below
130 * 16 * 2.2e-16 = 4.6e-13 where differences do not grow; 1e-11 leaves room for the growth of the
schemes used here (at most e^0.2 per unit time and Heston's square root)."""
import numpy as np
import pytest

from conftest import GBM, HESTON

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

THREE = ["dA = (0.05 * A) * dt + (0.2 * A) * dW1", "dB = (0.1 * t) * dt + (0.1 * A) * dW2 + (0.3) * dW3", "C = max(A - B, 0)"]
JUMPS = ["dX = (2.0 * (0.5 - X)) * dt + (0.1) * dN1(9.0 * X)", "dY = (0.05 * Y) * dt + (0.2 * Y) * dW1 + (0.5) * dN1(9.0 * X)"]
FOUR = ["dX%d = (0.05 * X%d) * dt + (0.%d * X%d) * dW%d" % (i, i, i, i, i) for i in (1, 2, 3, 4)]
MODELS = {
    "gbm": (GBM, {"X": 100.0}, 4, 8),
    "heston": (HESTON, {"S": 100.0, "v": 0.04}, 4, 4),
    "three": (THREE, {"A": 1.0, "B": 0.5, "C": 0.5}, 3, 8),
    "jumps": (JUMPS, {"X": 0.5, "Y": 100.0}, 4, 4),
    "four": (FOUR, {"X1": 1.0, "X2": 2.0, "X3": 3.0, "X4": 4.0}, 4, 2),
}


@pytest.mark.parametrize("rng,scramble", [("pseudo", "shift"), ("sobol", "shift"), ("sobol", "xor")])
@pytest.mark.parametrize("model,scheme", [("gbm", "euler"), ("gbm", "runge-kutta"), ("heston", "runge-kutta"),
                                          ("three", "euler"), ("three", "runge-kutta"), ("jumps", "euler"),
                                          ("four", "euler")])
def test_team_matches_the_oracle(oracle, model, scheme, rng, scramble):
    import sde_sim_rs
    eqs, init, team, unit = MODELS[model]
    full = (team - 1) * unit  # steps of a round
    for S, N, uniform in ((1, full, True), (63, full + 1, False), (64, 2 * full, True), (65, 2 * full - 1, False),
                          (130, 5 * full + unit - 1, True)):
        print("case: team %s %s %s %s S=%d N=%d" % (model, scheme, rng, scramble, S, N), flush=True)
        times = np.arange(N + 1) * 2.0 ** -7 if uniform else np.linspace(0.0, 1.0, N + 1) ** 1.1
        kw = dict(seed=3, scramble=scramble, scramble_seed=4)
        plan = sde_sim_rs.Plan(eqs, times, S, init, rng, scheme, outputs=("filtration", "terminal"), **kw)
        assert "sde_team_kernel<SdeModel" in plan.source
        f = plan.new_filtration()
        plan.run(f)
        torch.cuda.synchronize()
        ref = np.asarray(oracle.simulate(eqs, times, S, init, scheme=scheme, rng=rng, **kw))
        got = f.cpu().numpy().transpose(2, 0, 1)
        np.testing.assert_allclose(got, ref, rtol=1e-11, atol=1e-11)
        for p, (name, (mean, var)) in enumerate(plan.moments().items()):
            end = ref[:, -1, p]
            np.testing.assert_allclose(mean, end.mean(), rtol=1e-11, atol=1e-11)
            np.testing.assert_allclose(var, end.var(ddof=1) if S > 1 else 0.0, rtol=1e-9, atol=1e-9)


@pytest.mark.parametrize("paths,steps,kw,team", [
    (98304, 24, {}, True), (98305, 24, {}, False), (1000, 23, {}, False), (1000, 24, dict(precision="f32"), False),
    (1000, 24, dict(block_size=256), False), (1000, 24, dict(paths_per_lane=1), False)])
def test_which_plans_are_team_plans(paths, steps, kw, team):
    import sde_sim_rs
    plan = sde_sim_rs.Plan(GBM, np.linspace(0.0, 1.0, steps + 1), paths, {"X": 100.0}, "pseudo", "euler", seed=1, **kw)
    assert ("sde_team_kernel<SdeModel" in plan.source) == team
