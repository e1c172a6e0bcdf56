"""A path of an f64 plan does not depend on how many paths run with it: plans of few paths (several waves to 64
of them) and plans with a given block size (a path per lane) have the same filtration, bit for bit, so a run that is
split into slices of scenarios gives the rows of the whole."""
import numpy as np
import pytest

from conftest import GBM, HESTON

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

MIXED = ["dA = (0.05 * A - 0.1 * B * A) * dt + (0.2 * A) * dW1 + (0.1 * B) * dW2",
         "dB = (0.3 * t - 0.2 * B) * dt + (0.1 * A + 0.05 * B) * dW2 + (0.3) * dW3", "C = max(A * B - 0.5 * A, 0)"]
JUMPS = ["dX = (2.0 * (0.5 - X)) * dt + (0.1) * dN1(9.0 * X)",
         "dY = (0.05 * Y) * dt + (0.2 * Y) * dW1 + (0.5 * X) * dN1(9.0 * X)"]
MODELS = {"gbm": (GBM, {"X": 100.0}), "heston": (HESTON, {"S": 100.0, "v": 0.04}),
          "mixed": (MIXED, {"A": 1.0, "B": 0.5, "C": 0.5}), "jumps": (JUMPS, {"X": 0.5, "Y": 100.0})}


@pytest.mark.parametrize("rng,scramble", [("pseudo", "shift"), ("sobol", "shift"), ("sobol", "xor")])
@pytest.mark.parametrize("scheme", ["euler", "runge-kutta"])
@pytest.mark.parametrize("model", sorted(MODELS))
@pytest.mark.parametrize("uniform", [True, False])
def test_paths_do_not_depend_on_the_kernel(model, scheme, rng, scramble, uniform):
    import sde_sim_rs
    eqs, init = MODELS[model]
    S, N = 200, 101
    print("case: path bits %s %s %s %s uniform=%s" % (model, scheme, rng, scramble, uniform), flush=True)
    times = np.arange(N + 1) * 2.0 ** -7 if uniform else np.linspace(0.0, 1.0, N + 1) ** 1.1
    out = []
    for kw in ({}, dict(block_size=256), dict(block_size=128, paths_per_lane=2)):
        plan = sde_sim_rs.Plan(eqs, times, S, init, rng, scheme, seed=3, scramble=scramble, scramble_seed=4, **kw)
        assert ("sde_team_kernel<SdeModel" in plan.source) == (not kw)
        out.append(plan.new_filtration())
        plan.run(out[-1])
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


@pytest.mark.parametrize("scheme", ["euler", "runge-kutta"])
def test_slices_give_the_whole_run(scheme):
    """2 slices of a run of 2^17 paths: the second of 1000 paths only, from path 130,072 on."""
    import sde_sim_rs
    S, first, N = 1 << 17, (1 << 17) - 1000, 40
    print("case: slices %s" % scheme, flush=True)
    times, init = np.arange(N + 1) * 2.0 ** -6, {"S": 100.0, "v": 0.04}
    kinds = []
    for rng in ("pseudo", "sobol"):
        kw = dict(scramble="xor", scramble_seed=4)
        whole = sde_sim_rs.Plan(HESTON, times, S, init, rng, scheme, seed=3, **kw)
        part = sde_sim_rs.Plan(HESTON, times, 1000, init, rng, scheme, seed=3 + first, sobol_first=first, **kw)
        a, b = whole.new_filtration(), part.new_filtration()
        whole.run(a)
        part.run(b)
        torch.cuda.synchronize()
        assert torch.equal(a[:, :, first:], b)
        kinds.append("sde_team_kernel<SdeModel" in part.source and "sde_team_kernel<SdeModel" not in whole.source)
    assert all(kinds)
