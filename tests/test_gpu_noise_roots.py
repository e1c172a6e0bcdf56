"""f64 universes whose noise vanishes like a root elsewhere than at 0, where differences in a last bit grow."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("eqs,init", [
    (["dX = (0.5 * (0.97 - X)) * dt + (0.8 * max(X * (1 - X), 0)^0.5) * dW1"], {"X": 0.5}),
    (["dX = (0.5 * (0.012 - X)) * dt + (0.3 * max(X - 0.01, 0)^0.5) * dW1"], {"X": 0.05}),
])
def test_other_roots_take_the_general_inverse_normal(oracle, eqs, init):
    """Processes whose noise vanishes like a root elsewhere than at 0: their long paths from pseudo-random draws are
    bit for bit those of the same uniforms given by the caller, which take the general inverse normal."""
    import sde_sim_rs
    S, N, seed = 192, 1550, 7
    print("case: f64 roots elsewhere %s" % eqs[0], flush=True)
    times = np.arange(N + 1) / 256.0
    kw = dict(seed=seed, precision="f64")
    plan = sde_sim_rs.Plan(eqs, times, S, init, "pseudo", "euler", **kw)
    f = plan.new_filtration()
    plan.run(f)
    given = sde_sim_rs.Plan(eqs, times, S, init, "injected", "euler", **kw)
    u = torch.tensor(np.stack([oracle.pseudo_f64(seed + s, N) for s in range(S)], axis=1)).cuda()
    g = given.new_filtration()
    given.run(g, injected=u)
    torch.cuda.synchronize()
    assert torch.equal(f, g)
