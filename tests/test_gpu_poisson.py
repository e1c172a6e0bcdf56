"""The inverse Poisson CDF around its first step: jump counts from given uniforms at, just below and just above
1 - lambda and exp(-lambda) equal the oracle's exactly (counts are whole numbers: no tolerance)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("lam", [0.0, 1e-17, 1e-9, 5e-4, 0.3, 0.999, 1.0, 1.5, 40.0])
def test_counts_at_the_edges_equal_the_oracle(oracle, lam):
    import sde_sim_rs
    edges = [0.0, 2.0 ** -53, 0.5, 1.0 - 2.0 ** -53]
    for mid in (1.0 - lam, np.exp(-lam), (1.0 - lam) - 2.0 ** -48):
        edges += [mid + k * 2.0 ** -53 for k in (-40, -32, -3, -2, -1, 0, 1, 2, 3, 31, 32, 33)]
    u = np.array([x for x in edges if 0.0 <= x < 1.0])
    eqs, times, S = ["dX = (1.0) * dN1(%r)" % lam], [0.0, 1.0], len(u)
    print("case: inverse Poisson lambda=%g, %d uniforms" % (lam, S), flush=True)
    plan = sde_sim_rs.Plan(eqs, times, S, {"X": 0.0}, "injected", "euler")
    f = plan.new_filtration()
    plan.run(f, injected=torch.tensor(u.reshape(1, S), dtype=torch.float64, device="cuda"))
    torch.cuda.synchronize()
    ref = oracle.simulate(eqs, times, S, {"X": 0.0}, scheme="euler", rng="injected", injected=u.reshape(S, 1))
    assert np.array_equal(f[-1, 0].cpu().numpy(), np.asarray(ref)[:, -1, 0])
