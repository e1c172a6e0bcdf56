"""The inverse Poisson CDF where its argument or intensity is at or past the ends: no jumps for an intensity that is not
positive whatever the uniform, and counts from uniforms around 1 - lambda by the slack of the device's short cut
equal to the oracle's (whole numbers: no tolerance)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("lam", [-40.0, -0.2, -1e-17, 0.0, 1e-17, 2.0 ** -41, 2.0 ** -39, 1e-3, 0.9999999, 2.5, 600.0])
def test_counts_past_the_edges_equal_the_oracle(oracle, lam):
    import sde_sim_rs
    base = 1.0 - lam
    u = [0.0, 0.25, 1.0 - 2.0 ** -53, 1.0] + ([1.25, 2.0] if lam <= 0.0 else [])
    u += [x for k in range(30, 54) for x in (base - 2.0 ** -k, base + 2.0 ** -k) if 0.0 <= x <= 1.0]
    u = np.array(u)
    eqs, times, S = ["dX = (1.0) * dN1(%r)" % lam], [0.0, 1.0], len(u)
    print("case: inverse Poisson lambda=%g, %d uniforms" % (lam, S), flush=True)
    for precision in ("f64", "f32"):
        plan = sde_sim_rs.Plan(eqs, times, S, {"X": 0.0}, "injected", "euler", precision=precision)
        f = plan.new_filtration()
        plan.run(f, injected=torch.tensor(u.reshape(1, S), dtype=torch.float64, device="cuda"))
        torch.cuda.synchronize()
        ref = oracle.simulate(eqs, times, S, {"X": 0.0}, scheme="euler", rng="injected", injected=u.reshape(S, 1))
        got = f[-1, 0].cpu().numpy().astype(np.float64)
        if precision == "f64":
            assert np.array_equal(got, np.asarray(ref)[:, -1, 0])
        elif lam <= 0.0:
            assert not got.any()
