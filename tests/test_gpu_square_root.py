"""f64 square-root processes: the batch kernel's CIR and its DSL form agree bit for bit on both sides
of the rule that keeps the library's inverse normal (4 kappa theta < sigma^2), and only universes on its
near side are generated with it."""
import numpy as np
import pytest

from conftest import GBM, HESTON

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("kappa,theta,sigma", [(0.65, 0.0068, 0.31), (0.5, 0.02, 0.2), (0.5, 0.02, 0.2001),
                                               (2.0, 0.07, 0.25)])
def test_cir_batch_equals_its_dsl_form(kappa, theta, sigma):
    import sde_sim_rs
    from sde_sim_rs import models
    S, N = 321, 300
    print("case: f64 CIR kappa=%g theta=%g sigma=%g" % (kappa, theta, sigma), flush=True)
    inst = dict(kind=models.CIR, steps=N, paths=S, x0=0.03, horizon=N * 2.0 ** -8, p0=kappa, p1=theta, p2=sigma, seed=5)
    b = sde_sim_rs.Batch([inst], precision="f64", keep_terminal=True)
    b.run()
    plan = sde_sim_rs.Plan(models.cir(kappa, theta, sigma), np.arange(N + 1) * 2.0 ** -8, S, {"X": 0.03}, "pseudo", "euler",
                           seed=5)
    assert ("SDE_LIBRARY_F64" in plan.source) == (4.0 * (kappa * theta) < sigma * sigma)
    f = plan.new_filtration()
    plan.run(f)
    torch.cuda.synchronize()
    assert np.array_equal(b.terminal(), f[-1, 0].cpu().numpy())


@pytest.mark.parametrize("eqs,init,library", [
    (GBM, {"X": 100.0}, False),
    (HESTON, {"S": 100.0, "v": 0.04}, False),
    ([HESTON[0], HESTON[1].replace("0.5 * max", "2.0 * max")], {"S": 100.0, "v": 0.04}, True),
    (["dX = (0.1) * dt + (0.3) * dW1"], {"X": 0.0}, False),
    (["dX = (0.1 * (1.0 - X)) * dt + (abs(X)^0.4) * dW1"], {"X": 1.0}, True),
])
def test_library_inverse_normal_is_kept_where_differences_grow(eqs, init, library):
    import sde_sim_rs
    for precision in ("f64", "f32"):
        plan = sde_sim_rs.Plan(eqs, [0.0, 0.5, 1.0], 4, init, "pseudo", "euler", seed=1, precision=precision)
        assert ("SDE_LIBRARY_F64" in plan.source) == (library and precision == "f64")


@pytest.mark.parametrize("rng,scramble", [("pseudo", "shift"), ("sobol", "shift"), ("sobol", "xor")])
@pytest.mark.parametrize("scheme", ["euler", "runge-kutta"])
def test_library_kernels_match_the_oracle(oracle, rng, scramble, scheme):
    """Few steps of a universe on the library side, before differences can grow."""
    import sde_sim_rs
    from sde_sim_rs import models
    eqs, S, times = models.cir(0.65, 0.0068, 0.31), 200, np.linspace(0.0, 0.05, 9)
    print("case: f64 library kernel %s %s %s" % (rng, scramble, scheme), flush=True)
    kw = dict(seed=3, scramble=scramble, scramble_seed=4)
    plan = sde_sim_rs.Plan(eqs, times, S, {"X": 0.05}, rng, scheme, **kw)
    assert "SDE_LIBRARY_F64" in plan.source
    f = plan.new_filtration()
    plan.run(f)
    torch.cuda.synchronize()
    ref = oracle.simulate(eqs, times, S, {"X": 0.05}, scheme=scheme, rng=rng, **kw)
    assert np.all(np.abs(f.cpu().numpy().transpose(2, 0, 1) - ref) <= 1e-12 * np.abs(ref) + 1e-12)
