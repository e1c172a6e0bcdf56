"""Forward-rate model at the edges of its kernels: one step, odd step counts (the reverse sweep takes two at
a time), one and odd numbers of steps per accrual period, most forwards dead at expiry, ragged paths;
both storages, f64 against reverse-mode autodiff of the same paths (torch, CPU float64), f32 against f64.

Tolerances: f64 differs in rounding only, 40 steps of a few 1e-16 each against sums over paths, well below
1e-11 of the price and 1e-10 of the largest sensitivity. An f32 step rounds each L four times (6e-8): 40 x 4
x 6e-8 = 1e-5 of L, so 1e-4 of the largest sensitivity, and of the price's sum |dV/dL L|."""
import numpy as np
import pytest

from test_gpu_lmm import _sobol_normals

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _reference(c, eps, e, spp, K, tau=0.25):
    S, N = eps.shape[:2]
    L0 = torch.tensor(c["L0"], requires_grad=True)
    vol, B, dt = torch.tensor(c["vol"]), torch.tensor(c["loadings"]), tau * e / N
    L = L0.expand(S, 40).clone()
    for n in range(N):
        eta = n // spp + 1
        a = tau * vol[eta:] * L[:, eta:] / (1 + tau * L[:, eta:])
        C = torch.cumsum(a[:, :, None] * B[None, eta:, :], dim=1)
        x = (vol[eta:] * (B[None, eta:, :] * C).sum(-1) - 0.5 * vol[eta:] ** 2) * dt
        x = x + vol[eta:] * np.sqrt(dt) * (B[None, eta:, :] * eps[:, n, None, :]).sum(-1)
        L = torch.cat([L[:, :eta], L[:, eta:] * torch.exp(x)], dim=1)
    P = torch.cumprod(1 / (1 + tau * L[:, e:]), dim=1)
    V = torch.clamp(K * tau * P.sum(1) - (1 - P[:, -1]), min=0) / torch.prod(1 + tau * L[:, :e], dim=1)
    V.mean().backward()
    return float(V.mean().detach()), L0.grad.numpy()


@pytest.mark.parametrize("storage", ["tape", "checkpoints"])
@pytest.mark.parametrize("e,spp,S", [(1, 1, 1), (1, 2, 63), (3, 1, 65), (5, 3, 64), (8, 4, 257), (17, 2, 130), (39, 1, 300)])
def test_lmm_edges(oracle, e, spp, S, storage):
    from sde_sim_rs.lmm import ForwardRateModel, forward_rate_config
    c, N, K = forward_rate_config(seed=5), e * spp, 0.05
    print("case: lmm e=%d spp=%d S=%d %s" % (e, spp, S, storage), flush=True)
    price, grad = _reference(c, torch.tensor(_sobol_normals(oracle, S, N, 5)), e, spp, K)
    assert price > 0.0
    out = {}
    for precision in ("f64", "f32"):
        m = ForwardRateModel(steps=N, paths=S, expiry_index=e, strike=K, scramble_seed=5, precision=precision,
                             storage=storage)
        out[precision] = m.evaluate(c["L0"], c["vol"], c["loadings"])
        assert abs(m.evaluate(c["L0"], c["vol"], c["loadings"], adjoint=False)["price"] - out[precision]["price"]) <= \
            1e-12 * abs(out[precision]["price"])
    scale = np.max(np.abs(grad))
    assert abs(out["f64"]["price"] - price) <= 1e-11 * price
    np.testing.assert_allclose(out["f64"]["dL0"], grad, rtol=0, atol=1e-10 * scale)
    assert abs(out["f32"]["price"] - price) <= 1e-4 * np.sum(np.abs(grad * c["L0"]))
    np.testing.assert_allclose(out["f32"]["dL0"], grad, rtol=0, atol=1e-4 * scale)
