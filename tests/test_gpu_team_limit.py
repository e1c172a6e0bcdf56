"""Up to which path count f64 plans step 64 paths with several waves: 3/2 waves of paths per SIMD of the device."""
import numpy as np
import pytest

from conftest import GBM

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_limit_follows_the_device():
    import sde_sim_rs
    limit = 64 * 4 * torch.cuda.get_device_properties(0).multi_processor_count * 3 // 2
    for paths, team in ((limit, True), (limit + 1, False)):
        plan = sde_sim_rs.Plan(GBM, np.linspace(0.0, 1.0, 25), paths, {"X": 100.0}, "pseudo", "euler", seed=1)
        assert ("sde_team_kernel<SdeModel" in plan.source) == team
