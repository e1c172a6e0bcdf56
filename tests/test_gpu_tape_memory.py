"""A forward-rate model's state tape, its largest allocation, is given back with the handle."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_tape_is_released():
    """220 MB a handle (21 states x 40 forwards x 2^16 paths in f32); five more handles leave free memory within one
    2 MiB page of the driver's."""
    import gc
    from sde_sim_rs.lmm import ForwardRateModel, forward_rate_config
    c = forward_rate_config(seed=5)
    print("case: forward-rate tape release", flush=True)

    def cycle():
        m = ForwardRateModel(steps=40, paths=1 << 16, precision="f32", storage="tape")
        held = torch.cuda.mem_get_info()[0]
        m.evaluate(c["L0"], c["vol"], c["loadings"])
        del m
        gc.collect()
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0] - held

    cycle()
    before = torch.cuda.mem_get_info()[0]
    for _ in range(5):
        assert cycle() >= 200 << 20
    assert torch.cuda.mem_get_info()[0] >= before - (2 << 20)
