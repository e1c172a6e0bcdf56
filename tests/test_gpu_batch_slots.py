"""Batch moments on both sides of the number of work items up to which a thread sums an instance's: 8 items of 64
paths and 9, alone and beside instances of other sizes, against the moments of the terminal values.

Tolerance: f64 sums of at most 1280 values of order 1, compensated across items: 1280 roundings of 1.1e-16 are
1.4e-13 of the sums of magnitudes; 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("sizes", [[1], [64], [65], [512], [513], [576], [577], [512, 1, 300, 64], [513, 1, 300, 64],
                                   [1] * 300, [1] * 299 + [1280]])
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("paths_per_lane", [1, 2])
def test_moments(sizes, precision, paths_per_lane):
    import sde_sim_rs
    print("case: batch slots %s x%d %s ppl=%d" % (sizes[:4], len(sizes), precision, paths_per_lane), flush=True)
    inst = [dict(kind=i % 3, steps=3, paths=S, x0=1.0, horizon=0.5, p0=0.5, p1=0.8, p2=0.3, seed=100 + i)
            for i, S in enumerate(sizes)]
    b = sde_sim_rs.Batch(inst, precision=precision, keep_terminal=True)
    b.set_config(paths_per_lane, 128)
    b.run()
    m = np.asarray(b.moments())
    ends = np.split(np.asarray(b.terminal(), dtype=np.float64), np.cumsum(sizes)[:-1])
    for i, x in enumerate(ends):
        var = x.var(ddof=1) if len(x) > 1 else 0.0
        assert abs(m[i, 0] - x.mean()) <= 1e-12 * (1.0 + abs(x.mean())), i
        assert abs(m[i, 1] - var) <= 1e-12 * (1.0 + var), i
