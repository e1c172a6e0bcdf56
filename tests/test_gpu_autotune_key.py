"""The batch autotuner uses a remembered configuration only for the kernels and the device it was timed with."""
import subprocess
import sys

import pytest

from conftest import _PKG_ROOT

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CHILD = """
import sys
sys.path.insert(0, %r)
import sde_sim_rs
from sde_sim_rs import models
p, b, ms = sde_sim_rs.Batch(models.batched_instances(n=8, seed=9), precision="f32").autotune()
print("tuned", p, b, "timed" if ms > 0 else "remembered")
"""


def _tune(cache):
    import os
    r = subprocess.run([sys.executable, "-c", CHILD % _PKG_ROOT], env=dict(os.environ, SDESIM_CACHE_DIR=str(cache)),
                       capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout.split("tuned ")[1].split()


def test_key(tmp_path):
    print("case: autotune key", flush=True)
    p, b, how = _tune(tmp_path)
    assert how == "timed"
    assert _tune(tmp_path) == [p, b, "remembered"]
    entry = (tmp_path / "autotune.txt").read_text().split()
    key, rest = entry[0], " ".join(entry[1:])
    shape = "-".join(key.split("-")[:3])  # precision, instances, sizes: the whole key once
    assert key != shape
    code, device = key.split("-")[3], "-".join(key.split("-")[4:])
    others = [shape, "%s-%s-%s" % (shape, "0" * len(code), device), "%s-%s-%s" % (shape, code, device + "0")]
    (tmp_path / "autotune.txt").write_text("".join("%s %s\n" % (k, rest) for k in others))
    assert _tune(tmp_path)[2] == "timed"
