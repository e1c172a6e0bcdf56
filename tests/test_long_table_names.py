"""The long table's name column where one scenario's names exceed what a string chunk holds, with the limit brought down to
a few bytes."""
import numpy as np
import pytest

import sde_sim_rs.api as api

pa = pytest.importorskip("pyarrow")


@pytest.mark.parametrize("limit", [1, 3, 11, 22, 23, 54, 55, 1000, (1 << 31) - 1])
@pytest.mark.parametrize("names", [["X"], ["A", "long name", "ü"], ["", "B"]])
@pytest.mark.parametrize("scenarios", [1, 4])
def test_names_in_any_chunking(monkeypatch, limit, names, scenarios):
    monkeypatch.setattr(api, "_STRING_CHUNK_BYTES", limit)
    times = [0.0, 0.25, 0.5, 0.75, 1.0]
    values = np.arange(scenarios * len(times) * len(names), dtype=np.float64)
    t = api.long_table(names, times, scenarios, values)
    t = t.to_arrow() if hasattr(t, "to_arrow") else t
    t.validate(full=True)
    assert t.column("process_name").to_pylist() == names * (scenarios * len(times))
    assert t.column("time").to_pylist() == [x for x in times for _ in names] * scenarios
    assert t.column("value").to_pylist() == values.tolist()
    size = sum(len(n.encode()) for n in names)
    for chunk in t.column("process_name").chunks:
        assert len(chunk) * size // len(names) <= max(limit, size)


@pytest.mark.parametrize("names,times,scenarios", [(["X"], [], 3), ([], [0.0, 1.0], 2), (["X"], [0.0], 0)])
def test_no_rows(names, times, scenarios):
    t = api.long_table(names, times, scenarios, np.empty(0))
    t = t.to_arrow() if hasattr(t, "to_arrow") else t
    assert t.num_rows == 0 and t.column_names == ["scenario", "time", "process_name", "value"]
