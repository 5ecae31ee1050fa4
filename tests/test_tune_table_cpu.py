"""The autotuner's table: a cost of each configuration for a batch on the
canonical template, for one image and for a batch on the tap-list kernel
(host side only)."""
import json

import numpy as np
import pytest

import opencuda_amd as oc
from opencuda_amd import autotune


@pytest.fixture(autouse=True)
def clean():
    autotune.reset()
    yield
    autotune.reset()


def test_taps_of_an_entry_that_is_not_set():
    c = np.ones(9, np.float32)
    with pytest.raises(oc.BfError) as e:
        oc._check(oc.lib().bf_tune_set_taps(5, 0, c.ctypes.data, c.ctypes.data), "bf_tune_set_taps")
    assert e.value.code == oc.INVALID_DATA
    assert autotune.get_taps(5, 0) == (-1, None, None)


def test_costs_through_a_file(tmp_path):
    n = oc.lib().bf_tune_count()
    a, b, c = ([float(k + s * j) for j in range(n)] for k, s in ((2, 1), (20, -1), (7, 2)))
    path = str(tmp_path / "t.json")
    autotune.save({"0:5": {"best": 0, "ms_per_mpix": a, "taps_ms_per_mpix": b, "batch_taps_ms_per_mpix": c},
                   "1:6": {"best": 0, "ms_per_mpix": a}}, path)
    assert autotune.load(path) == 2
    assert autotune.get(5, 0) == (0, a) and autotune.get_taps(5, 0) == (n - 1, b, c)
    assert autotune.get(6, 1) == (0, a) and autotune.get_taps(6, 1) == (0, a, a)


def test_the_shipped_table_holds_every_cost():
    with open(autotune.DEFAULT_TABLE) as f:
        doc = json.load(f)
    for key, ent in doc["entries"].items():
        cost, taps, many = ent["ms_per_mpix"], ent["taps_ms_per_mpix"], ent["batch_taps_ms_per_mpix"]
        assert len(cost) == len(taps) == len(many) == doc["configs"], key
        assert min(cost + taps + many) > 0, key
        assert many[2:] == cost[2:], key     # the unrolled kernels have configurations 0 and 1
    assert autotune.load() == len(doc["entries"])
