"""A batch of many more solves than workgroups: each small solve is visited once
or so, so sixteen times the solves take a few times the time (3 measured; 30
when workgroups looking for work at the same moment went to the same solves),
and every solve runs whole."""
import numpy as np
import pytest

from montecarlocpp_amd import abi, engine, materials, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [abi.FP64, abi.FP32_FLIGHT])
def test_many_small_solves(precision):
    with engine.Scene(materials.si_like(300.0), scenes.slab(1e-7, 50)) as sc:
        ms = {}
        for n in (250, 4000):
            probs = [scenes.problem(200, seed=k, precision=precision) for k in range(n)]
            runs = [engine.batch_solve([sc] * n, probs) for _ in range(4)]
            ms[n] = min(stats[0]["kernel_ms"] for _, stats in runs)
            for fields, stats in runs[:2]:
                assert all(s["bundles"] == 200 for s in stats)
                for k in range(0, n, n // 25):
                    field, one, _ = sc.solve(probs[k])
                    assert stats[k]["steps"] == one["steps"]
                    assert np.linalg.norm(fields[k] - field) <= 1e-9 * np.linalg.norm(field)
    print("250 solves", ms[250], "ms, 4000", ms[4000], "ms")
    assert ms[4000] <= 12 * ms[250]
