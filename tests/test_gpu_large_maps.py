"""Large FP64 solves of 3-D maps take no longer a bundle than smaller ones: four
times the bundles, at most 4.3 times the time (2.4 and 3.4 times measured; 5.1
in the one-box kernel of 1024 threads, which spills), statistics and tallies as
the event engine has them (exactly, and to 1e-9: sums in another order)."""
import numpy as np
import pytest

from montecarlocpp_amd import abi, engine, materials, scenes

pytestmark = pytest.mark.gpu


def box12():
    s = scenes.face(abi.DIFF)
    d = scenes.Domain("box")
    d.add_box((0, 0, 0), (3e-7,) * 3, (12, 12, 12), [scenes.face(abi.ISOT, 1.0), s, s, scenes.face(abi.ISOT, -1.0), s, s])
    return d


@pytest.mark.parametrize("dom", [box12, lambda: scenes.porous_film(div=(16, 16, 4))])
def test_large_3d_maps(dom):
    with engine.Scene(materials.si_like(300.0), dom()) as sc:
        ms = {}
        for n in (1_000_000, 4_000_000):
            prob = scenes.problem(n, maxscat=30, seed=7)
            runs = [sc.solve(prob) for _ in range(4)]
            ms[n] = min(r[1]["kernel_ms"] for r in runs)
        sc.set_tune(abi.Tune(engine=abi.ENGINE_EVENT))
        field, stats, _ = sc.solve(prob)
    print(ms)
    for k in ("bundles", "steps", "escapes", "absorbed", "truncated"):
        assert runs[0][1][k] == stats[k]
    assert np.linalg.norm(runs[0][0] - field) <= 1e-9 * np.linalg.norm(field)
    assert ms[4_000_000] <= 4.3 * ms[1_000_000]
