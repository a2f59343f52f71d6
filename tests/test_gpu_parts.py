"""Maps past the LDS are tallied in parts, each running every bundle, only where
that pays: against the general kernel (chosen by walking inside the step),
whose tally is one map in global memory.  Where flights cross about one cell
the parts' repeated flights cost up to six times as much; where they cross
tens of cells parts are several times faster.  The bounds leave a factor of two
to three to what was measured.  Statistics exactly, tallies to 1e-9 in FP64 and
1e-5 in FP32 (whose shares are rounded to FP32)."""
import numpy as np
import pytest

from montecarlocpp_amd import abi, engine, materials, scenes

pytestmark = pytest.mark.gpu

F32, F64 = abi.FP32_FLIGHT, abi.FP64


def cube(edge, div):
    s = scenes.face(abi.DIFF)
    d = scenes.Domain("cube")
    d.add_box((0, 0, 0), (edge,) * 3, div,
              [scenes.face(abi.ISOT, 1.0), s, s, scenes.face(abi.ISOT, -1.0), s, s])
    return d


@pytest.mark.parametrize("dom,tally,precision,n,most", [
    (lambda: cube(5e-5, (64, 64, 64)), abi.MULTI, F64, 100_000, 1.6),
    (lambda: cube(5e-5, (64, 64, 64)), abi.MULTI, F32, 200_000, 1.6),
    (lambda: cube(5e-5, (64, 64, 64)), abi.TEMP, F64, 200_000, 1.6),
    (lambda: cube(1e-5, (1140, 1140, 0)), abi.TEMP, F64, 100_000, 1.6),
    (lambda: scenes.porous_film(div=(128, 128, 0)), abi.MULTI, F64, 50_000, 0.4),
    (lambda: scenes.porous_film(div=(128, 128, 0)), abi.MULTI, F32, 50_000, 0.4),
    (lambda: cube(1e-6, (128, 128, 0)), abi.MULTI, F32, 200_000, 0.5),
])
def test_parts_only_where_they_pay(dom, tally, precision, n, most):
    ms, got = {}, {}
    with engine.Scene(materials.si_like(300.0), dom()) as sc:
        for walks in (0, -1):
            sc.set_tune(abi.Tune(defer_walks=walks))
            prob = scenes.problem(n, tally=tally, maxscat=100, seed=3, precision=precision)
            runs = [sc.solve(prob) for _ in range(4)]
            ms[walks] = min(r[1]["kernel_ms"] for r in runs)
            got[walks] = runs[0]
    print("default", ms[0], "ms, walked inside the step", ms[-1], "ms")
    for k in ("bundles", "steps", "escapes", "absorbed", "truncated"):
        assert got[0][1][k] == got[-1][1][k]
    a, b = got[0][0], got[-1][0]
    assert np.linalg.norm(a - b) <= (1e-9 if precision == F64 else 1e-5) * np.linalg.norm(b)
    assert ms[0] <= most * ms[-1]
