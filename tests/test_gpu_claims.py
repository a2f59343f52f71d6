"""Every bundle runs once, whatever the grabs of ids: solves from one bundle to
past one a lane of the largest launch, absorbing and not, default and tuned
grabs, against the event engine (which claims no ids): per-bundle counts
exactly, tallies to 1e-9 (FP64, other summation orders) or 1e-5 (FP32, whose
grid walks round their shares to FP32)."""
import numpy as np
import pytest

from montecarlocpp_amd import abi, engine, materials, scenes

pytestmark = pytest.mark.gpu

SCENES = {
    "slab": (lambda: scenes.slab(1e-7, 20), 10 ** 9),                               # one box, absorbing
    "film": (lambda: scenes.film((2e-7, 1e-7, 2e-7), (4, 2, 0), 0.1), 3),           # one box, periodic
    "tee": (lambda: scenes.tee((1e-7,) * 4 + (5e-8,), (2, 2, 2, 2, 0), 0.3), 3),    # several boxes
}


@pytest.mark.parametrize("precision", [abi.FP64, abi.FP32_FLIGHT])
@pytest.mark.parametrize("name", sorted(SCENES))
@pytest.mark.parametrize("n,chunk", [(1, 0), (64, 0), (65, 5000), (4097, 64), (262145, 0), (600001, 0), (600001, 70)])
def test_every_bundle_once(name, n, chunk, precision):
    dom, maxscat = SCENES[name]
    mat = materials.si_like(300.0)
    prob = scenes.problem(n, maxscat=maxscat, seed=n, precision=precision)
    with engine.Scene(mat, dom()) as sc:
        sc.set_tune(abi.Tune(chunk=chunk))
        fa, sa, ca = sc.solve(prob, counts=True)
        sc.set_tune(abi.Tune(engine=abi.ENGINE_EVENT))
        fb, sb, cb = sc.solve(prob, counts=True)
    for k in ("nscat", "nbdry", "nstep", "fate"):
        np.testing.assert_array_equal(getattr(ca, k), getattr(cb, k), err_msg=k)
    for k in ("bundles", "steps", "escapes", "absorbed", "truncated"):
        assert sa[k] == sb[k]
    assert np.linalg.norm(fa - fb) <= (1e-9 if precision == abi.FP64 else 1e-5) * np.linalg.norm(fb)
