"""Every bundle of a batch, replayed batch or served request runs once, whatever
the grab of ids asked for: grabs smaller than a wavefront, of one wavefront and
uneven ones, for one-box scenes (absorbing and periodic) and several boxes,
against single solves: statistics exactly, tallies to 1e-9 (FP64 sums in
another order; FP32 shares are added in FP64)."""
import numpy as np
import pytest

from montecarlocpp_amd import abi, engine, materials, scenes

pytestmark = pytest.mark.gpu

CASES = [
    (lambda: scenes.slab(1e-7, 20), 10 ** 9, 1),
    (lambda: scenes.slab(1e-7, 20), 10 ** 9, 5003),
    (lambda: scenes.film((2e-7, 1e-7, 2e-7), (4, 2, 0), 0.1), 20, 4097),
    (lambda: scenes.tee((1e-7,) * 4 + (5e-8,), (2, 2, 2, 2, 0), 0.3), 20, 65),
    (lambda: scenes.tee((1e-7,) * 4 + (5e-8,), (2, 2, 2, 2, 0), 0.3), 20, 4099),
]


def check(got, want):
    for (fa, sa), (fb, sb) in zip(got, want):
        for k in ("bundles", "steps", "escapes", "absorbed", "truncated"):
            assert sa[k] == sb[k], k
        assert np.linalg.norm(fa - fb) <= 1e-9 * np.linalg.norm(fb)


@pytest.mark.parametrize("precision", [abi.FP64, abi.FP32_FLIGHT])
@pytest.mark.parametrize("chunk", [1, 32, 63, 64, 70])
def test_every_bundle_once(chunk, precision):
    mat, tune = materials.si_like(300.0), abi.Tune(chunk=chunk)
    scs = [engine.Scene(mat, dom()) for dom, _, _ in CASES]
    probs = [scenes.problem(n, maxscat=m, seed=30 + i, precision=precision) for i, (_, m, n) in enumerate(CASES)]
    want = [sc.solve(p)[:2] for sc, p in zip(scs, probs)]
    check(list(zip(*engine.batch_solve(scs, probs, tune))), want)
    with engine.Batch(scs, probs, tune) as b:
        for _ in range(2):
            check(list(zip(*b.run())), want)
    with engine.Server(step_bundles=6000, tune=tune) as sv:
        ids = [sv.submit(mat, sc.dom, p) for sc, p in zip(scs, probs)]
        done = {}
        for _ in range(1000):
            sv.step()
            done.update({r: sv.poll(r) for r in sv.completed()})
            if len(done) == len(ids):
                break
        check([done[i] for i in ids], want)
    for sc in scs:
        sc.close()
