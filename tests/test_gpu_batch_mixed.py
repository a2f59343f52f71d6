"""A batch of one-box scenes and scenes of several cells runs its two launches
side by side: a film and a tee of a few long bundles each take little more than
the longer of the two, eagerly and in a replayed graph (0.55 of the sum
measured, the sum itself one after the other), and every solve equals its
single one: statistics exactly, tallies to 1e-9 (sums in another order), on
every replay, with eager work between."""
import numpy as np
import pytest

from montecarlocpp_amd import abi, engine, materials, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [abi.FP64, abi.FP32_FLIGHT])
def test_mixed_batch_side_by_side(precision):
    mat = materials.si_like(300.0)
    tee = engine.Scene(mat, scenes.tee((1e-7,) * 4 + (5e-8,), (6, 6, 6, 6, 0), 0.3))
    film = engine.Scene(mat, scenes.film((2e-7, 1e-7, 2e-7), (12, 6, 0), 0.1))
    scs = [tee, film]
    probs = [scenes.problem(100, maxscat=m, seed=4, precision=precision) for m in (100, 400)]
    want = [sc.solve(p)[:2] for sc, p in zip(scs, probs)]

    def check(run):
        for (fa, sa), (fb, sb) in zip(zip(*run), want):
            for k in ("bundles", "steps", "escapes", "absorbed", "truncated"):
                assert sa[k] == sb[k], k
            assert np.linalg.norm(fa - fb) <= 1e-9 * np.linalg.norm(fb)
        return run[1][0]["kernel_ms"]

    alone = [min(engine.batch_solve([sc], [p])[1][0]["kernel_ms"] for _ in range(4)) for sc, p in zip(scs, probs)]
    eager = min(check(engine.batch_solve(scs, probs)) for _ in range(4))
    with engine.Batch(scs, probs) as b:
        replay = []
        for _ in range(5):
            replay.append(check(b.run()))
            check(engine.batch_solve(scs, probs))
    print("alone", alone, "together", eager, "replayed", min(replay))
    assert eager <= 0.8 * sum(alone)
    assert min(replay) <= 0.8 * sum(alone)
    for sc in scs:
        sc.close()
