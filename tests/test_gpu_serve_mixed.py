"""A server step of every kind at once: scenes of several cells (the general
launch), a slab and a porous map in parts (the one-box launch, its parts' claim
counters cleared every step), each over several steps (a request gets at least
65,536 bundles a step): statistics as of single solves, tallies of a batch of
the four to 1e-9 (the same kernels, which add FP32 shares in FP64, in another
order; a single octet solve walks its few cells inside the step, with shares
rounded to FP32)."""
import numpy as np
import pytest

from montecarlocpp_amd import abi, engine, materials, octet, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [abi.FP64, abi.FP32_FLIGHT])
def test_every_kind_over_several_steps(precision):
    mat = materials.si_like(300.0)
    doms = [(scenes.porous_film(div=(128, 128, 0)), 20, 150_011), (scenes.slab(1e-7, 50), 10 ** 9, 200_001),
            (scenes.tee((1e-7,) * 4 + (5e-8,), (6, 6, 6, 6, 0), 0.3), 20, 140_007),
            (octet.octet((6e-7, 1e-7, 1e-7, 1e-8), (4, 2, 2, 1), 1.0), 20, 135_001)]
    probs = [scenes.problem(n, maxscat=m, seed=40 + i, precision=precision) for i, (_, m, n) in enumerate(doms)]
    with engine.Server(step_bundles=12_000) as sv:
        ids = [sv.submit(mat, dom, p) for (dom, _, _), p in zip(doms, probs)]
        done, steps = {}, 0
        while len(done) < len(ids) and steps < 1000:
            sv.step()
            steps += 1
            done.update({r: sv.poll(r) for r in sv.completed()})
    assert len(done) == len(ids) and steps >= 3
    scs = [engine.Scene(mat, dom) for dom, _, _ in doms]
    for rid, field, stats, sc, p in zip(ids, *engine.batch_solve(scs, probs), scs, probs):
        alone = sc.solve(p)[1]
        for k in ("bundles", "steps", "escapes", "absorbed", "truncated"):
            assert done[rid][1][k] == stats[k] == alone[k], k
        assert np.linalg.norm(done[rid][0] - field) <= 1e-9 * np.linalg.norm(field)
    for sc in scs:
        sc.close()
