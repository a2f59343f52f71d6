"""The one-box kernel at the edges of its rule and of its tally layout: 1-D
tallies up to the fixed LDS row stride and past it (the general kernel), a
single cell, no tally, 2-D and 3-D maps, maps larger than the LDS (in parts
of several rows, one row, or a range of columns, and past the most parts), each tally kind, every face kind it
takes, a box away from the origin, a pore of each kind of wall.

FP64 is compared with the oracle: per-bundle counts exactly, tallies to 1e-9
(sums of at most 1e6 terms in another order: about 1e6 * 2^-53 = 1e-10 of the
largest partial sum).  FP32 flight is compared with the event engine, which
takes the general kernel's steps: counts exactly, tallies to 1e-5 (a grid
walk's shares are rounded to FP32 there, 6e-8 each)."""
import numpy as np
import pytest

from montecarlocpp_amd import abi, engine, materials, scenes

pytestmark = pytest.mark.gpu

COUNTS = ("nscat", "nbdry", "nstep", "fate")


def box(dim, div, faces, origin=(0.0, 0.0, 0.0), grad=(0.0, 0.0, 0.0), peri=()):
    d = scenes.Domain("box")
    s = d.add_box(origin, dim, div, faces, grad_t=grad)
    for a in peri:
        shift = [0.0, 0.0, 0.0]
        shift[a] = dim[a]
        d.pair(s, a, s, a + 3, transl=shift)
    return d


def faces(*kinds):
    """Bac Lef Bot Fro Rig Top: (kind, T or specularity)."""
    out = []
    for k, v in kinds:
        out.append(scenes.face(k, v if k == abi.ISOT else 0.0, v if k == abi.PARTIAL else 0.0))
    return out


I, S, D, P = abi.ISOT, abi.SPEC, abi.DIFF, abi.PARTIAL
WALLS = faces((I, 2.0), (D, 0), (P, 0.4), (I, -2.0), (S, 0), (P, 0.7))
L = (2e-7, 1e-7, 6e-8)


def pored(kind, spec, div):
    d = scenes.porous_film(div=div, pore=kind, walls=abi.PARTIAL, specularity=spec)
    return d


CASES = {
    "cols_255": (lambda: box(L, (255, 0, 0), WALLS), abi.MULTI),
    "cols_256": (lambda: box(L, (256, 0, 0), WALLS), abi.MULTI),
    "one_col": (lambda: box(L, (1, 0, 0), WALLS), abi.MULTI),
    "single_cell": (lambda: box(L, (0, 0, 0), WALLS), abi.MULTI),
    "no_tally": (lambda: box(L, (-1, 0, 0), WALLS), abi.MULTI),
    "along_y_temp": (lambda: box(L, (0, 17, 0), WALLS), abi.TEMP),
    "along_z_flux": (lambda: box(L, (0, 0, 9), WALLS), abi.FLUX),
    "offset": (lambda: box(L, (13, 0, 0), WALLS, origin=(3e-7, -2e-7, 1e-7)), abi.MULTI),
    "grid_yz_flux": (lambda: box(L, (0, 11, 6), WALLS, origin=(1e-7, 0.0, -5e-8)), abi.FLUX),
    "grid_xz_temp": (lambda: box(L, (8, 0, 3), WALLS), abi.TEMP),
    "grid_2x2": (lambda: box(L, (2, 2, 0), WALLS), abi.MULTI),
    "grid_3d": (lambda: box(L, (7, 5, 3), WALLS), abi.MULTI),
    "parts_rows": (lambda: box(L, (100, 60, 0), WALLS), abi.MULTI),
    "parts_3d": (lambda: box(L, (40, 16, 16), WALLS), abi.MULTI),
    "parts_cols_odd": (lambda: box(L, (211, 149, 0), WALLS), abi.TEMP),
    "parts_cols_flux": (lambda: scenes.porous_film(div=(160, 131, 0)), abi.FLUX),
    "parts_past_most": (lambda: box(L, (1200, 1201, 0), WALLS), abi.TEMP),
    "film": (lambda: scenes.film((2e-7, 1e-7, 2e-7), (6, 3, 0), 0.2), abi.MULTI),
    "bulk_all_periodic": (lambda: box(L, (9, 0, 0), [scenes.face(abi.PERI)] * 6, grad=(-1e6, 0.0, 0.0), peri=(0, 1, 2)),
                          abi.MULTI),
    "pore_diffuse": (lambda: pored(abi.DIFF, 0.3, (20, 20, 0)), abi.MULTI),
    "pore_specular": (lambda: pored(abi.SPEC, 0.3, (9, 0, 0)), abi.MULTI),
    "pore_partial": (lambda: pored(abi.PARTIAL, 0.5, (5, 6, 4)), abi.FLUX),
}


def solved(scene, prob):
    field, stats, counts = scene.solve(prob, counts=True)
    return field, stats, {k: getattr(counts, k) for k in COUNTS}


def close(a, b, tol):
    assert np.linalg.norm(a - b) <= tol * max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("name", sorted(CASES))
def test_fp64_matches_oracle(name):
    from oracle import oracle
    dom, tally = CASES[name]
    mat, dom = materials.si_like(300.0), dom()
    prob = scenes.problem(3001, tally=tally, maxscat=60, seed=11, precision=abi.FP64)
    fo, _, co = oracle.solve(mat, dom, prob, counts=True)
    with engine.Scene(mat, dom) as sc:
        fg, _, cg = solved(sc, prob)
    for k in COUNTS:
        np.testing.assert_array_equal(cg[k], getattr(co, k), err_msg=k)
    if fo.size:
        close(fg, fo, 1e-9)


@pytest.mark.parametrize("name", sorted(CASES))
def test_fp32_matches_general_steps(name):
    dom, tally = CASES[name]
    mat, dom = materials.si_like(300.0), dom()
    prob = scenes.problem(20011, tally=tally, maxscat=60, seed=12, precision=abi.FP32_FLIGHT)
    with engine.Scene(mat, dom) as sc:
        fb, sb, cb = solved(sc, prob)
        sc.set_tune(abi.Tune(engine=abi.ENGINE_EVENT))
        fe, se, ce = solved(sc, prob)
    for k in COUNTS:
        np.testing.assert_array_equal(cb[k], ce[k], err_msg=k)
    for k in ("bundles", "steps", "escapes", "absorbed", "truncated"):
        assert sb[k] == se[k]
    if fe.size:
        close(fb, fe, 1e-5)


@pytest.mark.parametrize("precision", [abi.FP64, abi.FP32_FLIGHT])
def test_batch_of_all_matches_single(precision):
    """Every case above in one batch, several sizes of each: the one-box solves
    share a launch (1-D, 2-D and 3-D tallies, parts, all tally kinds), the
    others the general batch kernel.  Statistics exactly, tallies to 1e-9
    (other summation orders)."""
    mat = materials.si_like(300.0)
    scs, probs = [], []
    for i, name in enumerate(sorted(CASES)):
        dom, tally = CASES[name]
        scs.append(engine.Scene(mat, dom()))
        probs.append(scenes.problem((7, 1500, 9001)[i % 3], tally=tally, maxscat=60, seed=20 + i, precision=precision))
    alone = [sc.solve(p) for sc, p in zip(scs, probs)]
    fields, stats = engine.batch_solve(scs, probs)
    with engine.Batch(scs, probs) as b:
        replays = [b.run() for _ in range(2)]
    for got_f, got_s in [(fields, stats)] + replays:
        for (fa, sa, _), fb, sb in zip(alone, got_f, got_s):
            for k in ("bundles", "steps", "escapes", "absorbed", "truncated"):
                assert sa[k] == sb[k]
            if fa.size:
                close(fb, fa, 1e-9)
    for sc in scs:
        sc.close()


def test_batch_of_one_tiny_solve():
    mat, dom = materials.si_like(300.0), CASES["cols_255"][0]()
    with engine.Scene(mat, dom) as sc:
        prob = scenes.problem(2, seed=3, precision=abi.FP32_FLIGHT)
        fa, sa, _ = sc.solve(prob)
        fb, sb = engine.batch_solve([sc], [prob])
    assert sa["steps"] == sb[0]["steps"]
    close(fb[0], fa, 1e-9)


@pytest.mark.parametrize("block", [0, 64, 1024])
@pytest.mark.parametrize("name,n", [("grid_3d", 5003), ("parts_rows", 5003), ("grid_2x2", 1 << 21)])
def test_fp64_grid_launch_shapes(name, n, block):
    """FP64 grids, single and in a batch: a small solve's kernel of at most 512
    threads (launched with those where the tuning says more) and, at the last
    size, a large solve's of up to 1024, against the event engine: counts
    exactly, tallies to 1e-9 (other summation orders)."""
    dom, tally = CASES[name]
    mat, dom = materials.si_like(300.0), dom()
    prob = scenes.problem(n, tally=tally, maxscat=20, seed=14, precision=abi.FP64)
    with engine.Scene(mat, dom) as sc:
        sc.set_tune(abi.Tune(engine=abi.ENGINE_EVENT))
        fa, sa, ca = solved(sc, prob)
        sc.set_tune(abi.Tune(block=block))
        fb, sb, cb = solved(sc, prob)
        fc, stats = engine.batch_solve([sc], [prob], tune=abi.Tune(block=block))
    for k in COUNTS:
        np.testing.assert_array_equal(cb[k], ca[k], err_msg=k)
    assert sb["steps"] == sa["steps"] == stats[0]["steps"]
    close(fb, fa, 1e-9)
    close(fc[0], fa, 1e-9)
