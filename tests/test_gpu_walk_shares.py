"""FP64 shares of a flight among the cells of a 2-D or 3-D map, to the last bit
the crossing parameters allow.

One-flight bundles from the wall x = 0 of a box whose edges and divisions are
powers of two, so that cell coordinates are exact: a flight to x = e cells
gives each cell it crosses whole 1 / e of its x-flux and the last the rest, as
fractions.  A crossing parameter is a quotient in [0, 1], rounded by at most
2^-54, and a share is the difference of two: within 2^-53, and products and the
scale of the field add a few 2^-53 of a share of 1 / 64 at most (flights of 64
cells and more are compared)."""
from fractions import Fraction

import pytest

from montecarlocpp_amd import abi, engine, materials, scenes

pytestmark = pytest.mark.gpu

N, EDGE, BUNDLES = 128, 2.0 ** -20, 200


@pytest.mark.parametrize("how", ["solve", "batch", "replay"])
@pytest.mark.parametrize("div", [(N, 16, 0), (N, 4, 4)])
def test_shares_are_quotients(div, how):
    s = scenes.face(abi.SPEC)
    d = scenes.Domain("wide")
    d.add_box((0, 0, 0), (EDGE, 2.0 ** -16, 2.0 ** -16), div,
              [scenes.face(abi.ISOT, 1.0), s, s, scenes.face(abi.ISOT, -1.0), s, s])
    with engine.Scene(materials.si_like(300.0), d) as sc:
        def prob(i):
            return scenes.problem(4 * BUNDLES, tally=abi.FLUX, maxloop=1, seed=9, first=i, count=1)
        probs = [prob(i) for i in range(BUNDLES)]
        if how == "solve":
            fields = [sc.solve(p)[0] for p in probs]
        elif how == "batch":
            fields = engine.batch_solve([sc] * BUNDLES, probs)[0]
        else:
            with engine.Batch([sc] * BUNDLES, probs) as b:
                fields = b.run()[0]
        whole = scenes.problem(4 * BUNDLES, tally=abi.FLUX, maxloop=1, seed=9)
        ends = [sc.trace(whole, i, cap=4)[0][3] for i in range(BUNDLES)]
    compared, worst = 0, 0.0
    for field, end in zip(fields, ends):
        e = Fraction(end) * N / Fraction(EDGE)
        if not 64 <= e < N:
            continue
        cells = field[0].reshape(-1, N)     # x runs fastest
        got = [sum(Fraction(float(v)) for v in cells[:, j]) for j in range(N)]
        total = sum(got)
        last = int(e)
        for j in range(N):
            exact = Fraction(1) / e if j < last else (e - last) / e if j == last else Fraction(0)
            worst = max(worst, abs(float(got[j] / total - exact)))
        compared += 1
    print("flights", compared, "worst share error", worst)
    assert compared >= 20
    assert worst <= 2.0 ** -53 + 8 * 2.0 ** -53 / 64
