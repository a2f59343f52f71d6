"""The cell an Inter face with several partners continues in, FP32 flight
(partners tested with their faces together) against FP64 (face by face):
partners of five, six and ten faces, more than the six tested together."""
import numpy as np
import pytest

from montecarlocpp_amd import abi, engine, materials, scenes
from tests.ngon_scenes import ngon_mat

pytestmark = pytest.mark.gpu

A, C, H = 1e-7, 2.5e-8, 5e-8
WALL = scenes.face(abi.SPEC)
JOIN = scenes.face(abi.INTER)


def roofed():
    """A box whose top face joins an octagonal prism, triangular prisms over
    two of its corners and boxes over the other two (which reach into the
    prism's plan: the pair listed first wins there)."""
    d = scenes.Domain("roofed")
    base = d.add_box((0.0, 0.0, 0.0), (A, A, H), (0, 0, 0), [scenes.face(abi.ISOT, 1.0)] + [WALL] * 4 + [JOIN])
    octagon = np.array([[C, 0], [A - C, 0], [A, C], [A, A - C], [A - C, A], [C, A], [0, A - C], [0, C]])
    cells = [d.add_cell(abi.PRISM, (C, 0.0, H), ngon_mat(np.array([0.0, 0.0, H]), octagon - octagon[0]), 0,
                        [JOIN] + [WALL] * 9)]
    for origin, e0, e1 in (((0, 0), (C, 0), (0, C)), ((A, A), (-C, 0), (0, -C))):
        m = np.zeros((3, 3))
        m[:2, 0], m[:2, 1], m[2, 2] = e0, e1, H
        cells.append(d.add_cell(abi.TRIPRISM, (*map(float, origin), H), m, (0, 0, 0),
                                [WALL, WALL, JOIN, WALL, WALL]))
    for origin in ((A - C, 0.0), (0.0, A - C)):
        cells.append(d.add_box((*origin, H), (C, C, H), (0, 0, 0), [WALL, WALL, JOIN, WALL, WALL, WALL]))
    for c in cells:
        d.pair(base, 5, c, 0 if c == cells[0] else 2)
    return d, base, cells


def test_partner_matches_fp64():
    mat = materials.si_like(300.0)
    d, base, cells = roofed()
    rng = np.random.default_rng(5)
    # starts just below the joined face, aimed at points at least 1e-3 of an
    # edge (far over FP32's rounding) from every partner's outline
    pts = [(A / 2, A / 2), (0.3 * C, 0.3 * C), (A - 0.3 * C, A - 0.3 * C), (A - 0.2 * C, 0.2 * C), (0.2 * C, A - 0.2 * C)]
    while len(pts) < 65:
        x, y = rng.uniform(0.02, 0.98, 2) * A
        cuts = [x + y - C, 2 * A - C - x - y, x - (A - C), y - C, x - C, y - (A - C),
                A - C - (x - y), A - C - (y - x)]
        if min(abs(v) for v in cuts) > 1e-3 * A:
            pts.append((x, y))
    got = {}
    with engine.Scene(mat, d) as sc:
        for prec in (abi.FP64, abi.FP32_FLIGHT):
            prob = scenes.problem(10, seed=3, maxscat=1, precision=prec)
            got[prec] = [sc.trace_from(prob, (x, y, H * 0.999), dir=(0.0, 0.0, 1.0), cap=8)[0] for x, y in pts]
    seen = set()
    for a, b in zip(got[abi.FP64], got[abi.FP32_FLIGHT]):
        assert int(a[1]) == int(b[1])
        assert int(a[12]) == int(b[12])
        if int(a[1]) >= 0:
            seen.add(int(a[12]))
    assert seen == set(cells)
