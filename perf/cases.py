"""The work this framework is used for, as a list of measurable cases.

A case is one pass through a public entry point of ``montecarlocpp_amd.engine``:

* ``solve``: ``Scene.solve``, one field solve on a scene already on the GPU,
* ``batch``: ``batch_solve``, many independent solves in one launch,
* ``replay``: ``Batch.run``, a batch captured once and run again with new seeds,
* ``serve``: ``Server.submit`` / ``step`` / ``poll``, requests that arrive together.

Geometry families, sizes and options are those of the repository's own
workloads, tests and benchmark: the cross-plane slab, the rectangular bar, the
porous film, the octet truss and the multi-box film / tee domains, the
Si-like three-branch material at 100 to 500 K, 1e3 to 1e7 bundles, both
precisions, 1-D to 3-D tallies and the cumulative tallies.
"""
import math

import numpy as np
import torch

from montecarlocpp_amd import abi, engine, materials, octet, scenes

PRECISION = {"fp64": abi.FP64, "fp32": abi.FP32_FLIGHT}
TALLY = {"temp": abi.TEMP, "flux": abi.FLUX, "multi": abi.MULTI, "cumtemp": abi.CUMTEMP, "cumflux": abi.CUMFLUX}
SIDE = {"specular": abi.SPEC, "diffuse": abi.DIFF, "partial": abi.PARTIAL}
CUM_BINS = 20

# scatter-steps per bundle, measured: periodic cells end a bundle after
# `maxscat` scatters, boundary crossings come on top
STEPS_PER_SCATTER = {"porous": 1.5, "film": 1.65, "tee": 3.5, "octet": 1.46}
FLOPS_PER_STEP = 120       # one flight, one tally share, one scatter
FLOPS_PER_CROSSING = 12    # one grid cell crossed by a flight: four shares


def listed():
    return [
        # a quick look at a slab: the smallest solve, all latency
        dict(name="slab_small", kind="solve", family="slab", length=1e-7, side="specular", p=0.0, bins=50,
             temp=300.0, bundles=10007, tally="multi", precision="fp32"),
        # the slab the reference runs on its CPU, in the deterministic mode
        dict(name="slab_fp64", kind="solve", family="slab", length=1e-7, side="specular", p=0.0, bins=50,
             temp=300.0, bundles=100000, tally="multi", precision="fp64"),
        # the headline solve
        dict(name="bar_large", kind="solve", family="bar", length=1e-6, width=1e-7, bins=100, temp=300.0,
             bundles=10000000, tally="multi", precision="fp32"),
        # an ordinary solve in the reference's precision
        dict(name="bar_fp64", kind="solve", family="bar", length=1e-6, width=1e-7, bins=100, temp=300.0,
             bundles=1000000, tally="multi", precision="fp64"),
        # a temperature and flux map of a porous film
        dict(name="porous_map", kind="solve", family="porous", nx=64, ny=64, nz=0, maxscat=100, temp=300.0,
             bundles=10000000, tally="multi", precision="fp32"),
        # the same film resolved twice as finely
        dict(name="porous_fine_map", kind="solve", family="porous", nx=128, ny=128, nz=0, maxscat=100, temp=300.0,
             bundles=200000, tally="multi", precision="fp32"),
        # the octet truss: 42 cells of every kind, joined by interfaces
        dict(name="octet", kind="solve", family="octet", maxscat=100, temp=300.0, bundles=1000000, tally="multi",
             precision="fp32"),
        # in-plane conduction along a film, on a coarse map
        dict(name="film_flux", kind="solve", family="film", size=1e-7, n=6, maxscat=100, temp=300.0, bundles=1000000,
             tally="flux", precision="fp32"),
        # flux by scatter order on a multi-box domain, deterministic
        dict(name="tee_cumflux_fp64", kind="solve", family="tee", size=1e-7, n=5, maxscat=200, temp=300.0,
             bundles=150000, tally="cumflux", precision="fp64"),
        # a parameter study: many slabs of every thickness and size at once
        dict(name="batch_slabs", kind="batch", family="slab", solves=256, nmin=1e4, nmax=1e6, precision="fp32"),
        # the seeds of a statistics run over a few geometries, replayed
        dict(name="replay_mix", kind="replay", family="mix", solves=24, nmin=1e4, nmax=1e6, precision="fp32"),
        # a burst of requests of all families at the server
        dict(name="serve_mix", kind="serve", family="mix", solves=60, nmin=1e4, nmax=1e6, precision="fp32"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["solve"] * 7 + ["batch", "replay", "serve"])
    prec = rng.choice(["fp32", "fp32", "fp64"])
    temp = round(rng.uniform(100.0, 500.0), 2)
    if kind in ("batch", "replay", "serve"):
        return dict(kind=kind, family=rng.choice(["slab", "mix"]), solves=int(_log(rng, 4, 65 if kind == "serve" else 129)),
                    nmin=1e4, nmax=_log(rng, 1e5, 1e6), precision=prec)
    family = rng.choice(["slab", "slab", "bar", "bar", "porous", "porous", "film", "octet", "tee"])
    case = dict(kind=kind, family=family, temp=temp, tally=rng.choice(["multi", "multi", "temp", "flux"]), precision=prec)
    half = 1.0 if prec == "fp32" else 0.4      # FP64 passes cost about 2.5 times as much
    if family == "slab":
        side = rng.choice(["specular", "diffuse", "partial"])
        case.update(length=_log(rng, 1e-8, 1e-5), side=side, p=round(rng.random(), 4) if side == "partial" else 0.0,
                    bins=rng.randint(1, 250), bundles=int(_log(rng, 1e3, 4e6 * half)))
    elif family == "bar":
        case.update(length=_log(rng, 1e-7, 3e-6), width=_log(rng, 3e-8, 3e-7), bins=rng.randint(1, 300),
                    bundles=int(_log(rng, 1e4, 6e6 * half)))
    elif family == "porous":
        fine = rng.random() < 0.3
        lo, hi = (73, 160) if fine else (5, 68)
        case.update(nx=rng.randint(lo, hi), ny=rng.randint(lo, hi), nz=0 if fine else rng.choice([0, 0, 0, 3]),
                    maxscat=rng.randint(20, 100), bundles=int(_log(rng, 1e3, 1e5 if fine else 3e6 * half)))
        if case["nz"]:
            case.update(nx=min(case["nx"], 36), ny=min(case["ny"], 36))
    elif family == "octet":
        case.update(maxscat=rng.randint(20, 100), bundles=int(_log(rng, 1e4, 2e6 * half)), tally="multi")
    else:
        case.update(size=_log(rng, 3e-8, 3e-7), n=rng.randint(2, 6), maxscat=rng.randint(41, 200),
                    bundles=int(_log(rng, 1e3, 3e5 * half)),
                    tally=rng.choice(["multi", "flux", "cumtemp", "cumflux"]))
    return case


# ------------------------------------------------------------------ inputs
def _domain(c):
    f = c["family"]
    if f == "slab":
        return scenes.slab(c["length"], c["bins"], side=SIDE[c["side"]], specularity=c["p"])
    if f == "bar":
        return scenes.bar(c["length"], c["width"], c["width"], c["bins"])
    if f == "porous":
        return scenes.porous_film(div=(c["nx"], c["ny"], c["nz"]))
    if f == "octet":
        return octet.octet((6e-7, 1e-7, 1e-7, 1e-8), (4, 2, 2, 1), 1.0)
    s, n = c["size"], c["n"]
    if f == "film":
        return scenes.film((2 * s, s, 2 * s), (2 * n, n, 0), 1e6 * s)
    return scenes.tee((s,) * 4 + (0.5 * s,), (n, n, n, n, 0), 3e6 * s)


def _problem(c, seed):
    cum = c["tally"].startswith("cum")
    return scenes.problem(c["bundles"], tally=TALLY[c["tally"]], maxscat=c.get("maxscat", 10 ** 9), seed=seed,
                          precision=PRECISION[c["precision"]], size=CUM_BINS if cum else 0)


def _many(c, seed):
    """(material, domain, problem) of each solve of a batch or request burst:
    thickness log-uniform in 10 nm to 10 um, T_ref uniform in 100 to 500 K,
    lateral specularity uniform, bundle counts log-uniform, the same for
    every seed; the solves' own seeds come from `seed`."""
    g = np.random.default_rng([c["solves"], 11])
    s = np.random.default_rng([seed, 12])
    out = []
    for i in range(c["solves"]):
        u = g.random(5)
        length = 10.0 ** (-8.0 + 3.0 * u[0])
        bundles = int(10.0 ** (math.log10(c["nmin"]) + math.log10(c["nmax"] / c["nmin"]) * u[3]))
        mat = materials.si_like(100.0 + 400.0 * u[1])
        bins = int(round(20 + 180 * math.log10(length / 1e-8) / 3))
        fam = "random_slab" if c["family"] == "slab" else ("slab", "bar", "random_slab", "porous")[int(4 * u[4])]
        maxscat = 10 ** 9
        if fam == "slab":
            dom = scenes.slab(1e-7, 50)
        elif fam == "bar":
            dom = scenes.bar(1e-6, 1e-7, 1e-7, 100)
        elif fam == "porous":
            dom, maxscat = scenes.porous_film(div=(64, 64, 0)), 100
        else:
            dom = scenes.slab(length, bins, side=abi.PARTIAL, specularity=u[2])
        out.append((mat, dom, scenes.problem(bundles, maxscat=maxscat, seed=int(s.integers(1 << 62)),
                                             precision=PRECISION[c["precision"]])))
    return out


class State:
    pass


def prepare(case, seed):
    st = State()
    st.case = case
    if case["kind"] == "solve":
        st.scene = engine.Scene(materials.si_like(case["temp"]), _domain(case))
        st.problem = _problem(case, _solve_seed(seed))
    else:
        st.requests = _many(case, seed)
        st.problems = [p for _, _, p in st.requests]
        if case["kind"] == "serve":
            st.server = engine.Server()
        else:
            st.scenes = [engine.Scene(m, d) for m, d, _ in st.requests]
            if case["kind"] == "replay":
                st.seeds = [int(p.seed) for p in st.problems]
                st.batch = engine.Batch(st.scenes, st.problems)
    return st


def _solve_seed(seed):
    return int(np.random.default_rng([seed, 10]).integers(1 << 62))


# ------------------------------------------------------------------ passes
WHOLE = ("bundles", "steps", "escapes", "absorbed", "truncated")


def _split(field, tally):
    """A solve's field by quantity: temperatures and heat fluxes have units
    (and sizes) of their own."""
    if tally in (abi.TEMP, abi.CUMTEMP):
        return {"temperature": field}
    if tally in (abi.FLUX, abi.CUMFLUX):
        return {"flux": field}
    return {"temperature": field[:1], "flux": field[1:]}


def _joined(results):
    """The results of many Multi solves, end to end."""
    return {"temperature": np.concatenate([f[0] for f, _ in results]),
            "flux": np.concatenate([f[1:].reshape(-1) for f, _ in results]),
            "counts": np.array([[s[k] for k in WHOLE] for _, s in results], np.int64)}


def run(state):
    kind = state.case["kind"]
    if kind == "solve":
        field, stats, _ = state.scene.solve(state.problem)
        return {**_split(field, state.problem.tally), "counts": np.array([stats[k] for k in WHOLE], np.int64)}
    if kind == "batch":
        return _joined(list(zip(*engine.batch_solve(state.scenes, state.problems))))
    if kind == "replay":
        return _joined(list(zip(*state.batch.run(seeds=state.seeds))))
    ids = [state.server.submit(*r) for r in state.requests]
    done = {}
    while len(done) < len(ids):
        state.server.step()
        for rid in state.server.completed():
            done[rid] = state.server.poll(rid)
    return _joined([done[i] for i in ids])


# ------------------------------------------------------------------ work
def _solve_work(bundles, family, cols, rows, maxscat, length=1e-7, width=1e-7, crossings=0.0, size=4):
    """Bytes and operations of one solve: the sampling tables and the geometry
    read once, the field written once; a flight, its tally share and a
    scatter per scatter-step."""
    if family == "slab":
        steps = bundles * (3.0 + 0.56 * length / 1e-7)
    elif family == "bar":
        steps = bundles * (1.0 + 2.4 * length / width)
    else:
        steps = bundles * STEPS_PER_SCATTER[family] * maxscat
    return {"bytes": 3000 * (16 + 4 * size) + 8 * rows * cols,
            "flops": steps * (FLOPS_PER_STEP + FLOPS_PER_CROSSING * crossings)}


def work(case):
    c, size = case, 4 if case["precision"] == "fp32" else 8
    if c["kind"] != "solve":
        total = {"bytes": 0.0, "flops": 0.0}
        for _, dom, p in _many(c, 0):
            d = list(dom.cells[0].div)
            porous = bool(dom.pores)
            fam = "porous" if porous else ("bar" if d[0] == 100 and dom.name == "bar" else "slab")
            mean_len = dom.cells[0].mat[0]
            w = _solve_work(p.nemit, fam, d[0] * max(1, d[1]), 4, p.maxscat, mean_len, 1e-7,
                            14.4 if porous else 0.0, size)
            total = {k: total[k] + w[k] for k in total}
        return total
    rows = {"temp": 1, "flux": 3, "multi": 4, "cumtemp": CUM_BINS + 1, "cumflux": 3 * (CUM_BINS + 1)}[c["tally"]]
    f = c["family"]
    crossings = 0.0
    if f == "porous":
        cols = c["nx"] * c["ny"] * max(1, c["nz"])
        crossings = 14.4 * (c["nx"] + c["ny"]) / 128.0
    elif f == "octet":
        cols, crossings = 40, 1.0
    elif f == "film":
        cols, crossings = 2 * c["n"] * c["n"], 0.3 * c["n"]
    elif f == "tee":
        cols, crossings = 4 * c["n"] * c["n"], 0.3 * c["n"]
    else:
        cols = c["bins"]
    return _solve_work(c["bundles"], f, cols, rows, c.get("maxscat", 0), c.get("length", 1e-7), c.get("width", 1e-7),
                       crossings, size)


# ------------------------------------------------------------------ 64-bit values
# The slab and bar solves of the same random streams, restated in plain torch
# in 64 bits: one axis-aligned box with isothermal ends and a 1-D tally.
HBAR, KB = 1.054560652927e-034, 1.380648e-023


def _material64(temp, nbins=1000):
    w, dw, vel, dos = [], [], [], []
    for v, cc in ((9.01e3, -2.0e-7), (5.23e3, -2.26e-7), (5.23e3, -2.26e-7)):
        kmax = 1.157e10
        d = (v * kmax + cc * kmax ** 2) / nbins
        om = (np.arange(nbins) + 0.5) * d
        k = (-v + np.sqrt(v * v + 4.0 * cc * om)) / (2.0 * cc)
        vg = v + 2.0 * cc * k
        w.append(om)
        dw.append(np.full(nbins, d))
        vel.append(vg)
        dos.append(k ** 2 / (2.0 * np.pi ** 2 * vg))
    w, dw, vel, dos = (np.concatenate(x) for x in (w, dw, vel, dos))
    rate = 1.32e-45 * w ** 4 + 2e-24 * w ** 2 * temp * math.exp(-140.0 / temp)
    x = HBAR / (KB * temp) * w
    energy = KB * (x / (2.0 * np.sinh(x / 2.0))) ** 2 * dos * dw
    return vel, vel / rate, energy, vel * energy, energy * rate


def _alias64(pdf):
    n, total = len(pdf), 0.0
    for x in pdf:
        total += x
    q = [x * float(n) / total for x in pdf]
    prob, other = [1.0] * n, list(range(n))
    small = [i for i in range(n) if q[i] < 1.0]
    large = [i for i in range(n) if not q[i] < 1.0]
    while small and large:
        s, b = small.pop(), large.pop()
        prob[s], other[s] = q[s], b
        q[b] = (q[b] + q[s]) - 1.0
        (small if q[b] < 1.0 else large).append(b)
    thr = [0xFFFFFFFF if p >= 1.0 else int(p * 4294967296.0) for p in prob]
    return thr, other


M32 = 0xFFFFFFFF


def _mul(a, m):
    """High and low 32 bits of a 32 x 32-bit product."""
    return (a * (m >> 16) + (a * (m & 0xFFFF) >> 16)) >> 16, (a * m) & M32


def _philox(j, event, n, seed):
    c0, c1, c2, c3 = torch.full_like(n, j), event, n & M32, n >> 32
    k0, k1 = seed & M32, seed >> 32
    for _ in range(10):
        h0, l0 = _mul(c0, 0xD2511F53)
        h1, l1 = _mul(c2, 0xCD9E8D57)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return c0, c1, c2, c3


def _uniform(a, b):
    return ((a >> 5).double() * 67108864.0 + (b >> 6).double()) * (1.0 / 9007199254740992.0)


def _rotation(axis, sign):
    """Rotation taking z onto sign * (unit vector of axis)."""
    n = [0.0, 0.0, 0.0]
    n[axis] = sign
    if n[2] < -0.5:
        q = (0.0, 1.0, 0.0)
    else:
        s = math.sqrt((1.0 + n[2]) * 2.0)
        q = (s * 0.5, -n[1] / s, n[0] / s)
    w, x, y = q
    return [[1 - 2 * y * y, 2 * x * y, 2 * y * w], [2 * x * y, 1 - 2 * x * x, -2 * x * w],
            [-2 * y * w, 2 * x * w, 1 - 2 * (x * x + y * y)]]


def exact(case, seed):
    c = case
    if c["kind"] != "solve" or c["family"] not in ("slab", "bar") or c["tally"] != "multi":
        return None
    # diffuse walls magnify a rounding difference by 1 / cos(incidence) a
    # bounce: in a long thin bar two correct 64-bit evaluations of one bundle
    # part, and only the sum over many bundles has a value
    if c["family"] == "bar" and (c["bundles"] < 1000000 or c["length"] > 12 * c["width"]):
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    bar = c["family"] == "bar"
    side = "diffuse" if bar else c["side"]
    width = c["width"] if bar else c["length"]
    dim, hot, bins = (c["length"], width, width), (10.0 if bar else 1.0), c["bins"]
    key = _solve_seed(seed)
    vel, mfp, energy, flux, scat = _material64(c["temp"])
    tab = {k: [torch.tensor(x, dtype=torch.int64, device=dev) for x in _alias64(v.tolist())]
           for k, v in (("flux", flux), ("scat", scat))}
    vel, mfp = (torch.tensor(x, dtype=torch.float64, device=dev) for x in (vel, mfp))
    half = int(max(1, math.ceil(0.5 * c["bundles"] - 0.5)))
    total = 2 * half
    thr = M32 if c.get("p", 0) >= 1 else int(c.get("p", 0) * 4294967296.0)
    rot = {(a, s): _rotation(a, s) for a in range(3) for s in (1.0, -1.0)}

    def pick(table, x):
        prod_hi, prod_lo = _mul(x, 3000)
        return torch.where(prod_lo < table[0][prod_hi], prod_hi, table[1][prod_hi])

    def turn(d, axis, sign):
        r = rot[(axis, sign)]
        return [r[i][0] * d[0] + r[i][1] * d[1] + r[i][2] * d[2] for i in range(3)]

    def cosine(b0, b1):
        r = _uniform(b0[0], b1[0]) * 2.0 - 1.0
        q = math.pi * (_uniform(b0[1], b1[1]) * 2.0 - 1.0)
        s = torch.sqrt(r.abs())
        return [s * torch.cos(q), s * torch.sin(q), torch.sqrt(1.0 - r.abs())], r, q

    def unit(d):
        norm = torch.sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])
        return [x / norm for x in d]

    n = torch.arange(total, dtype=torch.int64, device=dev)
    zero = torch.zeros_like(n)
    b0, b1, b2, b3 = (_philox(j, zero, n, key) for j in range(4))
    r1, r2 = _uniform(b2[0], b3[0]), _uniform(b2[1], b3[1])
    first = n < half                                   # the hot wall x = 0, then the cold wall
    d, _, _ = cosine(b0, b1)
    lo, hi = turn(d, 0, 1.0), turn(d, 0, -1.0)
    u = unit([torch.where(first, a, b) for a, b in zip(lo, hi)])
    p = [(~first).double() * dim[0], torch.where(first, r1, r2) * dim[1],
         torch.where(first, r2, r1) * dim[2]]
    sign = torch.where(first, 1.0, -1.0).double()
    mode = pick(tab["flux"], b0[3])
    path = mfp[mode] * -torch.log1p(-_uniform(b0[2], b1[2]))
    event = zero
    direct = torch.zeros(4, bins, dtype=torch.float64, device=dev)
    diff = torch.zeros(4, bins + 1, dtype=torch.float64, device=dev)
    while n.numel():
        # flight to the nearest face or the intrinsic event
        best, axis = path, torch.full_like(n, -1)
        for a in range(3):
            t = ((u[a] > 0).double() * dim[a] - p[a]) / u[a]
            take = (u[a] != 0) & (t < best)
            best, axis = torch.where(take, t, best), torch.where(take, a, axis)
        path = (path - best).clamp(min=0.0)
        q = [x + best * y for x, y in zip(p, u)]
        event = event + 1
        # tally along x
        amount = [sign * best / vel[mode]] + [sign * (y - x) for x, y in zip(p, q)]
        x0, x1 = p[0] * (bins / dim[0]), q[0] * (bins / dim[0])
        i0, i1 = (x.floor().long().clamp(0, bins - 1) for x in (x0, x1))
        one, up = i0 == i1, i0 < i1
        span = torch.where(one, 1.0, (x1 - x0).abs()).double()
        f0 = torch.where(one, 1.0, torch.where(up, i0 + 1 - x0, x0 - i0) / span)
        f1 = torch.where(one, 0.0, torch.where(up, x1 - i1, i1 + 1 - x1) / span)
        left, right = torch.minimum(i0, i1) + 1, torch.maximum(i0, i1)
        share = torch.where(right > left, 1.0 / span, 0.0)
        for r in range(4):
            direct[r] += torch.bincount(i0, amount[r] * f0, bins) + torch.bincount(i1, amount[r] * f1, bins)
            part = torch.where(right > left, amount[r] * share, 0.0)
            diff[r] += torch.bincount(left, part, bins + 1)[:bins + 1] - torch.bincount(right, part, bins + 1)[:bins + 1]
        # the event
        p = q
        alive = axis != 0
        n, event, mode, sign, path, axis = (x[alive] for x in (n, event, mode, sign, path, axis))
        p, u = [x[alive] for x in p], [x[alive] for x in u]
        b0, b1 = _philox(0, event, n, key), _philox(1, event, n, key)
        dif, r, phi = cosine(b0, b1)
        intr = axis < 0
        s = torch.sqrt(1.0 - r * r)
        iso = [s * torch.cos(phi), s * torch.sin(phi), r]
        new = u
        for a in (1, 2):
            for sg in (1.0, -1.0):
                at = (axis == a) & (torch.sign(u[a]) == -sg)
                mirror = [-x if k == a else x for k, x in enumerate(u)]
                if side == "specular":
                    out = mirror
                else:
                    out = turn(dif, a, sg)
                    if side == "partial":
                        spec = b1[3] < thr
                        out = [torch.where(spec, x, y) for x, y in zip(mirror, out)]
                new = [torch.where(at, x, y) for x, y in zip(out, new)]
        u = unit([torch.where(intr, x, y) for x, y in zip(iso, new)])
        mode = torch.where(intr, pick(tab["scat"], b0[3]), mode)
        path = torch.where(intr, mfp[mode] * -torch.log1p(-_uniform(b0[2], b1[2])), path)
    field = direct + diff.cumsum(1)[:, :bins]
    field[0] /= energy.sum()
    area = dim[1] * dim[2]
    power = 2.0 * area * hot / total * flux.sum() / 4.0
    field *= power / (area * dim[0] / bins)
    field = field.cpu().numpy()
    return {"temperature": field[:1], "flux": field[1:], "counts": None}
