"""Timed workloads of the residual-and-update path.

Every case is a pass that a program using this library makes: a chunk of
solver iterations with its residual and force histories and the state after
it (the drop-in executable's and the solve server's loop), a time-accurate
run, a batch of capped solves, one residual evaluation, a wall distance.
Meshes are built in memory and handed over as a csu_mesh_desc; the options
come from an input.dat that the host library reads.

`exact` restates the inviscid path in plain numpy FP64.
"""
from __future__ import annotations

import ctypes as C
import functools
import math
import tempfile

import numpy as np

from csu_amd import cases as gen
from csu_amd import native, renumber

CHUNK = 25            # iterations a pass asks for: the solve server's chunk
CHUNK_LARGE = 100     # the same of large explicit runs, nearer the executable's 200
FLUXES = ("ROE", "AUSM", "AUSMDV")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one residual evaluation with all its fields to the host: the
        # smallest call, on a small odd mesh
        {"name": "residual_small", "kind": "residual", "nx": 41, "ny": 17, "flux": "AUSMDV", "split": True,
         "morton": False, "precision": 0},
        # the reference's own configuration: 40k-cell Euler ramp, RK5, FP64,
        # in the generator's cell order
        {"name": "ramp_rk_40k", "kind": "rk", "nx": 200, "ny": 100, "flux": "ROE", "split": True, "morton": False,
         "precision": 0},
        # the same far above the caches, renumbered along a Morton curve (the
        # benchmark's form): the largest
        {"name": "ramp_rk_2m", "kind": "rk", "nx": 1414, "ny": 707, "flux": "ROE", "split": True, "morton": True,
         "precision": 0},
        # mixed precision, an odd size in between
        {"name": "ramp_rk_mixed_400k", "kind": "rk", "nx": 613, "ny": 331, "flux": "ROE", "split": True,
         "morton": True, "precision": 1},
        # explicit laminar plate: viscous terms, quads with some triangles
        {"name": "plate_rk_100k", "kind": "plate", "nx": 701, "ny": 131, "scheme": "RK", "precision": 0},
        # implicit laminar plate, DPLUR at CFL 50 (56k cells)
        {"name": "plate_dplur_56k", "kind": "plate", "nx": 500, "ny": 100, "scheme": "DPLUR", "precision": 0},
        # airfoil with a turbulence model, LU-SGS on the colour order
        {"name": "naca_sa_250k", "kind": "naca", "ni": 1000, "nfar": 105, "model": "sa", "flux": "ROE",
         "precision": 0},
        {"name": "naca_sst_110k", "kind": "naca", "ni": 611, "nfar": 70, "model": "sst", "flux": "AUSMDV",
         "precision": 0},
        # what the solve server runs: several Euler ramps at once, LU-SGS, to
        # an iteration cap
        {"name": "served_lusgs", "kind": "served", "ny": 50, "solves": 4, "cap": 50},
        # the many-solve mix's ramps: one batch of unlike sizes, mixed precision
        {"name": "batch_rk_mixed", "kind": "batch", "ny": 71, "solves": 8, "precision": 1},
        # time-accurate shock tube to its end time
        {"name": "tube", "kind": "tube", "nx": 400, "ny": 41, "tmax": 0.008},
        # wall distance of an airfoil mesh, the set-up step of SA and SST runs
        {"name": "wall_distance_250k", "kind": "walldist", "ni": 1000, "nfar": 105},
    ]


def _chunk(case):
    return CHUNK_LARGE if case["kind"] in ("rk", "plate") and _cells_of(case) > 1e5 and \
        case.get("scheme", "RK") == "RK" else CHUNK


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["residual", "rk", "rk", "rk", "plate", "plate", "naca", "naca", "served", "batch", "tube",
                       "walldist"])
    if kind in ("residual", "rk"):
        n = _log(rng, 500, 20e3) if kind == "residual" else _log(rng, 3e3, 1.2e6)
        ny = max(8, int(math.sqrt(n / 4) * rng.uniform(0.8, 1.25)))
        split = rng.random() < 0.75
        nx = max(8, int(n / ny / (2 if split else 1)))
        return {"kind": kind, "nx": nx, "ny": ny, "flux": rng.choice(FLUXES), "split": split,
                "morton": rng.random() < 0.5, "precision": rng.choice([0, 0, 1])}
    if kind == "plate":
        ny = int(_log(rng, 40, 140))
        return {"kind": kind, "nx": int(ny * rng.uniform(3.5, 6.0)), "ny": ny, "scheme": rng.choice(["RK", "DPLUR"]),
                "precision": rng.choice([0, 0, 1])}
    if kind == "naca":
        return {"kind": kind, "ni": 2 * int(_log(rng, 60, 480)), "nfar": rng.randint(30, 100),
                "model": rng.choice(["sa", "sst"]), "flux": rng.choice(["ROE", "AUSMDV"]),
                "precision": rng.choice([0, 0, 1])}
    if kind == "served":
        return {"kind": kind, "ny": rng.randint(30, 90), "solves": rng.randint(2, 8), "cap": rng.choice([50, 75])}
    if kind == "batch":
        return {"kind": kind, "ny": rng.randint(30, 110), "solves": rng.randint(3, 10), "precision": rng.choice([0, 1])}
    if kind == "tube":
        return {"kind": kind, "nx": rng.randint(100, 420), "ny": rng.randint(8, 45), "tmax": 0.008}
    return {"kind": "walldist", "ni": 2 * int(_log(rng, 60, 500)), "nfar": rng.randint(30, 105)}


# ---------------------------------------------------------------------------
# meshes in memory
# ---------------------------------------------------------------------------
class MeshCase:
    """A mesh in memory with the options of an input.dat, in the shape of
    native.HostCase that Device, Batch and wall_distance_dev take."""

    def __init__(self, nodes, cells, markers, inputs):
        self.a = a = _connect(nodes, cells, [e for _, e in markers])
        bc = {v: k for k, v in gen.BC_NAMES.items()}
        a["mark_type"] = np.array([bc[inputs["BC:" + name]] for name, _ in markers], np.int32)
        with tempfile.TemporaryDirectory(prefix="pc") as d:   # options through the host's own reader, on a tiny mesh
            tiny = gen.ramp_mesh(2, 2, jitter=0.0)
            tiny.markers = [(n, e) for (n, _), e in zip(markers, [m[1] for m in tiny.markers] + [[]] * 9)]
            hc = native.HostCase(gen.write_case(d, tiny, inputs), host_wall_distance=False)
            self.params = native.Params.from_buffer_copy(hc.params)
            hc.close()
        self.nvar = self.params.nvar
        self.ncell, self.nnode = len(a["cell_vert"]), len(a["node_xy"])
        self.nface, self.nbface, self.nmark = len(a["face"]), len(a["bface"]), len(markers)
        p = lambda k, t: a[k].ctypes.data_as(C.POINTER(t))   # noqa: E731
        i, d = C.c_int32, C.c_double
        self.mesh = native.MeshDesc(self.ncell, self.nnode, self.nface, self.nbface, self.nmark, 0,
                                    p("node_xy", d), p("cell_vert", i), p("face", i), p("bface", i),
                                    p("bface_mark", i), p("mark_type", i), p("cell_nbr", i), p("cell_face", i), None)


def _connect(nodes, cells, marks):
    """csu_mesh_desc arrays from vertex lists [n, 4] (-1 pads triangles;
    counter-clockwise) and boundary edges per marker."""
    n, npt = len(cells), len(nodes)
    tri = cells[:, 3] < 0
    nxt = np.stack([cells[:, 1], cells[:, 2], np.where(tri, cells[:, 0], cells[:, 3]), cells[:, 0]], axis=1)
    m = cells >= 0
    cell = np.broadcast_to(np.arange(n)[:, None], (n, 4))[m]
    p0, p1 = cells[m].astype(np.int64), nxt[m].astype(np.int64)
    key = np.minimum(p0, p1) * npt + np.maximum(p0, p1)
    o = np.argsort(key, kind="stable")
    ks = key[o]
    first = np.flatnonzero(ks[1:] == ks[:-1])
    a, b = o[first], o[first + 1]                  # the two directed edges of a face, lower cell first
    seq = np.argsort(a, kind="stable")
    a, b = a[seq], b[seq]
    face = np.stack([cell[a], cell[b], p0[a], p1[a]], axis=1).astype(np.int32)
    nf = len(face)
    nbr = np.full((n, 4), np.iinfo(np.int32).max, np.int32)
    cfc = np.zeros((n, 4), np.int32)
    # slots: interior faces in face order, then boundary faces in marker order
    be = np.concatenate([np.asarray(e, np.int64).reshape(-1, 2) for e in marks])
    bm = np.concatenate([np.full(len(e), k, np.int32) for k, e in enumerate(marks)])
    bkey = np.minimum(be[:, 0], be[:, 1]) * npt + np.maximum(be[:, 0], be[:, 1])
    bd = o[np.searchsorted(ks, bkey)]
    bface = np.stack([cell[bd], p0[bd], p1[bd]], axis=1).astype(np.int32)
    own = np.concatenate([face[:, 0], face[:, 1], bface[:, 0]])
    rank = np.concatenate([np.arange(nf), np.arange(nf), nf + np.arange(len(be))])
    other = np.concatenate([face[:, 1], face[:, 0], -1 - np.arange(len(be))])
    sgn = np.concatenate([np.arange(nf) + 1, -(np.arange(nf) + 1), np.zeros(len(be), np.int64)])
    q = np.lexsort((rank, own))
    start = np.searchsorted(own[q], np.arange(n))
    slot = np.arange(len(q)) - start[own[q]]
    nbr[own[q], slot] = other[q]
    cfc[own[q], slot] = sgn[q]
    return {"node_xy": np.ascontiguousarray(nodes, dtype=np.float64), "cell_vert": np.ascontiguousarray(cells, np.int32),
            "face": face, "bface": bface, "bface_mark": bm, "cell_nbr": nbr, "cell_face": cfc}


def _cells4(mesh):
    return np.array([list(c) + [-1] * (4 - len(c)) for c in mesh.cells], np.int64)


def _ramp_arrays(nx, ny, split, seed=0, angle=15.0, x_ramp=0.3, height=0.5, jitter=0.1):
    """gen.ramp_mesh's compression ramp, without its per-node loops."""
    rng = np.random.default_rng(seed)
    x = np.linspace(0.0, 1.0, nx + 1)
    yw = np.maximum(0.0, x - x_ramp) * math.tan(math.radians(angle))
    X = np.repeat(x[:, None], ny + 1, axis=1)
    Y = yw[:, None] + (height - yw)[:, None] * np.linspace(0.0, 1.0, ny + 1)
    dy = (Y[:, 2:] - Y[:, :-2])[1:-1] * 0.5
    X[1:-1, 1:-1] += rng.uniform(-jitter, jitter, (nx - 1, ny - 1)) / nx
    Y[1:-1, 1:-1] += rng.uniform(-jitter, jitter, (nx - 1, ny - 1)) * dy
    nid = np.arange((nx + 1) * (ny + 1)).reshape(nx + 1, ny + 1)
    a, b, c, d = nid[:-1, :-1].ravel(), nid[1:, :-1].ravel(), nid[1:, 1:].ravel(), nid[:-1, 1:].ravel()
    if split:
        none = np.full_like(a, -1)
        cells = np.stack([np.stack([a, b, c, none], 1), np.stack([a, c, d, none], 1)], 1).reshape(-1, 4)
    else:
        cells = np.stack([a, b, c, d], 1)
    pairs = lambda p, q: np.stack([p, q], 1)   # noqa: E731
    markers = [("inlet", pairs(nid[0, 1:], nid[0, :-1])), ("outlet", pairs(nid[-1, :-1], nid[-1, 1:])),
               ("ramp", pairs(nid[:-1, 0], nid[1:, 0])), ("top", pairs(nid[1:, -1], nid[:-1, -1]))]
    return np.stack([X.ravel(), Y.ravel()], 1), cells, markers


@functools.lru_cache(maxsize=3)
def _ramp(nx, ny, split, morton, flux, precision):
    nodes, cells, markers = _ramp_arrays(nx, ny, split)
    if morton:
        cells = cells[renumber.morton_order(nodes, cells)]
    return MeshCase(nodes, cells, markers, gen.ramp_input(threads=1, nmax=CHUNK, flux=flux, precision=precision))


@functools.lru_cache(maxsize=3)
def _ramp_group(ny, solves, scheme, precision):
    """Unlike ramps around 4 ny^2 cells each: sizes and Mach numbers spread."""
    out = []
    for k in range(solves):
        h = max(6, int(round(ny * (0.6 + 0.8 * k / max(1, solves - 1)))))
        nodes, cells, markers = _ramp_arrays(2 * h + k % 3, h, True, seed=k)
        over = {"mach": f"{2.4 + 0.8 * k / max(1, solves - 1):.3f}"}
        if scheme == "LUSGS":
            cells = cells[renumber.colour_order(cells)]
            over |= {"timeScheme": "LUSGS", "CFL": "5"}
        out.append(MeshCase(nodes, cells, markers, gen.ramp_input(threads=1, nmax=CHUNK, precision=precision, **over)))
    return out


@functools.lru_cache(maxsize=3)
def _plate(nx, ny, scheme, precision):
    m = gen.plate_mesh(nx=nx, ny=ny, growth=1.08, tri_frac=0.2, seed=1)
    over = {"timeScheme": "DPLUR", "CFL": 50} if scheme == "DPLUR" else {}
    return MeshCase(m.nodes, _cells4(m), m.markers, gen.plate_input(threads=1, nmax=CHUNK, precision=precision, **over))


@functools.lru_cache(maxsize=3)
def _naca(ni, nfar, model, flux, precision, colour=True):
    m = gen.naca_mesh(ni=ni, nwall=40, nfar=nfar, seed=2)
    cells = _cells4(m)
    x, y = m.nodes[cells.clip(0), 0], m.nodes[cells.clip(0), 1]
    q = cells[:, 3] >= 0
    x3, y3 = np.where(q, x[:, 3], x[:, 0]), np.where(q, y[:, 3], y[:, 0])
    area = sum(u0 * v1 - u1 * v0 for u0, v0, u1, v1 in ((x[:, 0], y[:, 0], x[:, 1], y[:, 1]),
                                                       (x[:, 1], y[:, 1], x[:, 2], y[:, 2]),
                                                       (x[:, 2], y[:, 2], x3, y3), (x3, y3, x[:, 0], y[:, 0])))
    flip = area < 0                                   # the host reader's orientation fix
    t, f = flip & ~q, flip & q
    cells[t, :3] = cells[t, 2::-1]
    cells[f] = cells[f, ::-1]
    if colour:
        cells = cells[renumber.colour_order(cells)]
    over = {"sa": "1"} if model == "sa" else {"sa": "0", "sst": "1"}
    return MeshCase(m.nodes, cells, m.markers,
                    gen.naca_input(threads=1, nmax=CHUNK, aoa=2.6, flux=flux, precision=precision, **over))


@functools.lru_cache(maxsize=2)
def _tube(nx, ny):
    m = gen.tube_mesh(nx=nx, ny=ny, seed=0)
    return MeshCase(m.nodes, _cells4(m), m.markers, gen.tube_input(threads=1))


def _case_of(c):
    k = c["kind"]
    if k in ("residual", "rk"):
        return _ramp(c["nx"], c["ny"], c["split"], c["morton"], c["flux"], c["precision"])
    if k == "plate":
        return _plate(c["nx"], c["ny"], c["scheme"], c["precision"])
    if k == "naca":
        return _naca(c["ni"], c["nfar"], c["model"], c["flux"], c["precision"])
    if k == "tube":
        return _tube(c["nx"], c["ny"])
    return _naca(c["ni"], c["nfar"], "sa", "ROE", 0, False)


# ---------------------------------------------------------------------------
# states
# ---------------------------------------------------------------------------
def _centres(a):
    v = a["cell_vert"]
    m = v >= 0
    xy = a["node_xy"][v.clip(0)] * m[..., None]
    return xy.sum(1) / m.sum(1)[:, None]


def _state(mc, seed, smooth=0.03, rough=1e-3):
    """The free stream with a smooth disturbance (a few random waves) and a
    little cell-to-cell noise, as a run in progress holds."""
    rng = np.random.default_rng(seed)
    p = mc.params
    c = _centres(mc.a)
    c = (c - c.min(0)) / np.maximum(np.ptp(c, 0), 1e-300)
    w = rough * rng.standard_normal((4, len(c)))
    for _ in range(4):
        kx, ky, ph = rng.uniform(1, 9), rng.uniform(1, 9), rng.uniform(0, 7)
        w += smooth / 3 * rng.uniform(-1, 1, (4, 1)) * np.sin(2 * math.pi * (kx * c[:, 0] + ky * c[:, 1]) + ph)
    r, u, v, pr = p.pin[0], p.pin[1], p.pin[2], p.pin[3]
    speed = math.hypot(u, v)
    r, u, v, pr = r * (1 + w[0]), u + speed * w[1], v + speed * w[2], pr * (1 + w[3] * min(1.0, p.mach_inf))
    k = p.pin[5] if p.sst else 0.0
    U = [r, r * u, r * v, pr / (p.gamma - 1) + 0.5 * r * (u * u + v * v) + r * k]
    for q in range(4, p.nvar):
        U.append(r * p.pin[q + 1])
    return np.ascontiguousarray(U)


def _tube_state(mc, seed):
    rng = np.random.default_rng(seed)
    left = _centres(mc.a)[:, 0] < 25.0
    f = 1 + 0.05 * rng.uniform(-1, 1, 4)
    p = np.where(left, 1e5 * f[0], 1e4 * f[1])
    t = np.where(left, 300.0 * f[2], 240.0 * f[3])
    r = p / (mc.params.gas_r * t)
    z = np.zeros_like(p)
    return np.ascontiguousarray([r, z, z, p / (mc.params.gamma - 1)])


def prepare(case, seed):
    k = case["kind"]
    if k == "walldist":
        base = _case_of(case)                     # an airfoil scaled and shifted: other coordinates, same cells
        rng = np.random.default_rng(seed)
        mc = MeshCase.__new__(MeshCase)
        mc.__dict__.update(base.__dict__)
        xy = base.a["node_xy"] * rng.uniform(0.7, 1.4) + rng.uniform(-1, 1, 2)
        mc.a = dict(base.a, node_xy=np.ascontiguousarray(xy))
        mc.mesh = native.MeshDesc.from_buffer_copy(base.mesh)
        mc.mesh.node_xy = mc.a["node_xy"].ctypes.data_as(C.POINTER(C.c_double))
        return {"kind": k, "case": mc}
    if k in ("served", "batch"):
        group = _ramp_group(case["ny"], case["solves"], "LUSGS" if k == "served" else "RK", case.get("precision", 0))
        b = native.Batch(group)
        U = [_state(m, seed * 64 + q) for q, m in enumerate(group)]
        for q, u in enumerate(U):
            b.set_state(q, u)
        return {"kind": k, "batch": b, "U": U, "cap": case.get("cap")}
    mc = _case_of(case)
    dev = native.Device(mc)
    U = _tube_state(mc, seed) if k == "tube" else _state(mc, seed)
    dev.set_state(U)
    return {"kind": k, "dev": dev, "U": U, "tmax": case.get("tmax"),
            "n": _chunk(case)}


def run(s):
    k = s["kind"]
    if k == "walldist":
        return native.wall_distance_dev(s["case"])
    if k == "residual":
        return s["dev"].residual()
    if k == "tube":
        s["dev"].set_state(s["U"])
        t, n, done = s["dev"].advance_time(s["tmax"])
        return {"t": t, "steps": n, "done": done, "U": s["dev"].get_state()}
    if k == "batch":
        b = s["batch"]
        res, coef = b.iterate(CHUNK)
        return {"res": res, "coef": coef, "U": [b.get_state(q) for q in range(b.n)]}
    if k == "served":
        b = s["batch"]
        for q in range(b.n):                       # new solves enter the batch
            b.set_active(q, True)
            b.set_state(q, s["U"][q])
        r = b.run(drop=1e-8, max_iter=s["cap"], chunk=CHUNK)
        return {"iters": [x["iters"] for x in r], "converged": [x["converged"] for x in r],
                "res": [x["res_last"] for x in r], "coef": np.array([x["coef_last"] for x in r]),
                "U": [b.get_state(q) for q in range(b.n)]}
    res, coef = s["dev"].iterate(s["n"])
    return {"res": res, "coef": coef, "U": s["dev"].get_state()}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _cells_of(case):
    k = case["kind"]
    if k in ("residual", "rk"):
        return case["nx"] * case["ny"] * (2 if case["split"] else 1)
    if k == "plate":
        return int(case["nx"] * case["ny"] * 1.12)
    if k == "tube":
        return case["nx"] * case["ny"] * 2
    if k in ("served", "batch"):
        n = 0
        for q in range(case["solves"]):
            h = max(6, int(round(case["ny"] * (0.6 + 0.8 * q / max(1, case["solves"] - 1)))))
            n += 2 * h * (2 * h + q % 3)
        return n
    return case["ni"] * (40 + 2 * case["nfar"])


def work(case):
    """Bytes: the state read and written once per stage or sweep, the stage's
    start state, the time step, and the mesh (vertex and neighbour ids, node
    coordinates: 32 B per cell) once per stage; FP64 operations from the
    formulas."""
    n, k = _cells_of(case), case["kind"]
    if k == "walldist":
        return {"bytes": 8.0 * 3 * n, "flops": 25.0 * n * case["ni"]}
    if k == "residual":
        return {"bytes": n * (32 + 32 + 3 * 32 + 40 + 32.0), "flops": 900.0 * n}
    if k == "plate" and case["scheme"] == "DPLUR":
        # residual, the four 4x4 blocks written and read once, 20 sweeps of
        # the increment
        return {"bytes": CHUNK * n * (96 + 32 + 2 * 512 + 20 * 64.0),
                "flops": CHUNK * n * (1500 + 20 * 140.0)}
    if k in ("naca", "served"):
        nv = 4 if k == "served" else 5 if case["model"] == "sa" else 6
        it = case["cap"] if k == "served" else CHUNK
        return {"bytes": it * n * (8.0 * nv * 7 + 64), "flops": it * n * (1100 + 250.0 * nv)}
    it = 5 * (_chunk(case) if k != "tube" else 0.175 * case["nx"])   # the tube's steps go with its resolution
    return {"bytes": it * n * (96 + 8 + 32.0), "flops": it * n * (900.0 if k != "plate" else 1500.0)}


# ---------------------------------------------------------------------------
# the inviscid path in plain numpy, FP64
# ---------------------------------------------------------------------------
class _Np:
    """Second-order inviscid residual, RK5 and LU-SGS of one mesh: least
    squares, the Venkatakrishnan limiter, Roe / AUSM / AUSMDV, weak walls."""

    RK5 = (0.0533, 0.1263, 0.2375, 0.4414, 1.0)

    def __init__(self, mc):
        a, p = mc.a, mc.params
        self.p, self.g, self.R = p, p.gamma, p.gas_r
        self.Cv = self.g * self.R / (self.g - 1) - self.R
        xy, v, face, bf = a["node_xy"], a["cell_vert"], a["face"], a["bface"]
        n = len(v)
        tri = v[:, 3] < 0
        self.np = np.where(tri, 3, 4)
        self.c = _centres(a)
        x, y = xy[v.clip(0), 0], xy[v.clip(0), 1]
        ta = lambda i, j, k: 0.5 * ((x[:, i] - x[:, j]) * (y[:, i] + y[:, j]) + (x[:, j] - x[:, k]) *   # noqa: E731
                                    (y[:, j] + y[:, k]) + (x[:, k] - x[:, i]) * (y[:, k] + y[:, i]))
        self.om = ta(0, 1, 2) + np.where(tri, 0.0, ta(2, 3, 0))
        nxt = np.stack([v[:, 1], v[:, 2], np.where(tri, v[:, 0], v[:, 3]), v[:, 0]], 1)
        self.edge = v >= 0
        d = xy[nxt.clip(0)] - xy[v.clip(0)]
        self.sx = 0.5 * np.where(self.edge, np.abs(d[..., 1]), 0).sum(1)
        self.sy = 0.5 * np.where(self.edge, np.abs(d[..., 0]), 0).sum(1)
        self.off = 0.5 * (xy[nxt.clip(0)] + xy[v.clip(0)]) - self.c[:, None]
        self.e0, self.e1 = face[:, 0], face[:, 1]
        seg = xy[face[:, 3]] - xy[face[:, 2]]
        self.fs = np.stack([seg[:, 1], -seg[:, 0]])
        self.fl = np.hypot(*self.fs)

        def edge_no(cell, p0, p1):
            j = np.zeros(len(cell), int)
            for q in range(4):
                hit = ((v[cell, q] == p0) & (nxt[cell, q] == p1)) | ((v[cell, q] == p1) & (nxt[cell, q] == p0))
                j[hit & self.edge[cell, q]] = q
            return j
        self.s0, self.s1 = edge_no(self.e0, face[:, 2], face[:, 3]), edge_no(self.e1, face[:, 2], face[:, 3])
        self.be, self.bt = bf[:, 0], a["mark_type"][a["bface_mark"]]
        seg = xy[bf[:, 2]] - xy[bf[:, 1]]
        self.bs = np.stack([seg[:, 1], -seg[:, 0]])
        self.bl = np.hypot(*self.bs)
        bm = 0.5 * (xy[bf[:, 1]] + xy[bf[:, 2]])
        nb = a["cell_nbr"]
        self.has = np.arange(4) < self.np[:, None]
        self.nb = np.where(self.has, np.where(nb >= 0, nb, n - 1 - nb), np.arange(n)[:, None])   # ghosts after the cells
        dr = np.concatenate([self.c, bm])[self.nb] - self.c[:, None]
        dx, dy = dr[..., 0], dr[..., 1]
        A, B, D = (dx * dx).sum(1), (dx * dy).sum(1), (dy * dy).sum(1)
        det = (A * D - B * B)[:, None]
        self.wx, self.wy = (D[:, None] * dx - B[:, None] * dy) / det, (A[:, None] * dy - B[:, None] * dx) / det
        pin = np.array(p.pin[:4])
        q2 = pin[1] ** 2 + pin[2] ** 2
        self.ee = np.array([pin[0] ** 2, q2, q2, pin[3] ** 2])[:, None] * (p.lim_k * np.sqrt(self.om / self.om.max())) ** 3

    def prim(self, U):
        """Primitives r u v p; U clamped in place where the state leaves the
        physical range."""
        r = U[0] = np.maximum(U[0], self.p.rlim)
        u, v = U[1] / r, U[2] / r
        T = np.maximum(U[3] / r - 0.5 * (u * u + v * v), 717.6325) / self.Cv
        cold = T < 1
        T = np.where(cold, 1.0, T)
        U[3] = np.where(cold, (self.Cv * T + 0.5 * (u * u + v * v)) * r, U[3])
        return np.stack([r, u, v, self.R * T * r])

    def rot(self, P, s, l):
        return np.stack([P[0], (P[1] * s[0] + P[2] * s[1]) / l, (P[2] * s[0] - P[1] * s[1]) / l, P[3]])

    def flux(self, L, R):
        g = self.g
        (rL, uL, vL, pL), (rR, uR, vR, pR) = L, R
        if self.p.flux == 0:
            UL = np.stack([rL, rL * uL, rL * vL, pL / (g - 1) + 0.5 * rL * (uL * uL + vL * vL)])
            UR = np.stack([rR, rR * uR, rR * vR, pR / (g - 1) + 0.5 * rR * (uR * uR + vR * vR)])
            HL, HR = (UL[3] + pL) / rL, (UR[3] + pR) / rR
            a, b = np.sqrt(rL), np.sqrt(rR)
            u, v, H = (a * uL + b * uR) / (a + b), (a * vL + b * vR) / (a + b), (a * HL + b * HR) / (a + b)
            q = u * u + v * v
            c = np.sqrt((g - 1) * (H - 0.5 * q))
            d = UR - UL
            a4 = ((H - q) * d[0] + u * d[1] + v * d[2] - d[3]) * (g - 1) / (c * c)
            a2 = d[2] - d[0] * v
            a5, a1 = 0.5 * (d[0] - a4 + (d[1] - u * d[0]) / c), 0.5 * (d[0] - a4 - (d[1] - u * d[0]) / c)

            def fix(l):
                e = self.p.efix
                return np.abs(np.where(np.abs(l) < e, 0.5 * (l * l / e + e), l))
            l1, l2, l5 = fix(u - c), fix(u), fix(u + c)
            one, z = np.ones_like(u), np.zeros_like(u)
            FL = np.stack([UL[1], UL[1] * uL + pL, UL[1] * vL, uL * (UL[3] + pL)])
            FR = np.stack([UR[1], UR[1] * uR + pR, UR[1] * vR, uR * (UR[3] + pR)])
            return 0.5 * (FL + FR - a1 * l1 * np.stack([one, u - c, v, H - u * c]) - a2 * l2 * np.stack([z, z, one, v]) -
                          a4 * l2 * np.stack([one, u, v, 0.5 * q]) - a5 * l5 * np.stack([one, u + c, v, H + u * c]))
        HL = g / (g - 1) * pL / rL + 0.5 * (uL * uL + vL * vL)
        HR = g / (g - 1) * pR / rR + 0.5 * (uR * uR + vR * vR)
        cL, cR = np.sqrt(g * pL / rL), np.sqrt(g * pR / rR)
        psL, psR = np.stack([np.ones_like(uL), uL, vL, HL]), np.stack([np.ones_like(uR), uR, vR, HR])
        if self.p.flux == 1:
            def split(M, sg):
                sup, q = np.abs(M) >= 1, 0.25 * (M + sg) ** 2
                Ms = np.where(sup, 0.5 * (M + sg * np.abs(M)), sg * q)
                with np.errstate(all="ignore"):
                    return Ms, np.where(sup, Ms / M, q * (2 - sg * M))
            Mp, Pp = split(uL / cL, 1.0)
            Mm, Pm = split(uR / cR, -1.0)
            M = Mp + Mm
            F = np.where(M > 0, rL * cL * M * psL, rR * cR * M * psR)
            F[1] += Pp * pL + Pm * pR
            return F
        cm = np.maximum(cL, cR)
        aL, aR = 2 * (pL / rL) / (pL / rL + pR / rR), 2 * (pR / rR) / (pL / rL + pR / rR)

        def dv(u, p, al, sg):
            sub, h = np.abs(u) < cm, 0.5 * (u + sg * np.abs(u))
            with np.errstate(all="ignore"):
                return (np.where(sub, al * (sg * 0.25 * (u + sg * cm) ** 2 / cm - h) + h, h),
                        np.where(sub, 0.25 * p * (u + sg * cm) ** 2 * (2 - sg * u / cm) / (cm * cm), p * h / u))
        up, pp = dv(uL, pL, aL, 1.0)
        um, pm = dv(uR, pR, aR, -1.0)
        m = up * rL + um * rR
        F = 0.5 * (m * (psR + psL) - np.abs(m) * (psR - psL))
        s = 0.5 * np.minimum(1, 10 * np.abs(pR - pL) / np.minimum(pL, pR))
        F[1] = pp + pm + (0.5 + s) * (up * rL * uL + um * rR * uR) + (0.5 - s) * F[1]
        A, B = (uL - cL < 0) & (uR - cR > 0), (uL + cL < 0) & (uR + cR > 0)
        k = np.where(A & ~B, 0.125 * ((uR - cR) - (uL - cL)), 0) + np.where(B & ~A, 0.125 * ((uR + cR) - (uL + cL)), 0)
        return F - k * (rR * psR - rL * psL)

    def ghosts(self, P):
        """Ghost states and boundary fluxes (times length)."""
        p, t = self.p, self.bt
        Pi = P[:, self.be]
        n = self.bs / self.bl
        r, u, v, q = Pi
        c = np.sqrt(self.g * q / r)
        un = n[0] * u + n[1] * v
        wall = np.stack([r + r * un / c, u - n[0] * un, v - n[1] * un, q + r * c * un])
        sub = np.hypot(u, v) < c
        pa = np.array(p.pin[:4])[:, None] * np.ones_like(r)
        pb = 0.5 * (pa[3] + q - r * c * (n[0] * (pa[1] - u) + n[1] * (pa[2] - v)))
        k = (pa[3] - pb) / (r * c)
        inl = np.where(sub, np.stack([pa[0] + (pb - pa[3]) / (c * c), pa[1] - n[0] * k, pa[2] - n[1] * k, pb]), pa)
        k = (q - p.pout) / (r * c)
        out = np.where(sub, np.stack([r + (p.pout - q) / (c * c), u + n[0] * k, v + n[1] * k, p.pout + 0 * q]), Pi)
        rp = self.rot(Pi, self.bs, self.bl)
        sym = np.stack([r, -n[1] * rp[2], n[0] * rp[2], q])
        G = np.select([t == 0, t == 1, t == 2], [sym, inl, out], wall)
        mir = rp * np.array([1, -1, 1, 1.0])[:, None]
        F = self.flux(rp, np.where(t == 0, mir, self.rot(G, self.bs, self.bl)))
        w = self.rot(wall, self.bs, self.bl)
        H = self.g / (self.g - 1) * w[3] / w[0] + 0.5 * (w[1] ** 2 + w[2] ** 2)
        Fw = w[0] * w[1] * np.stack([np.ones_like(H), w[1], w[2], H])
        Fw[1] += w[3]
        return G, self.back(np.where(t == 3, Fw, F), self.bs)

    @staticmethod
    def back(F, s):
        l = np.hypot(*s)
        return np.stack([F[0] * l, F[1] * s[0] - F[2] * s[1], F[1] * s[1] + F[2] * s[0], F[3] * l])

    def residual(self, P, fields=False):
        G, Fb = self.ghosts(P)
        if self.p.order == 1:
            self.G = G
            return self.gather(P[:, self.e0], P[:, self.e1], Fb)
        d = np.concatenate([P, G], axis=1)[:, self.nb] - P[:, :, None]
        gx, gy = (self.wx * d).sum(2), (self.wy * d).sum(2)
        hi, lo = np.maximum(d.max(2), 0)[..., None], np.minimum(d.min(2), 0)[..., None]
        d2 = gx[..., None] * self.off[..., 0] + gy[..., None] * self.off[..., 1]
        d1 = np.where(d2 > 0, hi, lo)
        e = self.ee[..., None]
        with np.errstate(all="ignore"):
            ph = (d1 * d1 + e + 2 * d1 * d2) / (d1 * d1 + 2 * d2 * d2 + d1 * d2 + e)
        ph = np.where((d2 == 0) | ~self.edge, np.where(self.edge, 1.0, np.inf), ph).min(2)
        rec = P[:, :, None] + ph[..., None] * d2
        R = self.gather(rec[:, self.e0, self.s0], rec[:, self.e1, self.s1], Fb)
        self.G = G
        return (R, gx, gy, ph) if fields else R

    def gather(self, L, R, Fb):
        F = self.back(self.flux(self.rot(L, self.fs, self.fl), self.rot(R, self.fs, self.fl)), self.fs)
        n = len(self.c)
        return np.stack([np.bincount(self.e0, f, n) - np.bincount(self.e1, f, n) + np.bincount(self.be, b, n)
                         for f, b in zip(F, Fb)])

    def local_dt(self, U):
        u, v = U[1] / U[0], U[2] / U[0]
        c = np.sqrt(self.g * self.R * (U[3] / U[0] - 0.5 * (u * u + v * v)) / self.Cv)
        return self.om / ((np.abs(u) + c) * self.sx + (np.abs(v) + c) * self.sy)

    def norms(self, R):
        p = self.p
        q = 0.5 * p.pin[0] * (p.pin[1] ** 2 + p.pin[2] ** 2)
        w = self.bt >= 3
        with np.errstate(all="ignore"):
            f = ((self.G[3] - p.pin[3]) / q * self.bs)[:, w].sum(1) / p.sref
        return np.sqrt((R * R).mean(1)), [f[0], 0.0, f[1], 0.0]

    def rk(self, U, dt):
        U0 = None
        V = U
        for a in self.RK5:
            P = self.prim(V)
            U0 = V.copy() if U0 is None else U0
            R = self.residual(P)
            V = U0 - dt * 2.5 * a * R / self.om
        return V, R

    def levels(self):
        """Cells grouped by dependency level of the forward and the backward sweep."""
        n = len(self.c)
        inn = self.has & (self.nb < n)
        out = []
        for up in (False, True):
            dep = inn & ((self.nb > np.arange(n)[:, None]) if up else (self.nb < np.arange(n)[:, None]))
            lev = np.zeros(n, int)
            while True:
                new = np.where(dep, lev[self.nb % n] + 1, 0).max(1)
                if (new == lev).all():
                    break
                lev = new
            out.append([(np.flatnonzero(lev == l), dep) for l in range(lev.max() + 1)])
        return out

    def lusgs(self, U, lev, cfl):
        P = self.prim(U)
        R = self.residual(P)
        n = len(self.c)
        s = self.slot_s
        T = P[3] / (self.R * P[0])
        nn = self.nb % n
        inn = self.has & (self.nb < n)
        l = np.where(self.has, np.hypot(*s), 1.0)
        nx, ny = s[0] / l, s[1] / l
        m = lambda z: np.where(inn, 0.5 * (z[:, None] + z[nn]), z[:, None])   # noqa: E731
        lam = np.where(self.has, (np.abs(nx * m(P[1]) + ny * m(P[2])) + np.sqrt(self.g * self.R * m(T))) * l, 0).sum(1)
        D = 0.5 * self.p.wimp * lam
        D = D + self.om / (cfl * (self.om / lam).min())
        c = np.sqrt(self.g * self.R * T)

        def sweep(start, groups):
            W = np.zeros_like(R)
            for cells, dep in groups:
                acc = start[:, cells].copy()
                for q in range(4):
                    on = dep[cells, q]
                    j = np.where(on, nn[cells, q], 0)
                    a, b, ds = nx[cells, q], ny[cells, q], l[cells, q]
                    d = W[:, j]
                    r, u, v, pr = P[:, j]
                    E = self.Cv * T[j] + 0.5 * (u * u + v * v)
                    V = np.stack([r, r * u, r * v, r * E])
                    X = V + d
                    ux, vx = X[1] / X[0], X[2] / X[0]
                    T2 = T[j] + (X[3] / X[0] - 0.5 * (ux * ux + vx * vx) - self.Cv * T[j]) / self.Cv
                    p2 = self.R * T2 * X[0]

                    def f(Z, pz):
                        w = (a * Z[1] + b * Z[2]) / Z[0]
                        return np.stack([Z[0] * w, Z[1] * w + a * pz, Z[2] * w + b * pz, (Z[3] + pz) * w])
                    ra = self.p.wimp * (np.abs(a * u + b * v) + c[j]) * ds
                    acc -= np.where(on, 0.5 * ((f(X, p2) - f(V, pr)) * ds - ra * d), 0)
                W[:, cells] = acc / D[cells]
            return W
        W = sweep(-R, lev[0])
        U += sweep(D * W, lev[1])
        return U, R

    def slots(self, a):
        """Outward face vectors per neighbour slot."""
        n = len(self.c)
        s = np.zeros((2, n, 4))
        for q in range(4):
            f, b = a["cell_face"][:, q], a["cell_nbr"][:, q]
            i = f != 0
            s[:, i, q] = np.sign(f[i]) * self.fs[:, np.abs(f[i]) - 1]
            i = (f == 0) & (b < 0)
            s[:, i, q] = self.bs[:, -1 - b[i]]
        self.slot_s = s


def _exact_wall(a):
    xy, c = a["node_xy"], _centres(a)
    w = a["mark_type"][a["bface_mark"]] >= 3
    p, q = xy[a["bface"][w, 1]], xy[a["bface"][w, 2]]
    best = np.full(len(c), 1e12)
    for k in range(len(p)):
        e = q[k] - p[k]
        t = np.clip(((c - p[k]) @ e) / (e @ e), 0, 1)
        d = p[k] + t[:, None] * e - c
        np.minimum(best, d[:, 0] ** 2 + d[:, 1] ** 2, out=best)
    return np.minimum(np.sqrt(best), 1e6)


def exact(case, seed):
    """Plain numpy for the inviscid cases and the wall distance.  The viscous
    cases, and inviscid ones of more cell-stages than numpy does in about
    twenty seconds, have None."""
    k = case["kind"]
    if k == "walldist":
        if _cells_of(case) * case["ni"] > 3e8:
            return None
        return _exact_wall(prepare(case, seed)["case"].a)
    if k in ("plate", "naca"):
        return None
    stages = {"residual": 1, "rk": _chunk(case) * 5, "batch": CHUNK * 5, "tube": 0.5 * case.get("nx", 0),
              "served": 2.0 * case.get("cap", 0)}[k]
    if _cells_of(case) * stages > 7e6:
        return None
    if k in ("served", "batch"):
        out = {"U": [], "res": [], "coef": []}
        group = _ramp_group(case["ny"], case["solves"], "LUSGS" if k == "served" else "RK", case.get("precision", 0))
        for q, mc in enumerate(group):
            s, U = _Np(mc), _state(mc, seed * 64 + q)
            if k == "batch":
                U, hist = _exact_rk(s, U, CHUNK)
                out["res"].append([h[0] for h in hist])
                out["coef"].append([h[1] for h in hist])
            else:
                s.slots(mc.a)
                lev = s.levels()
                for _ in range(case["cap"]):
                    U, R = s.lusgs(U, lev, mc.params.cfl)
                r, f = s.norms(R)
                out["res"].append(r[0])
                out["coef"].append(f)
                # a chunk runs to its end
                for _ in range(-case["cap"] % CHUNK):
                    U, R = s.lusgs(U, lev, mc.params.cfl)
            out["U"].append(U)
        if k == "batch":
            return {"res": np.array(out["res"]).transpose(1, 0, 2), "coef": np.array(out["coef"]).transpose(1, 0, 2),
                    "U": out["U"]}
        return {"iters": [None] * len(group), "converged": [None] * len(group), "res": out["res"],
                "coef": np.array(out["coef"]), "U": out["U"]}
    mc = _case_of(case)
    s = _Np(mc)
    if k == "tube":
        U, t, n, tmax = _tube_state(mc, seed), 0.0, 0, case["tmax"]
        for _ in range(5000):
            dt = mc.params.cfl * s.local_dt(U).min()
            last = t + dt > tmax
            dt = tmax - t if last else dt
            U, _ = s.rk(U, dt)
            t, n = t + 2.5 * dt, n + 1
            if last:
                return {"t": t, "steps": n, "done": True, "U": U}
    U = _state(mc, seed)
    if k == "residual":
        P = s.prim(U)
        R, gx, gy, ph = s.residual(P, True)
        T = lambda z: z[3] / (s.R * z[0])   # noqa: E731
        return {"R": R, "dPx": gx, "dPy": gy, "phi": ph, "P": np.column_stack([P.T, T(P)]),
                "Pb": np.column_stack([s.G.T, T(s.G)])}
    U, hist = _exact_rk(s, U, _chunk(case))
    return {"res": np.array([h[0] for h in hist]), "coef": np.array([h[1] for h in hist]), "U": U}


def _exact_rk(s, U, n):
    hist = []
    for _ in range(n):
        U, R = s.rk(U, s.p.cfl * s.local_dt(U))
        hist.append(s.norms(R))
    return U, hist
