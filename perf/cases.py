"""Performance cases of the pair-analysis path.

Each case is one piece of work that a user of the framework has it do, through
the Python API (small and ordinary systems, host arrays in and out, as a freud
script is written) or through the C-ABI with device-resident points (the large
systems, as ``bench.py`` and an embedding C++ program use it).  ``listed()``
holds the cases, ``draw(rng)`` gives further ones of the same ranges,
``prepare``/``run`` set one up and run one pass, and ``exact`` evaluates it in
64 bits without the framework.
"""

import ctypes
import functools
import math

import numpy as np
import torch

import freud_amd
from freud_amd import _lib

DEV = "cuda" if torch.cuda.is_available() else "cpu"
NO_K = 0xFFFFFFFF


def listed():
    return [
        # A script's neighbour search on a small liquid: host points in, the NeighborList's arrays out.
        dict(name="query_4k", kind="query", engine="aabb", n=4096, density=1.0, k=12),
        # The small RDF of the benchmark set: 4096 uniform points in a cube of side 16.
        dict(name="rdf_4k", kind="rdf", n=4096, density=1.0, r_max=4.0, bins=100),
        # Averaged q6 of an ordinary simulation snapshot over the neighbours within r_max.
        dict(name="order_20k", kind="order", n=20000, density=0.9, l=6, r_max=1.5, average=True, wl=False),
        # Partial g(r) between two species: query points that are not the points.
        dict(name="partial_rdf_100k", kind="partial_rdf", n=65000, n_query=35000, density=1.0, r_max=5.0, bins=200),
        # 2D hexagonal crystal: six nearest neighbours and the hexatic order psi_6.
        dict(name="hexatic_250k", kind="hexatic", n=250000, jitter=0.05, k=6),
        # Triclinic liquid stored in random order: ball query and q_l for a list of l.
        dict(name="triclinic_500k", kind="triclinic", n=500000, density=0.85, r_max=2.0, lmax=12),
        # Large jittered FCC frame: one AABBQuery, ball query and 12 nearest neighbours.
        dict(name="neighbors_1m", kind="neighbors", cells=64, sigma=0.05, r_max=1.5, k=12),
        # Large jittered FCC frame: RDF.
        dict(name="rdf_1m", kind="rdf_frame", cells=64, sigma=0.05, r_max=5.0, bins=200),
        # Large jittered FCC frame: q6 with w6, and averaged q6, over a ball NeighborList.
        dict(name="steinhardt_1m", kind="steinhardt", cells=64, sigma=0.05, r_max=1.5, l=6),
        # Parameter-free neighbours of the large frame: SANN and closed RAD over its candidates.
        dict(name="filters_1m", kind="filters", cells=64, sigma=0.05, r_max=1.9),
        # Two-phase box: ball query, then solid-like bonds and clusters.
        dict(name="solidliquid_2m", kind="solidliquid", cells=64, sigma=0.04, r_max=1.5),
        # A trajectory of uneven mixed frames through the batched path.
        dict(name="batch_256", kind="batch", frames=256, n_min=10000, n_max=200000, r_max=1.5, bins=200,
             rdf_r_max=5.0, l=6),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["query", "rdf", "order", "partial_rdf", "hexatic", "triclinic", "neighbors", "rdf_frame",
                       "steinhardt", "filters", "solidliquid", "batch"])
    if kind == "query":
        return dict(kind=kind, engine=rng.choice(["aabb", "aabb", "linkcell"]), n=int(_log(rng, 700, 30000)),
                    density=round(rng.uniform(0.5, 1.1), 3), k=rng.choice([6, 8, 12, 14, 18]))
    if kind == "rdf":
        return dict(kind=kind, n=int(_log(rng, 1500, 60000)), density=round(rng.uniform(0.5, 1.1), 3),
                    r_max=round(rng.uniform(2.0, 4.5), 3), bins=rng.randrange(50, 401))
    if kind == "order":
        return dict(kind=kind, n=int(_log(rng, 1500, 100000)), density=round(rng.uniform(0.6, 1.1), 3),
                    l=rng.choice([4, 6, 8]), r_max=round(rng.uniform(1.6, 2.0), 3), average=rng.random() < 0.5,
                    wl=rng.random() < 0.5)
    if kind == "partial_rdf":
        n = int(_log(rng, 3000, 200000))
        return dict(kind=kind, n=n, n_query=int(n * rng.uniform(0.1, 0.6)), density=round(rng.uniform(0.6, 1.1), 3),
                    r_max=round(rng.uniform(2.5, 5.0), 3), bins=rng.randrange(50, 401))
    if kind == "hexatic":
        return dict(kind=kind, n=int(_log(rng, 8000, 800000)), jitter=round(rng.uniform(0.03, 0.12), 3),
                    k=rng.choice([4, 6, 6]))
    if kind == "triclinic":
        return dict(kind=kind, n=int(_log(rng, 20000, 700000)), density=round(rng.uniform(0.7, 1.0), 3),
                    r_max=round(rng.uniform(1.4, 2.0), 3), lmax=rng.choice([6, 8, 12]))
    cells = int(_log(rng, 14, 64))
    sigma = round(rng.uniform(0.03, 0.08), 3)
    if kind == "neighbors":
        return dict(kind=kind, cells=cells, sigma=sigma, r_max=round(rng.uniform(1.3, 1.9), 3),
                    k=rng.choice([6, 8, 12, 14, 18]))
    if kind == "rdf_frame":
        return dict(kind=kind, cells=cells, sigma=sigma, r_max=round(rng.uniform(3.0, 5.0), 3),
                    bins=rng.randrange(100, 401))
    if kind == "steinhardt":
        return dict(kind=kind, cells=cells, sigma=sigma, r_max=round(rng.uniform(1.4, 1.7), 3),
                    l=rng.choice([4, 6, 6, 8]))
    if kind == "filters":
        return dict(kind=kind, cells=cells, sigma=sigma, r_max=round(rng.uniform(1.7, 1.9), 3))
    if kind == "solidliquid":
        return dict(kind=kind, cells=cells, sigma=sigma, r_max=round(rng.uniform(1.35, 1.5), 3))
    n_min = int(_log(rng, 2000, 20000))
    return dict(kind=kind, frames=int(_log(rng, 8, 128)), n_min=n_min, n_max=int(n_min * _log(rng, 2, 10)),
                r_max=round(rng.uniform(1.3, 1.6), 3), bins=rng.randrange(100, 301),
                rdf_r_max=round(rng.uniform(3.0, 5.0), 3), l=rng.choice([4, 6]))


# ------------------------------------------------------------------ systems
# A box is the tuple (Lx, Ly, Lz, xy, xz, yz, is2D); points are float32 on the
# device, inside the box.


def _gen(seed, stream=0):
    return torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + stream)


def _f32(x):
    return float(np.float32(x))


def _lattice(box):
    lx, ly, lz, xy, xz, yz, two_d = box
    return torch.tensor([[lx, 0, 0], [xy * ly, ly, 0], [xz * lz, yz * lz, 1.0 if two_d else lz]],
                        dtype=torch.float64, device=DEV)


def _place(frac, box):
    """Fractional coordinates (any image) to float32 points inside the box."""
    f = (frac - torch.floor(frac)).clamp_(1e-6, 1 - 1e-6) - 0.5
    if box[6]:
        f[:, 2] = 0
    return (f @ _lattice(box)).to(torch.float32).contiguous()


def _uniform(n, density, g, tilts=(0.0, 0.0, 0.0)):
    side = _f32((n / density) ** (1 / 3))
    box = (side, side, side, *map(_f32, tilts), False)
    return box, _place(torch.rand((n, 3), generator=g, device=DEV, dtype=torch.float64), box)


def _crystal(basis, cells, density, sigma, g, tilts=(0.0, 0.0, 0.0), cells_x=None):
    """cells^3 unit cells (x slowest, basis innermost), Gaussian jitter sigma in units of the lattice constant."""
    m = len(basis)
    a = (m / density) ** (1 / 3)
    ax = torch.arange(cells, device=DEV, dtype=torch.float64)
    grid = torch.cartesian_prod(ax, ax, ax)
    frac = ((grid[:, None, :] + torch.tensor(basis, device=DEV, dtype=torch.float64)[None]) / cells).reshape(-1, 3)
    frac = frac + torch.randn(frac.shape, generator=g, device=DEV, dtype=torch.float64) * (sigma / cells)
    side = _f32(cells * a)
    box = (side, side, side, *map(_f32, tilts), False)
    return box, _place(frac, box)


FCC = [[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]]
BCC = [[0, 0, 0], [0.5, 0.5, 0.5]]


def _hexagonal(n, jitter, g):
    ny = max(4, int(math.sqrt(n / (2 * math.sqrt(3)))))
    nx = max(6, round(n / (2 * ny)))
    x = torch.arange(nx, device=DEV, dtype=torch.float64)
    y = torch.arange(ny, device=DEV, dtype=torch.float64)
    grid = torch.cartesian_prod(x, y)
    pos = torch.stack([grid, grid + 0.5], 1).reshape(-1, 2)
    pos = pos + torch.randn(pos.shape, generator=g, device=DEV, dtype=torch.float64) * torch.tensor(
        [jitter, jitter / math.sqrt(3)], device=DEV, dtype=torch.float64)
    frac = torch.zeros((len(pos), 3), device=DEV, dtype=torch.float64)
    frac[:, 0] = pos[:, 0] / nx
    frac[:, 1] = pos[:, 1] / ny
    box = (_f32(nx), _f32(ny * math.sqrt(3)), 0.0, 0.0, 0.0, 0.0, True)
    return box, _place(frac, box)


def _two_phase(cells, sigma, g):
    """A jittered FCC slab (density 1.05) and as many liquid points (density 0.95), stacked along x."""
    a = (4 / 1.05) ** (1 / 3)
    side = cells * a
    n = 4 * cells ** 3
    lx = side + n / (0.95 * side * side)
    ax = torch.arange(cells, device=DEV, dtype=torch.float64)
    sol = ((torch.cartesian_prod(ax, ax, ax)[:, None] + torch.tensor(FCC, device=DEV, dtype=torch.float64)) * a)
    sol = sol.reshape(-1, 3)
    sol = sol + torch.randn(sol.shape, generator=g, device=DEV, dtype=torch.float64) * (sigma * a)
    ext = torch.tensor([lx, side, side], device=DEV, dtype=torch.float64)
    liq = torch.rand((n, 3), generator=g, device=DEV, dtype=torch.float64)
    liq[:, 0] = (side + liq[:, 0] * (lx - side)) / lx
    box = (_f32(lx), _f32(side), _f32(side), 0.0, 0.0, 0.0, False)
    return box, _place(torch.cat([sol / ext, liq]), box)


def _trajectory(case, seed):
    """Frames of uneven size: liquids and jittered FCC / BCC crystals, half of them in triclinic boxes.
    The sizes belong to the case, the seed gives the positions."""
    r = np.random.default_rng([case["frames"], case["n_min"], case["n_max"]])
    g = _gen(seed, 9)
    out = []
    for _ in range(case["frames"]):
        n = int(math.exp(r.uniform(math.log(case["n_min"]), math.log(case["n_max"]))))
        tilts = r.uniform(-0.3, 0.3, 3) if r.random() < 0.5 else (0.0, 0.0, 0.0)
        which = int(r.integers(3))
        if which == 0:
            out.append(_uniform(n, r.uniform(0.8, 1.0), g, tilts))
        else:
            basis = FCC if which == 1 else BCC
            cells = max(2, round((n / len(basis)) ** (1 / 3)))
            out.append(_crystal(basis, cells, 1.0, r.uniform(0.03, 0.1), g, tilts))
    return out


def _system(case, seed):
    """(box, points, query points or None) of a single-frame case."""
    kind, g = case["kind"], _gen(seed)
    if kind in ("query", "rdf", "order"):
        return (*_uniform(case["n"], case["density"], g), None)
    if kind == "partial_rdf":
        box, both = _uniform(case["n"] + case["n_query"], case["density"], g)
        return box, both[:case["n"]].contiguous(), both[case["n"]:].contiguous()
    if kind == "hexatic":
        return (*_hexagonal(case["n"], case["jitter"], g), None)
    if kind == "triclinic":
        tilts = np.random.default_rng([int(seed), 5]).uniform(-0.3, 0.3, 3)
        return (*_uniform(case["n"], case["density"], g, tilts), None)
    if kind == "solidliquid":
        return (*_two_phase(case["cells"], case["sigma"], g), None)
    return (*_crystal(FCC, case["cells"], 1.0, case["sigma"], g), None)


# ------------------------------------------------------------------ one pass


class _DeviceView:
    """Exposes library-owned device memory to torch without a copy, and keeps its owner alive as long."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": shape, "typestr": typestr, "version": 2}


def _view(state, name, ptr, shape, typestr):
    key = (name, ptr, shape)
    if state["views"].get(name, (None,))[0] != key:
        owner = state["batch"] if "batch" in state else state["lists"]
        t = (torch.as_tensor(_DeviceView(owner, ptr, shape, typestr), device=DEV) if 0 not in shape
             else torch.zeros(shape, device=DEV, dtype=torch.int32 if "i" in typestr else torch.float32))
        state["views"][name] = (key, t)
    return state["views"][name][1]


def _bonds(state, name, nl):
    # the list's buffers up to their capacity: a program reads num_bonds entries of them
    nb = state["capacity"]
    assert int(nl.num_bonds) <= nb, "more bonds than the case makes room for"
    return {"bonds": int(nl.num_bonds), "neighbors": _view(state, name + "n", nl.neighbors, (nb, 2), "<i4"),
            "distances": _view(state, name + "d", nl.distances, (nb,), "<f4"),
            "weights": _view(state, name + "w", nl.weights, (nb,), "<f4"),
            "vectors": _view(state, name + "v", nl.vectors, (nb, 3), "<f4")}


class _Lists:
    """NeighborLists owned by a program that calls the C-ABI, with room for `capacity` bonds each (zeroed), which
    a query that fits reuses; freed with the program."""

    def __init__(self, count, capacity):
        self.lists = [_lib.fa_nlist() for _ in range(count)]
        zeros = torch.zeros(3 * capacity, device=DEV, dtype=torch.float32)
        if DEV == "cuda":
            torch.cuda.synchronize()
        for nl in self.lists:
            z = zeros.data_ptr()
            _lib.check(_lib.lib().fa_nlist_from_arrays(1, 1, z, z, z, z, capacity, ctypes.byref(nl)))

    def __del__(self):
        for nl in self.lists:
            _lib.lib().fa_nlist_free(ctypes.byref(nl))


def _ball(r_max):
    return _lib.fa_query_args(_lib.MODE_BALL, NO_K, r_max, 0.0, -1.0, -1.0, 1)


def _nearest(k):
    return _lib.fa_query_args(_lib.MODE_NEAREST, k, -1.0, 0.0, -1.0, -1.0, 1)


class _Query:
    """A NeighborQuery handle over the state's points, for the duration of a with block."""

    def __init__(self, s):
        self.s, self.h = s, ctypes.c_void_p()

    def __enter__(self):
        s = self.s
        _lib.check(_lib.lib().fa_nq_create(ctypes.byref(s["cbox"]), s["points"].data_ptr(), s["n"], _lib.NQ_AABB, 0.0,
                                           ctypes.byref(self.h)))
        return self

    def __call__(self, args, nl):
        s = self.s
        _lib.check(_lib.lib().fa_query(self.h, s["points"].data_ptr(), s["n"], ctypes.byref(args), 0,
                                       ctypes.byref(nl)))

    def __exit__(self, *exc):
        _lib.lib().fa_nq_destroy(self.h)


def prepare(case, seed):
    _lib.init()
    kind = case["kind"]
    if kind == "batch":
        frames = _trajectory(case, seed)
        host = [(freud_amd.Box(*b[:6], is2D=b[6]), p.cpu().numpy()) for b, p in frames]
        batch = freud_amd.batch.TrajectoryBatch(host, ball_r_max=case["r_max"], rdf_bins=case["bins"],
                                                rdf_r_max=case["rdf_r_max"], l=case["l"])
        return {"case": case, "batch": batch, "views": {}, "total": sum(len(p) for _, p in host)}
    box, points, query = _system(case, seed)
    n = len(points)
    s = {"case": case, "box": freud_amd.Box(*box[:6], is2D=box[6]), "n": n, "views": {}}
    s["cbox"] = _lib.make_box(s["box"])
    if kind in ("query", "rdf", "order", "partial_rdf"):
        s["points"] = points.cpu().numpy()
        if query is not None:
            s["query_points"] = query.cpu().numpy()
        return s
    s["points"] = points
    if kind != "rdf_frame":
        s["capacity"] = _capacity(case)
        lists = s["lists"] = _Lists({"neighbors": 2, "filters": 3}.get(kind, 1), s["capacity"])

    def empty(*shape, dtype=torch.float32):
        return torch.empty(shape, device=DEV, dtype=dtype)

    ls = {"triclinic": list(range(4, case.get("lmax", 0) + 1, 2)), "steinhardt": [case.get("l")],
          "solidliquid": [6]}.get(kind)
    if ls:
        total = sum(2 * l + 1 for l in ls)
        s["ls"] = np.asarray(ls, np.uint32)
        s["qlm"], s["ql"] = empty(n * total, 2), empty(n, len(ls))
        s["order"] = np.zeros(len(ls), np.float32)
    if kind == "steinhardt":
        s["qlmave"], s["qlave"], s["wl"] = empty(n * total, 2), empty(n, 1), empty(n, 1)
        s["order_ave"] = np.zeros(1, np.float32)
    if kind == "rdf_frame":
        s["counts"] = empty(case["bins"], dtype=torch.int32)
    if kind == "hexatic":
        s["psi"] = empty(n, 2)
    if kind == "solidliquid":
        s["connections"], s["cluster"], s["sizes"] = (empty(n, dtype=torch.int32).zero_() for _ in range(3))
        s["qlij"] = empty(s["capacity"]).zero_()
    if kind == "filters":
        s["unfilled"] = [empty(n, dtype=torch.uint8) for _ in range(2)]
    if DEV == "cuda":
        torch.cuda.synchronize()
    if kind in ("steinhardt", "filters"):
        # the list a program already holds
        with _Query(s) as query:
            query(_ball(case["r_max"]), lists.lists[0])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    L, check = _lib.lib(), _lib.check
    if kind == "query":
        cls = {"aabb": freud_amd.AABBQuery, "linkcell": freud_amd.LinkCell}[case["engine"]]
        nq = cls(s["box"], s["points"])
        nl = nq.query(s["points"], dict(mode="nearest", num_neighbors=case["k"], exclude_ii=True)).toNeighborList()
        return {"neighbors": nl[:].view(np.int32), "distances": nl.distances, "vectors": nl.vectors}
    if kind in ("rdf", "partial_rdf"):
        rdf = freud_amd.density.RDF(bins=case["bins"], r_max=case["r_max"])
        rdf.compute((s["box"], s["points"]), query_points=s.get("query_points"))
        return {"counts": rdf.bin_counts.view(np.int32), "rdf": rdf.rdf, "n_r": rdf.n_r}
    if kind == "order":
        st = freud_amd.order.Steinhardt(case["l"], average=case["average"], wl=case["wl"])
        st.compute((s["box"], s["points"]), neighbors=dict(r_max=case["r_max"]))
        return {"particle_order": st.particle_order, "order": st.order}
    if kind == "batch":
        b = s["batch"].compute()
        p, q, h = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        check(L.fa_batch_rdf_counts(b._h, ctypes.byref(p)))
        check(L.fa_batch_ql(b._h, ctypes.byref(q), ctypes.byref(h), None))
        return {"bonds": b.num_bonds.astype(np.int64), "order": b.order,
                "counts": _view(s, "counts", p.value, (case["frames"], case["bins"]), "<i4"),
                "ql": _view(s, "ql", q.value, (s["total"],), "<f4"),
                "qlm": _view(s, "qlm", h.value, (s["total"], 2 * case["l"] + 1, 2), "<f4")}
    n, points = s["n"], s["points"].data_ptr()
    lists = s["lists"].lists if "lists" in s else None
    cbox = ctypes.byref(s["cbox"])

    def steinhardt(flags, order):
        check(L.fa_steinhardt(cbox, points, n, ctypes.byref(lists[0]), s["ls"].ctypes.data, len(s["ls"]), flags,
                              s["qlm"].data_ptr(), s["ql"].data_ptr(),
                              s["qlave"].data_ptr() if flags & _lib.ST_AVERAGE else None,
                              s["qlmave"].data_ptr() if flags & _lib.ST_AVERAGE else None,
                              s["wl"].data_ptr() if flags & _lib.ST_WL else None, order.ctypes.data))

    if kind == "neighbors":
        with _Query(s) as query:
            query(_ball(case["r_max"]), lists[0])
            query(_nearest(case["k"]), lists[1])
        return {"ball": _bonds(s, "ball", lists[0]), "nearest": _bonds(s, "nearest", lists[1])}
    if kind == "rdf_frame":
        check(L.fa_memset(s["counts"].data_ptr(), 0, 4 * case["bins"]))
        with _Query(s) as query:
            check(L.fa_rdf_accumulate_query(query.h, points, n, case["r_max"], 0.0, 1, case["bins"], 0.0,
                                            case["r_max"], s["counts"].data_ptr()))
        return {"counts": s["counts"]}
    if kind == "steinhardt":
        steinhardt(_lib.ST_WL, s["order"])
        steinhardt(_lib.ST_AVERAGE, s["order_ave"])
        return {k: s[k] for k in ("qlm", "ql", "wl", "order", "qlmave", "qlave", "order_ave")}
    if kind == "triclinic":
        with _Query(s) as query:
            query(_ball(case["r_max"]), lists[0])
        steinhardt(0, s["order"])
        return {"bonds": _bonds(s, "ball", lists[0]), "qlm": s["qlm"], "ql": s["ql"], "order": s["order"]}
    if kind == "hexatic":
        with _Query(s) as query:
            query(_nearest(case["k"]), lists[0])
        check(L.fa_hexatic(cbox, points, n, ctypes.byref(lists[0]), case["k"], 0, s["psi"].data_ptr()))
        return {"bonds": _bonds(s, "nearest", lists[0]), "psi": s["psi"]}
    if kind == "filters":
        missing = ctypes.c_uint32()
        check(L.fa_filter_sann(ctypes.byref(lists[0]), ctypes.byref(lists[1]), s["unfilled"][0].data_ptr(),
                               ctypes.byref(missing)))
        check(L.fa_filter_rad(cbox, points, n, points, None, ctypes.byref(lists[0]), 1, ctypes.byref(lists[2]),
                              s["unfilled"][1].data_ptr(), ctypes.byref(missing)))
        return {"sann": _bonds(s, "sann", lists[1]), "rad": _bonds(s, "rad", lists[2]), "unfilled": s["unfilled"]}
    clusters = ctypes.c_uint32()
    with _Query(s) as query:
        query(_ball(case["r_max"]), lists[0])
    check(L.fa_solidliquid(cbox, points, n, ctypes.byref(lists[0]), 6, 0.7, 6, 1, s["qlm"].data_ptr(),
                           s["ql"].data_ptr(), s["qlij"].data_ptr(), s["connections"].data_ptr(),
                           s["cluster"].data_ptr(), s["sizes"].data_ptr(), ctypes.byref(clusters)))
    return {"qlm": s["qlm"], "ql": s["ql"], "qlij": s["qlij"], "connections": s["connections"],
            "cluster": s["cluster"], "sizes": s["sizes"], "clusters": clusters.value}


# ------------------------------------------------------------------ what a pass cannot do without


def _points(case):
    if "cells" in case:
        return 4 * case["cells"] ** 3 * (2 if case["kind"] == "solidliquid" else 1)
    return case["n"]


def _density(case):
    return 1.0 if case["kind"] != "hexatic" and "density" not in case else case.get("density", 2 / math.sqrt(3))


def _capacity(case):
    """Bonds that a list of the case never exceeds (crystals hold less in this range of r_max than a liquid's mean
    and half)."""
    n = _points(case)
    if case["kind"] == "hexatic":
        return (n + 64 * int(math.sqrt(n)) + 64) * case["k"]
    return int(n * max(1.5 * _density(case) * 4.19 * case["r_max"] ** 3, case.get("k", 0)))


def _ylm_flops(ls):
    """Per bond: the direction (14), the Legendre recurrence up to max(l), and the sums over m >= 0 of each l."""
    top = max(ls)
    return 14 + 10 * top + 2 * top * (top - 1) + 4 * sum(l + 1 for l in ls)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        lo, hi = case["n_min"], case["n_max"]
        n = case["frames"] * (hi - lo) / math.log(hi / lo)  # mean of the log-uniform sizes
        bonds = n * 4.19 * case["r_max"] ** 3
        pairs = n * 4.19 * case["rdf_r_max"] ** 3 / 2
        l = case["l"]
        return {"bytes": 12 * n + 28 * bonds + 8 * (2 * l + 1) * n + 4 * n,
                "flops": 8 * bonds / 2 + 10 * pairs + _ylm_flops([l]) * bonds}
    n, rho = _points(case), _density(case)
    r = case.get("r_max", 0.0)
    ball = n * rho * 4.19 * r ** 3
    if kind == "query":
        return {"bytes": 12 * n + 28 * n * case["k"], "flops": 8 * n * case["k"]}
    if kind in ("rdf", "rdf_frame"):
        return {"bytes": 12 * n + 4 * case["bins"], "flops": 10 * ball / 2}
    if kind == "partial_rdf":
        share = case["n"] / (case["n"] + case["n_query"])
        return {"bytes": 12 * (n + case["n_query"]), "flops": 10 * case["n_query"] * rho * share * 4.19 * r ** 3}
    if kind == "order":
        return {"bytes": 12 * n + 4 * n, "flops": (_ylm_flops([case["l"]]) + 8) * ball}
    if kind == "hexatic":
        return {"bytes": 12 * n + 28 * n * case["k"] + 8 * n, "flops": 30 * n * case["k"]}
    if kind == "triclinic":
        ls = range(4, case["lmax"] + 1, 2)
        return {"bytes": 12 * n + 28 * ball + n * sum(8 * (2 * l + 1) + 4 for l in ls),
                "flops": (8 + _ylm_flops(ls)) * ball}
    if kind == "neighbors":
        return {"bytes": 12 * n + 28 * ball + 28 * n * case["k"], "flops": 8 * ball / 2 + 8 * n * case["k"]}
    if kind == "steinhardt":
        nm = 2 * case["l"] + 1
        return {"bytes": 12 * n + 8 * ball + 2 * 8 * nm * n + 3 * 4 * n,
                "flops": (_ylm_flops([case["l"]]) + 2 * nm) * ball + 3 * nm * nm * n}
    if kind == "filters":
        return {"bytes": 28 * ball + 12 * n + 28 * n * 26, "flops": 20 * ball}
    nm = 13
    return {"bytes": 12 * n + 28 * ball + 8 * nm * n + 4 * ball + 12 * n, "flops": (_ylm_flops([6]) + 4 * nm) * ball}


def tolerance(case):
    kind = case["kind"]
    # NeighborLists and bin counts are the reference's bit for bit; their floats are single operations on them
    if kind in ("query", "rdf", "partial_rdf", "rdf_frame", "neighbors", "filters"):
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    # The bond directions come from float32 vectors wrapped into the box (about half an ulp of half the box length
    # off), so the harmonics are off by that angle: measured against 64 bits, 5.4e-5 for psi_6 in a box of 500,
    # 6.5e-5 for q_lm at l = 12 in a box of 84, 4e-6 to 3.5e-5 for q_l and w_l in boxes of 12 to 50.
    rel = {"hexatic": 4e-4, "order": 1.5e-4}.get(kind, 2.5e-4)
    return {"rel": rel, "max": 5e-2, "differ": 0.0}


# ------------------------------------------------------------------ 64-bit evaluation


def _plane_distances(box):
    inv = torch.linalg.inv(_lattice(box))
    return [float(1 / inv[:, k].norm()) for k in range(2 if box[6] else 3)]


def _candidates(box, points, query, r):
    """Yields (query rows, point rows, vectors, squared distances) of every pair closer than r, in pieces."""
    lat = _lattice(box)
    inv = torch.linalg.inv(lat)
    p, q = points.double(), query.double()
    axes = 2 if box[6] else 3
    dims = [max(1, int(d / (r * 1.0001))) for d in _plane_distances(box)] + [1] * (3 - axes)

    lat32, reach = lat.float(), torch.tensor(r, dtype=torch.float32, device=p.device) ** 2

    def close(i, j):
        d = p[j] - q[i]
        image = torch.round(d @ inv)
        # which pairs are bonds is decided on the float32 vector p_j - (q_i + image), as the query is defined
        im = image.float()
        shift = (im[:, 0:1] * lat32[0] + im[:, 1:2] * lat32[1]) + im[:, 2:3] * lat32[2]
        v = points[j] - (query[i] + shift)
        v = v * v
        hit = ((v[:, 0] + v[:, 1]) + v[:, 2] < reach).nonzero()[:, 0]
        d = d[hit] - image[hit] @ lat
        return i[hit], j[hit], d, (d * d).sum(-1)

    if min(dims[:axes]) < 3:
        step = max(1, 20_000_000 // len(p))
        for k in range(0, len(q), step):
            i = torch.arange(k, min(k + step, len(q)), device=p.device)
            j = torch.arange(len(p), device=p.device)
            yield close(i.repeat_interleave(len(p)), j.repeat(len(i)))
        return
    dim = torch.tensor(dims, device=p.device)

    def cells(x):
        c = torch.floor((x @ inv + 0.5) * dim).long()
        return torch.remainder(c, dim)

    def flat(c):
        return (c[:, 2] * dims[1] + c[:, 1]) * dims[0] + c[:, 0]

    fp = flat(cells(p))
    order = torch.argsort(fp, stable=True)
    counts = torch.bincount(fp, minlength=dims[0] * dims[1] * dims[2])
    start = torch.cumsum(counts, 0) - counts
    cq = cells(q)
    by_cell = torch.argsort(flat(cq), stable=True)
    cq = cq[by_cell]
    spans = [range(-1, 2)] * axes + [range(1)] * (3 - axes)
    for dx in spans[0]:
        for dy in spans[1]:
            for dz in spans[2]:
                cell = flat(torch.remainder(cq + torch.tensor([dx, dy, dz], device=p.device), dim))
                cnt, st = counts[cell], start[cell]
                for slot in range(int(counts.max())):
                    has = (cnt > slot).nonzero()[:, 0]
                    if len(has):
                        yield close(by_cell[has], order[st[has] + slot])


def _pairs64(box, points, r, exclude=True):
    """Bonds (i, j, vector, distance) sorted by (i, j)."""
    parts = [x for x in _candidates(box, points, points, r)]
    i, j, d, r2 = (torch.cat([x[k] for x in parts]) for k in range(4))
    if exclude:
        keep = (i != j).nonzero()[:, 0]
        i, j, d, r2 = i[keep], j[keep], d[keep], r2[keep]
    o = torch.argsort(i * len(points) + j)
    return i[o], j[o], d[o], torch.sqrt(r2[o])


def _nearest64(box, points, k, density):
    """The k nearest bonds of every point, sorted by (i, j)."""
    n = len(points)
    two_d = box[6]
    r = 1.4 * (math.sqrt(2 * k / (math.pi * density)) if two_d else (3 * 2 * k / (4 * math.pi * density)) ** (1 / 3))
    i, j, d, dist = _pairs64(box, points, r)
    o = torch.argsort(dist, stable=True)
    o = o[torch.argsort(i[o], stable=True)]
    counts = torch.bincount(i, minlength=n)
    if int(counts.min()) < k:
        return None
    rank = torch.arange(len(o), device=o.device) - (torch.cumsum(counts, 0) - counts)[i[o]]
    o = torch.sort(o[rank < k])[0]
    return i[o], j[o], d[o], dist[o]


def _qlm64(i, d, dist, n, l):
    """(n, 2l + 1) complex q_lm, m = 0 .. l, -1 .. -l."""
    ct, rho = d[:, 2] / dist, torch.sqrt(d[:, 0] ** 2 + d[:, 1] ** 2)
    st = rho / dist
    e1 = torch.complex(torch.where(rho > 0, d[:, 0] / rho, torch.ones_like(rho)),
                       torch.where(rho > 0, d[:, 1] / rho, torch.zeros_like(rho)))
    counts = torch.bincount(i, minlength=n).double()
    out = torch.empty((n, 2 * l + 1), dtype=torch.complex128, device=d.device)
    pmm, em = torch.full_like(ct, 1 / math.sqrt(4 * math.pi)), torch.ones_like(e1)
    for m in range(l + 1):
        if m:
            pmm = -math.sqrt((2 * m + 1) / (2 * m)) * st * pmm
            em = em * e1
        low, p = torch.zeros_like(pmm), pmm
        for k in range(m + 1, l + 1):
            a = math.sqrt((4 * k * k - 1) / (k * k - m * m))
            b = math.sqrt(((k - 1) ** 2 - m * m) / (4 * (k - 1) ** 2 - 1))
            low, p = p, a * (ct * p - b * low)
        s = torch.zeros(n, dtype=torch.complex128, device=d.device).index_add_(0, i, p * em)
        out[:, m] = s / counts
        if m:
            out[:, l + m] = (-1) ** m * torch.conj(out[:, m])
    return out


def _norm64(q):
    return torch.sqrt(4 * math.pi / q.shape[-1] * (q.abs() ** 2).sum(-1))


@functools.lru_cache(None)
def _wigner(l, m1, m2):
    m3 = -m1 - m2
    f = math.factorial
    pre = f(l) ** 3 / f(3 * l + 1)
    pre *= f(l + m1) * f(l - m1) * f(l + m2) * f(l - m2) * f(l + m3) * f(l - m3)
    total = 0.0
    for k in range(max(0, -m1, m2), min(l, l - m1, l + m2) + 1):
        total += (-1) ** k / (f(k) * f(l - k) * f(l - m1 - k) * f(l + m2 - k) * f(m1 + k) * f(k - m2))
    return (-1) ** m3 * math.sqrt(pre) * total


def _wl64(q):
    l = (q.shape[-1] - 1) // 2
    out = torch.zeros(q.shape[:-1], dtype=torch.float64, device=q.device)
    for m1 in range(-l, l + 1):
        for m2 in range(max(-l - m1, -l), min(l - m1, l) + 1):
            m3 = -m1 - m2
            a, b, c = (q[..., m if m >= 0 else l - m] for m in (m1, m2, m3))
            out += _wigner(l, m1, m2) * (a * b * c).real
    return out


def _average64(q, i, j, n):
    counts = torch.bincount(i, minlength=n).double()
    out = torch.empty_like(q)
    for m in range(q.shape[1]):
        s = q[:, m].clone().index_add_(0, i, q[:, m][j])
        out[:, m] = s / (counts + 1)
    return out


def _rows(q):
    return torch.view_as_real(q.contiguous()).reshape(-1, 2)


def _rdf64(box, points, query, r, bins):
    counts = torch.zeros(bins, dtype=torch.float64, device=points.device)
    self_pairs = query is None
    for i, j, _, r2 in _candidates(box, points, points if self_pairs else query, r):
        if self_pairs:
            r2 = r2[i != j]
        counts += torch.bincount((torch.sqrt(r2) * (bins / r)).long().clamp_(max=bins - 1), minlength=bins)
    n, m = len(points), len(points if self_pairs else query)
    volume = float(torch.linalg.det(_lattice(box)))
    edges = torch.arange(bins + 1, dtype=torch.float64, device=points.device) * (r / bins)
    shells = 4 / 3 * math.pi * (edges[1:] ** 3 - edges[:-1] ** 3)
    return {"counts": None, "rdf": counts / (n * (m / volume)) / shells, "n_r": torch.cumsum(counts, 0) / m}


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        # every frame in turn: over about a million points that takes longer than a check should
        if case["frames"] * case["n_max"] > 1_000_000:
            return None
        qs, rows, orders = [], [], []
        for box, points in _trajectory(case, seed):
            i, j, d, dist = _pairs64(box, points, _f32(case["r_max"]))
            q = _qlm64(i, d, dist, len(points), case["l"])
            qs.append(_norm64(q))
            rows.append(torch.view_as_real(q))
            orders.append(float(_norm64(q.mean(0))))
        return {"bonds": None, "order": np.array(orders), "counts": None, "ql": torch.cat(qs),
                "qlm": torch.cat(rows)}
    # whole numbers and copies of given values only
    if kind in ("rdf_frame", "filters"):
        return None
    box, points, query = _system(case, seed)
    n = len(points)
    r = _f32(case.get("r_max", 0.0))

    def bond_list(d, dist):
        pad = torch.zeros(_capacity(case) - len(dist), dtype=torch.float64, device=d.device)
        return {"bonds": None, "neighbors": None, "distances": torch.cat([dist, pad]), "weights": None,
                "vectors": torch.cat([d, pad[:, None].expand(-1, 3)])}

    if kind in ("rdf", "partial_rdf"):
        return _rdf64(box, points, query, r, case["bins"])
    if kind in ("query", "hexatic"):
        near = _nearest64(box, points, case["k"], _density(case))
        if near is None:
            return None
        i, j, d, dist = near
        if kind == "query":
            return {"neighbors": None, "distances": dist, "vectors": d}
        e = torch.complex(d[:, 0] / dist, d[:, 1] / dist) ** case["k"]
        psi = torch.zeros(n, dtype=torch.complex128, device=d.device).index_add_(0, i, e) / case["k"]
        return {"bonds": bond_list(d, dist), "psi": _rows(psi)}
    i, j, d, dist = _pairs64(box, points, r)
    if kind == "order":
        q = _qlm64(i, d, dist, n, case["l"])
        if case["average"]:
            q = _average64(q, i, j, n)
        value = _wl64 if case["wl"] else _norm64
        return {"particle_order": value(q), "order": float(value(q.mean(0)))}
    if kind == "neighbors":
        near = _nearest64(box, points, case["k"], 1.0)
        return {"ball": bond_list(d, dist), "nearest": None if near is None else bond_list(*near[2:])}
    if kind == "triclinic":
        qs = [_qlm64(i, d, dist, n, l) for l in range(4, case["lmax"] + 1, 2)]
        return {"bonds": bond_list(d, dist), "qlm": torch.cat([_rows(q) for q in qs]),
                "ql": torch.stack([_norm64(q) for q in qs], 1),
                "order": np.array([float(_norm64(q.mean(0))) for q in qs])}
    q = _qlm64(i, d, dist, n, case.get("l", 6))
    if kind == "steinhardt":
        ave = _average64(q, i, j, n)
        return {"qlm": _rows(q), "ql": _norm64(q)[:, None], "wl": _wl64(q)[:, None],
                "order": np.array([float(_wl64(q.mean(0)))]), "qlmave": _rows(ave), "qlave": _norm64(ave)[:, None],
                "order_ave": np.array([float(_norm64(ave.mean(0)))])}
    ql = _norm64(q)
    dot = torch.zeros(len(i), dtype=torch.float64, device=d.device)
    for m in range(13):
        dot += (q[:, m][i] * torch.conj(q[:, m][j])).real
    dot *= 4 * math.pi / 13 / (ql[i] * ql[j])
    dot = torch.cat([dot, torch.zeros(_capacity(case) - len(dot), dtype=torch.float64, device=dot.device)])
    return {"qlm": _rows(q), "ql": ql[:, None], "qlij": dot, "connections": None, "cluster": None, "sizes": None, "clusters": None}
