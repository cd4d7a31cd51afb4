"""Sizes at which the launch shapes of the kernels change: tile edges and
remainders, the smallest systems, and the borders between two code paths."""

import ctypes

import numpy as np
import numpy.testing as npt
import pytest

import freud_amd
from freud_amd import _lib
from freud_amd.box import Box

pytestmark = pytest.mark.gpu


def _bt(box):
    return (box.Lx, box.Ly, box.Lz, box.xy, box.xz, box.yz, box.is2D)


def _uniform(n, density=1.0, seed=0, tilts=(0.0, 0.0, 0.0)):
    side = max((n / density) ** (1 / 3), 3.2)
    box = Box(side, side, side, *tilts)
    frac = np.random.default_rng(seed).random((n, 3)).astype(np.float32)
    return box, np.ascontiguousarray(box.make_absolute(frac), np.float32)


@pytest.mark.parametrize("l", [0, 1, 2, 3, 4, 6, 8, 9, 16, 17, 20])
@pytest.mark.parametrize("n", [3, 63, 64, 65, 1025])
def test_average_steinhardt_lane_groups(oracle, l, n):
    """Averaged q_l: lane groups of every width (1 to 16 lanes per row), points
    with no, few and many bonds.  Sums in bond order as the oracle's: the
    tolerance is the suite's 1e-5 for q_l."""
    box, pts = _uniform(n, seed=l)
    nl = freud_amd.AABBQuery(box, pts).query(pts, dict(r_max=1.5, exclude_ii=True)).toNeighborList()
    ref_nl = oracle.query(_bt(box), pts, pts, dict(r_max=1.5, exclude_ii=True), nthreads=4)
    st = freud_amd.order.Steinhardt(l, average=True).compute((box, pts), neighbors=nl)
    ref = oracle.steinhardt(_bt(box), pts, ref_nl, [l], average=True, nthreads=4)
    npt.assert_allclose(st.particle_order, ref["ql_ave"][:, 0], atol=1e-5, equal_nan=True)
    npt.assert_allclose(st.order, ref["order"][0], atol=1e-5, equal_nan=True)


@pytest.mark.parametrize("l", [4, 6])
@pytest.mark.parametrize("n", [4, 64, 65, 1027])
@pytest.mark.parametrize("normalize", [True, False])
def test_solid_bonds_lane_groups(oracle, l, n, normalize):
    """Bond dot products from the oracle's own formula on the q_lm of the same
    run: the same products added in the same order, so the difference allowed
    is one rounding of the normalisation (2^-23 relative, as 1e-6)."""
    box, pts = _uniform(n, seed=n + l)
    nl = freud_amd.AABBQuery(box, pts).query(pts, dict(r_max=1.5, exclude_ii=True)).toNeighborList()
    sl = freud_amd.order.SolidLiquid(l, 0.3, 4, normalize_q=normalize).compute((box, pts), neighbors=nl)
    st = freud_amd.order.Steinhardt(l).compute((box, pts), neighbors=nl)
    ref_nl = oracle.query(_bt(box), pts, pts, dict(r_max=1.5, exclude_ii=True), nthreads=4)
    ref = oracle.solidliquid(ref_nl, st.particle_harmonics, st.ql, l, 0.3, 4, normalize_q=normalize)
    npt.assert_allclose(sl.ql_ij, ref["ql_ij"], rtol=1e-6, atol=1e-7, equal_nan=True)
    if not np.any(np.abs(ref["ql_ij"] - 0.3) < 1e-6):
        npt.assert_array_equal(sl.num_connections, ref["num_connections"])
        npt.assert_array_equal(sl.cluster_idx, ref["cluster_idx"])


@pytest.mark.parametrize("l", [4, 6])
def test_steinhardt_and_solid_bonds_unstaged(oracle, l):
    """A clump whose tiles hold more bonds than the LDS stage next to ordinary
    tiles: both branches of the bond kernels and of the averaged q_l."""
    box = Box.cube(24.0)
    rng = np.random.default_rng(l)
    pts = ((rng.random((3000, 3)) - 0.5) * 24).astype(np.float32)
    pts[:400] = (rng.standard_normal((400, 3)) * 0.6).astype(np.float32)
    args = dict(r_max=1.5, exclude_ii=True)
    nl = freud_amd.AABBQuery(box, pts).query(pts, args).toNeighborList()
    assert nl.neighbor_counts[:256].sum() > 4096 and nl.neighbor_counts[512:768].sum() < 4096
    ref_nl = oracle.query(_bt(box), pts, pts, args, nthreads=4)
    st = freud_amd.order.Steinhardt(l, average=True).compute((box, pts), neighbors=nl)
    ref = oracle.steinhardt(_bt(box), pts, ref_nl, [l], average=True, nthreads=4)
    npt.assert_allclose(st.particle_order, ref["ql_ave"][:, 0], atol=1e-5, equal_nan=True)
    sl = freud_amd.order.SolidLiquid(l, 0.3, 4).compute((box, pts), neighbors=nl)
    one = freud_amd.order.Steinhardt(l).compute((box, pts), neighbors=nl)
    ref = oracle.solidliquid(ref_nl, one.particle_harmonics, one.ql, l, 0.3, 4, normalize_q=True)
    npt.assert_allclose(sl.ql_ij, ref["ql_ij"], rtol=1e-6, atol=1e-7, equal_nan=True)


@pytest.mark.parametrize("l", [4, 6])
def test_solid_bonds_past_two_to_the_31(l):
    """A list of 2,152,913,600 bonds (60 GB): those past 2^31, the last 117
    points', have the neighbours that the list says.  q_lm against a run with
    the points reversed, where those points come first: means of 46,399
    terms of size 1, each sum within a few hundred ulps of 2^-24 (1e-6 allowed).
    Dot products against float64 from the run's own q_lm: 13 products and sums
    of 2^-24 each of |q_i| |q_j| (4e-6 allowed).  Another neighbour differs by
    1e-3 and 1e-1."""
    n, tail = 46400, 117
    box = Box.cube(40.0)
    pts = ((np.random.default_rng(0).random((n, 3)) - 0.5) * 40).astype(np.float32)
    qlm = []
    for points in (pts[::-1].copy(), pts):
        nl = freud_amd.locality.NeighborList.all_pairs((box, points))
        sl = freud_amd.order.SolidLiquid(l, 0.5, n).compute((box, points), neighbors=nl)
        qlm.append(sl.particle_harmonics)
        first = (n - tail) * (n - 1)
        assert 2**31 < first < len(nl) == n * (n - 1)
        dots = _lib.copy_d2h(sl._d_qlij.ptr + 4 * first, (tail, n - 1), np.float32)
        del sl, nl
    npt.assert_allclose(qlm[1][-tail:], qlm[0][:tail][::-1], atol=1e-6)
    q = qlm[1].astype(np.complex128)
    q /= np.linalg.norm(q, axis=1)[:, None]
    ref = (q[-tail:] @ q.conj().T).real
    others = np.arange(n) != np.arange(n - tail, n)[:, None]
    npt.assert_allclose(dots, ref[others].reshape(tail, n - 1), atol=4e-6)


BOXES = {
    "cube": Box.cube(16),
    "triclinic": Box(12.0, 13.0, 14.0, 0.3, -0.2, 0.25),
    "square": Box.square(24.0),
    "flat": Box(30.0, 9.0, 12.0),
    # across the edge of a box this large the estimate's bound exceeds its table: every pair exact
    "large": Box.cube(900.0),
}


@pytest.mark.parametrize("name", sorted(BOXES))
@pytest.mark.parametrize("n", [2, 9, 513, 4096])
@pytest.mark.parametrize("bins,r_max,r_min", [(100, 4.0, 0.0), (37, 2.3, 0.5), (512, 4.2, 0.0), (513, 4.0, 0.0),
                                              (1, 3.0, 0.0)])
def test_rdf_estimate_borders(oracle, name, n, bins, r_max, r_min):
    """Bin counts bit for bit, self and with distinct query points, on both
    sides of the estimate table's largest bin count, in dense and nearly empty
    boxes."""
    box = BOXES[name]
    rng = np.random.default_rng(n + bins)
    pts = np.ascontiguousarray(box.make_absolute(rng.random((n, 3)).astype(np.float32)), np.float32)
    q = np.ascontiguousarray(box.wrap(pts[::2] + np.float32(0.07)), np.float32)
    if box.is2D:
        pts[:, 2] = q[:, 2] = 0
    rdf = freud_amd.density.RDF(bins, r_max, r_min=r_min)
    ref = oracle.rdf_accumulate(_bt(box), pts, pts, bins, r_max, r_min=r_min, exclude_ii=True, nthreads=4)
    npt.assert_array_equal(rdf.compute((box, pts)).bin_counts, ref)
    ref = oracle.rdf_accumulate(_bt(box), pts, q, bins, r_max, r_min=r_min, exclude_ii=False, nthreads=4)
    npt.assert_array_equal(rdf.compute((box, pts), query_points=q).bin_counts, ref)


def _rdf_kernels(run):
    _lib.profile_reset()
    _lib.profile_enable()
    counts = run()
    _lib.profile_enable(False)
    return counts, set(_lib.profile_stats())


@pytest.mark.parametrize("is2D", [False, True])
@pytest.mark.parametrize("n,n_query,r_max,kernel", [
    (30000, 1, 1.1, "rdf_wave_kernel"), (30000, 3001, 1.1, "rdf_wave_kernel"), (30000, 60001, 1.1, "rdf_query_kernel"),
    (30000, 7, 2.0, "rdf_wave_kernel"), (30000, 2003, 2.0, "rdf_wave_kernel"), (900, 20001, 2.0, "rdf_est_kernel"),
    (30000, 7, 3.5, "rdf_est_kernel"), (200001, 30001, 2.0, "rdf_est_kernel")])
def test_rdf_routes_of_query_points(oracle, is2D, n, n_query, r_max, kernel):
    """Each kernel that takes distinct query points, by the size of their
    stencils and by their number: bin counts bit for bit, with points and query
    points inside and outside the box, in a triclinic box too.  (2D boxes have
    fewer cells and candidates per point: the kernel is not asserted.)"""
    side = (n / 1.0) ** (1 / 3)
    rng = np.random.default_rng(n_query)
    for tilts in ((0.0, 0.0, 0.0), (0.2, -0.1, 0.15)):
        box = Box.square(n ** 0.5) if is2D else Box(side, side, side, *tilts)
        frac = rng.random((n + n_query, 3)).astype(np.float32)
        both = np.ascontiguousarray(box.make_absolute(frac), np.float32)
        if is2D:
            both[:, 2] = 0
        moved = both.copy()
        moved[::3, 0] += np.float32(box.Lx)
        for p, q in ((both, both), (moved, both), (both, moved), (moved, moved)):
            pts, query = p[:n], q[n:]
            ref = oracle.rdf_accumulate(_bt(box), pts, query, 60, r_max, r_min=0.2, exclude_ii=False, nthreads=16)
            rdf = freud_amd.density.RDF(60, r_max, r_min=0.2)
            counts, ran = _rdf_kernels(lambda: rdf.compute((box, pts), query_points=query).bin_counts)
            npt.assert_array_equal(counts, ref)
            if not is2D:
                assert any(kernel in name for name in ran), ran


@pytest.mark.parametrize("n_query", [2055, 2056, 4103, 4104, 8199, 8200, 49151, 49152, 200001])
def test_rdf_row_clusters_of_query_points(oracle, n_query):
    """Row clusters of distinct query points, and of the points themselves, on
    both sides of the sizes at which 8, 4, 2 waves share a cluster and at
    which a wave takes two."""
    n, r_max = 3000, 2.5
    box = Box.cube(14.5)
    both = ((np.random.default_rng(n_query).random((n + n_query, 3)) - 0.5) * 14.49).astype(np.float32)
    pts, q = both[:n], both[n:]
    ref = oracle.rdf_accumulate(_bt(box), pts, q, 80, r_max, exclude_ii=False, nthreads=16)
    rdf = freud_amd.density.RDF(80, r_max)
    counts, ran = _rdf_kernels(lambda: rdf.compute((box, pts), query_points=q).bin_counts)
    npt.assert_array_equal(counts, ref)
    assert any("rdf_est_kernel" in name for name in ran), ran
    box, pts = _uniform(n_query, seed=n_query)
    ref = oracle.rdf_accumulate(_bt(box), pts, pts, 80, 1.5, exclude_ii=True, nthreads=16)
    npt.assert_array_equal(freud_amd.density.RDF(80, 1.5).compute((box, pts)).bin_counts, ref)


@pytest.mark.parametrize("which", ["points", "query_points", "both"])
def test_rdf_points_outside_the_box(oracle, which):
    """Systems with points (or query points) outside the box leave the
    estimate kernel to the general walk."""
    box = Box.cube(14.0)
    rng = np.random.default_rng(3)
    pts = ((rng.random((1500, 3)) - 0.5) * 14).astype(np.float32)
    q = ((rng.random((700, 3)) - 0.5) * 14).astype(np.float32)
    if which != "query_points":
        pts[::7, 0] += np.float32(14.0)
    if which != "points":
        q[::5, 2] -= np.float32(14.0)
    rdf = freud_amd.density.RDF(60, 3.0)
    ref = oracle.rdf_accumulate(_bt(box), pts, q, 60, 3.0, exclude_ii=False, nthreads=4)
    npt.assert_array_equal(rdf.compute((box, pts), query_points=q).bin_counts, ref)
    ref = oracle.rdf_accumulate(_bt(box), pts, pts, 60, 3.0, exclude_ii=True, nthreads=4)
    npt.assert_array_equal(rdf.compute((box, pts)).bin_counts, ref)


@pytest.mark.parametrize("name, n, r", [("small", 300, 2.9), ("thin", 900, 1.9), ("square", 700, 3.0),
                                        ("square", 3000, 0.2), ("cube", 4000, 1.2), ("cube", 50000, 1.0),
                                        ("cube", 56000, 1.0)])
def test_rdf_outside_routes(oracle, name, n, r):
    """Systems off the box, a wave or a thread per point (above some 53,000
    points in the cube, 1,000 per candidate in two dimensions): rows of cells
    that wrap more than once, boxes of two dimensions and tilted ones, points
    boxes away; query points of their own, few and many, with the points in the
    box or off it."""
    box = {"small": Box(6.0, 6.0, 6.0, 0.2, -0.1, 0.15), "thin": Box(4.0, 30.0, 8.0),
           "square": Box.square(26.0), "cube": Box.cube((n / 0.8) ** (1 / 3))}[name]
    rng = np.random.default_rng(n)
    inside = box.make_absolute(rng.random((n, 3)).astype(np.float32))
    if box.is2D:
        inside[:, 2] = 0
    images = rng.integers(-3, 4, (n, 3))
    images[::3] = 0
    if box.is2D:
        images[:, 2] = 0
    off = box.unwrap(inside, images).astype(np.float32)
    rdf = freud_amd.density.RDF(70, r)
    ref = oracle.rdf_accumulate(_bt(box), off, off, 70, r, exclude_ii=True, nthreads=16)
    npt.assert_array_equal(rdf.compute((box, off)).bin_counts, ref)
    for pts, q in ((inside, off[::2]), (off, inside[: n // 3])):
        q = np.ascontiguousarray(q)
        ref = oracle.rdf_accumulate(_bt(box), pts, q, 70, r, exclude_ii=False, nthreads=16)
        npt.assert_array_equal(rdf.compute((box, pts), query_points=q).bin_counts, ref)


def test_rdf_query_ranges_inside_the_histogram(oracle):
    """A query radius inside the histogram's range cuts bins apart (exact
    kernel); index exclusion with distinct query points (general kernel)."""
    box, pts = _uniform(3000, seed=4)
    q = np.ascontiguousarray(box.wrap(pts + np.float32(0.2)), np.float32)
    rdf = freud_amd.density.RDF(80, 4.0)
    for nb in (dict(r_max=2.71), dict(r_max=4.0, r_min=1.3), dict(r_max=4.0, exclude_ii=True)):
        for query in (None, q):
            ex = nb.get("exclude_ii", query is None)
            nl = oracle.query(_bt(box), pts, pts if query is None else query, dict(nb, exclude_ii=ex), nthreads=4)
            ref = oracle.rdf_bin(nl["distances"], 80, 0.0, 4.0)
            got = rdf.compute((box, pts), query_points=query, neighbors=dict(nb)).bin_counts
            npt.assert_array_equal(got, ref)


@pytest.mark.parametrize("bonds", [1, 4096, 8191, 8192, 8193, 70001, (1 << 22) + 5])
def test_scan_sizes_through_filter(bonds):
    """The count scan at its tile, single-workgroup and library borders:
    filtering a list compacts it by a scan over its bonds, its segments by one
    over its points."""
    rng = np.random.default_rng(bonds)
    n = max(1, bonds // 7)
    i = np.sort(rng.integers(0, n, bonds)).astype(np.uint32)
    j = rng.integers(0, n, bonds).astype(np.uint32)
    v = rng.random((bonds, 3)).astype(np.float32)
    nl = freud_amd.locality.NeighborList.from_arrays(n, n, i, j, v)
    keep = rng.random(bonds) < 0.6
    nl.filter(keep)
    npt.assert_array_equal(nl[:], np.stack([i[keep], j[keep]], 1))
    npt.assert_array_equal(nl.vectors, v[keep])
    npt.assert_array_equal(nl.neighbor_counts, np.bincount(i[keep], minlength=n))


@pytest.mark.parametrize("n", [0, 1, 511, 512, 8192, 8193, 70001, (1 << 22), (1 << 22) + 5])
@pytest.mark.parametrize("largest", [3, 9_000_000, 2**32 - 1])
def test_scan_totals_beyond_32_bits(n, largest):
    """The total of a list is a 64-bit sum whatever its counts (a query refuses
    a list by it); offsets and segments are the sums modulo 2^32."""
    counts = np.random.default_rng(n).integers(largest // 2, largest + 1, n, dtype=np.uint32)
    counts[::5] = 0
    d_counts = _lib.DeviceArray.from_numpy(counts)
    d_offsets, d_segments = _lib.DeviceArray((n + 1,), np.uint32), _lib.DeviceArray((max(n, 1),), np.uint32)
    total = ctypes.c_uint64()
    _lib.check(_lib.lib().fa_nlist_offsets(d_counts.ptr, n, d_offsets.ptr, d_segments.ptr,
                                           ctypes.byref(total)))
    sums = np.cumsum(np.concatenate([[0], counts]), dtype=np.uint64)
    assert total.value == int(sums[-1])
    offsets = (sums & np.uint64(2**32 - 1)).astype(np.uint32)
    npt.assert_array_equal(d_offsets.numpy(), offsets)
    npt.assert_array_equal(d_segments.numpy()[:n], np.where(counts > 0, offsets[:-1], 0))


@pytest.mark.parametrize("n", [2, 4096, 8192, 8193, 40001, (1 << 22) + 5])
def test_query_segments(n):
    """Offsets, counts and segments (0 for points without bonds) of a query, up
    to more points than the library's own scan takes."""
    box, pts = _uniform(n, density=0.3, seed=n)
    for args in (dict(r_max=1.0, exclude_ii=True), dict(num_neighbors=1, r_max=0.9, exclude_ii=True)):
        nl = freud_amd.AABBQuery(box, pts).query(pts, args).toNeighborList()
        counts = np.bincount(nl[:][:, 0], minlength=n)
        npt.assert_array_equal(nl.neighbor_counts, counts)
        start = np.cumsum(counts) - counts
        npt.assert_array_equal(nl.segments, np.where(counts > 0, start, 0))


def _assert_same(nl, ref):
    npt.assert_array_equal(nl[:], ref["ij"])
    npt.assert_array_equal(nl.distances, ref["distances"])
    npt.assert_array_equal(nl.vectors, ref["vectors"])


@pytest.mark.parametrize("name", ["cube", "triclinic", "square", "flat"])
@pytest.mark.parametrize("n", [2, 65, 1500, 8193])
@pytest.mark.parametrize("outside", [False, True])
def test_wave_queries(oracle, name, n, outside):
    """One wave per query point, up to its largest kNN size and past it: ball
    and nearest queries against the oracle, self and with distinct query
    points, in every order, with points inside and outside the box, in boxes
    of a few cells and of many."""
    box = BOXES[name]
    rng = np.random.default_rng(n)
    pts = np.ascontiguousarray(box.make_absolute(rng.random((n, 3)).astype(np.float32)), np.float32)
    q = np.ascontiguousarray(box.wrap(pts[::3] + np.float32(0.31)), np.float32)
    if outside:
        pts[::5, 0] += np.float32(box.Lx)
        q[::4, 1] -= np.float32(box.Ly)
    if box.is2D:
        pts[:, 2] = q[:, 2] = 0
    nq = freud_amd.AABBQuery(box, pts)
    r = min(1.4, (60 * box.volume / n / 4.2) ** (1 / 3)) if not box.is2D else 1.2
    for args in (dict(r_max=r, exclude_ii=True), dict(r_max=r, r_min=0.4 * r), dict(num_neighbors=5, exclude_ii=True),
                 dict(num_neighbors=17, r_max=2.0), dict(num_neighbors=1, r_min=0.3)):
        for points in (pts, q):
            for by_distance in (False, True):
                ref = oracle.query(_bt(box), pts, points, args, sort_by_distance=by_distance, nthreads=4)
                nl = nq.query(points, args).toNeighborList(sort_by_distance=by_distance)
                _assert_same(nl, ref)


@pytest.mark.parametrize("n", [700, 40000])
@pytest.mark.parametrize("boxes", [-511, -505, -500, 499, 500, 501, 505, 510])
def test_points_many_boxes_out(oracle, n, boxes):
    """Unwrapped coordinates hundreds of box lengths out: the image offsets of a
    point and of its query cancel, on both sides of the wave queries' largest
    size.  Box lengths and coordinates are dyadic, so that the shift is exact."""
    side = 8.0 if n < 32768 else 32.0
    box = Box.cube(side)
    rng = np.random.default_rng(n)
    pts = ((rng.integers(0, 2**10, (n, 3)) + 0.5) * (side / 2**10) - side / 2).astype(np.float32)
    pts[:, 1] += np.float32(side * boxes)
    nq = freud_amd.AABBQuery(box, pts)
    q = pts[::3]
    for args in (dict(r_max=1.0, exclude_ii=True), dict(num_neighbors=6, exclude_ii=True)):
        for points in (pts, q):
            ref = oracle.query(_bt(box), pts, points, args, nthreads=16)
            nl = nq.query(points, args).toNeighborList()
            _assert_same(nl, ref)
            assert len(ref["distances"]) > 0


def test_nearest_query_at_the_stencil_radius(oracle):
    """A search radius equal to the radius that the cells cover (box length
    20, cells of 5, less 1e-4): a neighbour below it in r_sq whose rounded
    distance equals it belongs to the answer."""
    f = np.float32
    r = f(5) * (f(1) - f(1e-4))
    ang = np.random.default_rng(0).random(20000) * np.pi / 2
    x, y = (r * np.cos(ang)).astype(f), (r * np.sin(ang)).astype(f)
    r_sq = x * x + y * y
    on = np.nonzero((r_sq < r * r) & (np.sqrt(r_sq) == r))[0][:7]
    assert len(on) == 7
    box = Box.cube(20)
    pts = ((np.random.default_rng(1).random((1000, 3)) - 0.5) * 20).astype(f)
    pts[:7] = np.stack([x[on], y[on], 0 * x[on]], 1)
    q = np.zeros((1, 3), f)
    args = dict(num_neighbors=20, r_max=float(r), r_guess=float(r), r_min=4.999)
    ref = oracle.query(_bt(box), pts, q, args, nthreads=1)
    assert 7 <= len(ref["distances"]) < 20
    _assert_same(freud_amd.AABBQuery(box, pts).query(q, args).toNeighborList(), ref)


def _irregular(kind, n, is2D, rng):
    """(box, points): a droplet in a large box, two dense clumps and a vapour, or
    a slab in an elongated box."""
    dim = 2 if is2D else 3
    make = Box.square if is2D else Box.cube
    if kind == "droplet":
        box, pts = make(30.0), rng.standard_normal((n, dim)) * 1.7
    elif kind == "clumps":
        box, pts = make(24.0), (rng.random((n, dim)) - 0.5) * 24
        pts[: n // 2] = rng.standard_normal((n // 2, dim)) * 0.4
        pts[n // 3: n // 2] += 8
    else:
        box, pts = (Box(9.0, 60.0) if is2D else Box(9.0, 8.0, 60.0)), (rng.random((n, dim)) - 0.5) * 8
    if is2D:
        pts = np.concatenate([pts, np.zeros((n, 1))], 1)
    return box, np.ascontiguousarray(box.wrap(pts.astype(np.float32)), np.float32)


@pytest.mark.parametrize("is2D", [False, True])
@pytest.mark.parametrize("kind", ["droplet", "clumps", "slab"])
@pytest.mark.parametrize("n", [40, 900, 6000])
def test_wave_nearest_of_irregular_systems(oracle, kind, n, is2D):
    """Stencils with many times the wave's keys, and query points so far from
    every point that the search takes rings upon rings: all in the one kernel."""
    rng = np.random.default_rng(n + is2D)
    box, pts = _irregular(kind, n, is2D, rng)
    q = ((rng.random((500, 3)) - 0.5) * np.array([box.Lx, box.Ly, box.Lz])).astype(np.float32)
    if is2D:
        q[:, 2] = 0
    moved = pts.copy()
    moved[::5, 1] += np.float32(3 * box.Ly)
    nq, out = freud_amd.AABBQuery(box, pts), freud_amd.AABBQuery(box, moved)
    for args in (dict(num_neighbors=6, exclude_ii=True), dict(num_neighbors=17, r_max=3.9),
                 dict(num_neighbors=64, exclude_ii=True), dict(num_neighbors=9, r_min=0.3), dict(num_neighbors=1)):
        for obj, stored, points in ((nq, pts, pts), (nq, pts, q), (out, moved, moved)):
            ref = oracle.query(_bt(box), stored, points, args, nthreads=16)
            _lib.profile_reset()
            _lib.profile_enable()
            nl = obj.query(points, args).toNeighborList()
            _lib.profile_enable(False)
            _assert_same(nl, ref)
            assert "knn_wave_kernel" in _lib.profile_stats() and "knn_refine_kernel" not in _lib.profile_stats()


@pytest.mark.parametrize("by_distance", [False, True])
def test_wave_ball_query_of_clumps(oracle, by_distance):
    """A clump with more bonds per point than a wave keeps: the general emission
    takes over from the wave's walk, which is not done twice."""
    box = Box.cube(20.0)
    rng = np.random.default_rng(8)
    pts = ((rng.random((1500, 3)) - 0.5) * 20).astype(np.float32)
    pts[:600] = (rng.standard_normal((600, 3)) * 0.3).astype(np.float32)
    nq = freud_amd.AABBQuery(box, pts)
    for points in (pts, pts[300:900]):
        for args in (dict(r_max=1.5, exclude_ii=True), dict(num_neighbors=12, exclude_ii=True)):
            ref = oracle.query(_bt(box), pts, points, args, sort_by_distance=by_distance, nthreads=4)
            _lib.profile_reset()
            _lib.profile_enable()
            nl = nq.query(points, args).toNeighborList(sort_by_distance=by_distance)
            ran = _lib.profile_stats()
            _lib.profile_enable(False)
            _assert_same(nl, ref)
            assert "ball_walk_kernel" not in ran


@pytest.mark.parametrize("kind", ["aabb", "linkcell", "cellquery"])
@pytest.mark.parametrize("bonds", [7, 15, 30, 37, 45])
def test_large_ball_queries_by_bond_count(oracle, kind, bonds):
    """More points than the wave queries take, on both sides of the lists that
    the sort networks hold (16, 32, 48 keys) and of the walk's key stage, with a
    clump past every stage; consecutive and scattered storage orders."""
    n, side = 33000, 32.08
    box = Box.cube(side)
    rng = np.random.default_rng(bonds)
    pts = ((rng.random((n, 3)) - 0.5) * side).astype(np.float32)
    pts[:200] = (rng.standard_normal((200, 3)) * 0.5).astype(np.float32)
    r = (bonds / 4.18879) ** (1 / 3)
    cls = {"aabb": freud_amd.AABBQuery, "linkcell": freud_amd.LinkCell, "cellquery": freud_amd.CellQuery}[kind]
    for points in (pts, pts[np.lexsort((pts[:, 0] // 1, pts[:, 1] // 1, pts[:, 2] // 1))]):
        nq = cls(box, points) if kind != "linkcell" else cls(box, points, cell_width=r)
        args = dict(r_max=r, exclude_ii=True)
        for by_distance in (False, True):
            ref = oracle.query(_bt(box), points, points, args, nq_type=kind if kind != "cellquery" else "cellquery",
                               cell_width=r, sort_by_distance=by_distance, nthreads=16)
            nl = nq.query(points, args).toNeighborList(sort_by_distance=by_distance)
            _assert_same(nl, ref)


@pytest.mark.parametrize("kind", ["aabb", "linkcell", "cellquery"])
@pytest.mark.parametrize("bonds", [90, 130, 230, 300])
def test_ball_emission_of_long_lists(oracle, kind, bonds):
    """Lists of more keys than a wave has lanes, from 128 points per workgroup
    down to 32 and past what fits in LDS, with some points of few bonds; self
    and with distinct query points, by index and by distance."""
    n = 2501
    side = n ** (1 / 3)
    box = Box.cube(side * 1.2)
    rng = np.random.default_rng(bonds)
    pts = ((rng.random((n, 3)) - 0.5) * side).astype(np.float32)
    r = (bonds / 4.18879) ** (1 / 3)
    make = {"aabb": freud_amd.AABBQuery, "cellquery": freud_amd.CellQuery,
            "linkcell": lambda b, p: freud_amd.LinkCell(b, p, cell_width=r)}[kind]
    nq = make(box, pts)
    q = np.ascontiguousarray(box.wrap(pts[:1501] + np.float32(0.3)), np.float32)
    for points in (pts, q):
        for by_distance in (False, True):
            args = dict(r_max=r, exclude_ii=True)
            ref = oracle.query(_bt(box), pts, points, args, nq_type=kind, cell_width=r, sort_by_distance=by_distance,
                               nthreads=16)
            _assert_same(nq.query(points, args).toNeighborList(sort_by_distance=by_distance), ref)


@pytest.mark.parametrize("parts", [1, 3, 70])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 5000])
def test_cluster_chains(n, parts):
    """Chains interleaved through the indices (one, three or more clusters in
    every wave), every eleventh point alone: sizes and members are whole
    numbers, equal to a host union's."""
    members = np.arange(n, dtype=np.uint32)
    chained = members[members % 11 != 5]
    a, b = chained[:-parts], chained[parts:]
    if parts >= len(chained):
        a = b = chained[:0]
    label = members.copy()
    for x, y in zip(a, b):
        label[y] = label[x]
    _, inverse, count = np.unique(label, return_inverse=True, return_counts=True)
    order = np.argsort(-count, kind="stable")
    rank = np.empty_like(order)
    rank[order] = np.arange(len(order))
    box = Box.cube(100.0)
    pts = np.zeros((n, 3), np.float32)
    if len(a):
        nl = freud_amd.locality.NeighborList.from_arrays(n, n, a, b, np.ones((len(a), 3), np.float32))
    else:
        pts[:, 0] = np.arange(n) * np.float32(100.0 / (n + 1)) - 50
        nl = freud_amd.AABBQuery(box, pts).query(pts, dict(r_max=1e-3, exclude_ii=True)).toNeighborList()
    cl = freud_amd.cluster.Cluster().compute((box, pts), neighbors=nl)
    assert cl.num_clusters == len(count)
    npt.assert_array_equal(cl.cluster_idx, rank[inverse])


@pytest.mark.parametrize("store", ["random", "sorted", "lattice"])
@pytest.mark.parametrize("n", [500, 8192, 8193, 32000])
@pytest.mark.parametrize("bonds", [0.8, 2.5, 4, 9, 40])
def test_cluster_percolation(oracle, store, n, bonds):
    """Below, at and above percolation, with one to three hooking rounds over
    every, every other or every eighth bond, points stored in random and in
    spatial order: labels and sizes equal the oracle's, with and without
    a mask of kept bonds."""
    box, pts = _uniform(n, seed=n)
    if store == "sorted":
        pts = pts[np.lexsort((pts[:, 0] // 2, pts[:, 1] // 2, pts[:, 2] // 2))]
    elif store == "lattice":
        m = int(np.ceil((n / 4) ** (1 / 3)))
        a = np.arange(m)
        grid = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 1, 3)
        frac = (grid + np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])).reshape(-1, 3)[:n]
        frac = frac + np.random.default_rng(1).standard_normal(frac.shape) * 0.05
        box = Box.cube(m * 4 ** (1 / 3))
        pts = np.ascontiguousarray(box.wrap((frac - m / 2) * 4 ** (1 / 3)), np.float32)
    r = (bonds / 4.18879) ** (1 / 3)
    nl = freud_amd.AABBQuery(box, pts).query(pts, dict(r_max=r, exclude_ii=True)).toNeighborList()
    ref_nl = oracle.query(_bt(box), pts, pts, dict(r_max=r, exclude_ii=True), nthreads=16)
    cl = freud_amd.cluster.Cluster().compute((box, pts), neighbors=nl)
    idx, num = oracle.cluster(len(pts), ref_nl["ij"])
    npt.assert_array_equal(cl.cluster_idx, idx)
    assert cl.num_clusters == num
    st = freud_amd.order.Steinhardt(6).compute((box, pts), neighbors=nl)
    sl = freud_amd.order.SolidLiquid(6, 0.4, 2).compute((box, pts), neighbors=nl)
    ref = oracle.solidliquid(ref_nl, st.particle_harmonics, st.ql, 6, 0.4, 2, normalize_q=True)
    if not np.any(np.abs(ref["ql_ij"] - 0.4) < 1e-6):
        npt.assert_array_equal(sl.cluster_idx, ref["cluster_idx"])


@pytest.mark.parametrize("n, bonds", [(33001, 5), (33001, 13), (33001, 18), (33001, 28), (33001, 43), (33001, 52),
                                      (66000, 28), (140000, 18), (140000, 28), (300000, 18)])
def test_ball_emission_of_systems_of_middle_size(oracle, n, bonds):
    """Workgroups of 64, 128 and 256 points, up to as many as are resident and
    beyond, with each network for lists of about its length; in the caller's
    order and in the walk's."""
    side = n ** (1 / 3)
    box = Box.cube(side * 1.0001)
    rng = np.random.default_rng(bonds)
    pts = ((rng.random((n, 3)) - 0.5) * side).astype(np.float32)
    if n == 66000:
        pts = pts[np.argsort(np.floor(pts[:, 2] / 2), kind="stable")]
    args = dict(r_max=(bonds / 4.18879) ** (1 / 3), exclude_ii=True)
    ref = oracle.query(_bt(box), pts, pts, args, nthreads=16)
    _assert_same(freud_amd.AABBQuery(box, pts).query(pts, args).toNeighborList(), ref)
