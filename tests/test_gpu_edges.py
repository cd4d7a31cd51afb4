"""Sizes at which the launch shapes of the kernels change: tile edges and
remainders, the smallest systems, and the borders between two code paths."""

import numpy as np
import numpy.testing as npt
import pytest

import freud_amd
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
