"""Lists of particles that the count pass's error band does not cover: in a
kept grid, particles that turned non-finite or were carried far outside it (the
binning clamps them to an edge cell; the host learns of it one binning later),
radii far above the cells, and cells near the ends of the float range.  The rows must be those of the distance test
alone, and hold sources that exist.  Coordinates are multiples of 1/64, exact
in both precisions."""
import numpy as np
import pytest

from oracle import cpu_ref
from pysph_amd import _lib

pytestmark = pytest.mark.gpu

NAN, INF = np.nan, np.inf


def _cloud(dim, n=700, side=4):
    rng = np.random.default_rng(23)
    p = rng.integers(0, 64 * side, size=(n, 3)) / 64.0
    if dim == 2:
        p[:, 2] = 0.0
    return p


def _kept_lists(p, moved, precision):
    """Lists of p, then of `moved` on the grid kept from p, and the locator."""
    from pysph_amd.base import api as base
    from pysph_amd.base.nnps import CellManager, NNPSManager
    h = np.full(len(p), 0.5)
    pa = base.get_particle_array(name="f", cl_precision=precision, x=p[:, 0].copy(),
                                 y=p[:, 1].copy(), z=p[:, 2].copy(), h=h)
    cm = CellManager(arrays_to_bin=[pa], radius_scale=2.0, precision=precision)
    loc = NNPSManager(cell_manager=cm).get_neighbor_particle_locator(pa, pa, 2.0)
    loc.get_csr()
    # as the integrator's stage kernels leave the array
    pa.set(x=moved[:, 0].copy(), y=moved[:, 1].copy(), z=moved[:, 2].copy())
    pa._stepped_xyz = tuple(pa.version(k) for k in "xyz")
    builds = cm.grid_builds
    loc.update_status()
    off, idx = (t.cpu().numpy() for t in loc.get_csr())
    assert cm.grid_builds == builds  # the grid was kept
    return pa, loc, cm, off, idx


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("dim", [2, 3])
def test_non_finite_particles_have_no_neighbours_and_are_none(gpu, dim, precision):
    p = _cloud(dim)
    q = p.copy()
    values = [NAN, -NAN, INF, -INF]
    picks = [(v, k) for v in values for k in ((0,), (1,), (2,), (0, 1), (0, 1, 2))]
    lost = np.random.default_rng(4).choice(len(p), len(picks), replace=False)
    for i, (v, ks) in zip(lost, picks):
        for k in ks:
            q[i, k] = v
    pa, loc, cm, off, idx = _kept_lists(p, q, precision)
    left = np.setdiff1d(np.arange(len(p)), lost)
    d = dict(x=q[left, 0].copy(), y=q[left, 1].copy(), z=q[left, 2].copy(),
             h=np.full(len(left), 0.5))
    roff, ridx = cpu_ref.nnps(d, d, 2.0, cm.cell_size, True)
    counts = np.zeros(len(p), dtype=np.int64)
    counts[left] = np.diff(roff)
    assert np.array_equal(np.diff(off), counts)
    assert np.array_equal(idx, left[ridx])
    pa.set_dirty(True)
    loc.update_status()
    with pytest.raises(_lib.SphError, match="non-finite"):
        loc.update()


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("dim", [2, 3])
def test_particles_outside_a_kept_grid(gpu, dim, precision):
    """Some carried 50 and 2^20 cells out, among them neighbours of each other."""
    p = _cloud(dim)
    q = p.copy()
    out = np.flatnonzero((p[:, 0] < 1.0) & (p[:, 1] < 2.0))
    far = np.flatnonzero((p[:, 0] > 3.5) & (p[:, 1] > 3.0))
    assert len(out) > 20 and len(far) > 5
    q[out, 0] += 50.0
    q[far, 1] -= 2.0 ** 20
    pa, loc, cm, off, idx = _kept_lists(p, q, precision)
    t = np.float64 if precision == "double" else np.float32
    a = q.astype(t)
    d2 = sum((a[:, None, k] - a[None, :, k]) ** 2 for k in range(3))
    near = d2 < t(1.0)
    for i in range(len(p)):
        row = idx[off[i]:off[i + 1]]
        assert row[-1] == i
        assert np.array_equal(np.sort(row), np.flatnonzero(near[i])), i
    pa.set_dirty(True)
    loc.update_status()
    with pytest.raises(_lib.SphError, match="outside the cell grid"):
        loc.update()


@pytest.mark.parametrize("precision", ["double", "single"])
def test_radius_far_above_the_cells(gpu, precision):
    """A cell size clamped to 1e-16 of the radius: the reach is bounded and
    everyone is a neighbour."""
    from pysph_amd.base import api as base
    from pysph_amd.base.nnps import CellManager, NNPSManager
    p = _cloud(3, n=50, side=2)
    pa = base.get_particle_array(name="f", cl_precision=precision, x=p[:, 0].copy(),
                                 y=p[:, 1].copy(), z=p[:, 2].copy(), h=np.full(len(p), 1e16))
    cm = CellManager(arrays_to_bin=[pa], radius_scale=2.0, precision=precision,
                     max_cell_size=1.0)
    loc = NNPSManager(cell_manager=cm).get_neighbor_particle_locator(pa, pa, 2.0)
    for again in range(2):
        off, idx = (t.cpu().numpy() for t in loc.get_csr())
        assert np.array_equal(np.diff(off), np.full(len(p), len(p)))
        rows = idx.reshape(len(p), len(p))
        assert np.array_equal(rows[:, -1], np.arange(len(p)))
        assert np.array_equal(np.sort(rows, axis=1), np.tile(np.arange(len(p)), (len(p), 1)))
        pa.set_dirty(True)
        loc.update_status()


@pytest.mark.parametrize("precision,power", [("double", -200), ("double", -131), ("double", 131),
                                             ("double", 200), ("single", -70), ("single", 66)])
def test_cells_near_the_ends_of_the_float_range(gpu, precision, power):
    """The rows of the distance test in its own precision: at 2^-70 the float
    squares lose digits, at 2^66 the squared radius overflows."""
    from pysph_amd.base import api as base
    from pysph_amd.base.nnps import CellManager, NNPSManager
    t = np.float64 if precision == "double" else np.float32
    p = _cloud(3, n=300, side=2) * 2.0 ** power
    d = dict(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(),
             h=np.full(len(p), 0.5 * 2.0 ** power))
    pa = base.get_particle_array(name="f", cl_precision=precision, **d)
    cm = CellManager(arrays_to_bin=[pa], radius_scale=2.0, precision=precision)
    loc = NNPSManager(cell_manager=cm).get_neighbor_particle_locator(pa, pa, 2.0)
    a = p.astype(t)
    e = [(a[:, None, k] - a[None, :, k]) for k in range(3)]
    with np.errstate(over="ignore", under="ignore"):
        r = t(2.0 ** power)
        near = e[0] * e[0] + e[1] * e[1] + e[2] * e[2] < r * r
    for again in range(2):
        off, idx = (v.cpu().numpy() for v in loc.get_csr())
        for i in range(len(p)):
            row = idx[off[i]:off[i + 1]]
            assert row[-1] == i
            assert np.array_equal(np.sort(row), np.flatnonzero(near[i])), i
        pa.set_dirty(True)
        loc.update_status()
