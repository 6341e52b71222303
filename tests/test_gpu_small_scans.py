"""The one-launch forms of the binning's scan (grids of up to 4 tiles of 4,096
cells) and of the lists' slice offsets (up to 1,024 slices of 64 rows), at the
edges of their ranges and just past them, against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _arrays(n, side, seed):
    from pysph_amd.base import api as base
    rng = np.random.default_rng(seed)
    h = 0.5  # cells of 1.0
    pts = rng.uniform(0.01, side - 0.01, (n, 2))
    pts[0] = 0.01  # the grid spans the box
    pts[-1] = side - 0.01
    return base.get_particle_array(name="f", x=pts[:, 0].copy(), y=pts[:, 1].copy(),
                                   z=np.zeros(n), h=np.full(n, h), m=np.ones(n))


@pytest.mark.parametrize("n,side", [
    (1, 1.0), (63, 8.0), (64, 60.0), (65, 64.0), (4097, 122.0), (4097, 126.0), (65535, 250.0), (65536, 255.0),
    (65537, 258.0), (70000, 300.0)])
@pytest.mark.parametrize("order", ["linear", "morton"])
def test_scans_match_numpy(gpu, n, side, order):
    from pysph_amd.base import api as base
    pa = _arrays(n, side, n)
    particles = base.Particles([pa], cell_order=order)
    cm = particles.cell_manager
    loc = particles.nnps_manager.get_neighbor_particle_locator(pa, pa, 2.0)
    for _ in range(3):  # the first build synchronises, the later ones run on the device
        pa.set_dirty(True)
        particles.update()
        counts, slice_off, _ = (t.cpu().numpy() for t in loc.get_sorted_lists())
        b = cm.bins["f"]
        cell_of, start = b.cell_of.cpu().numpy()[:n], b.cell_start.cpu().numpy()
        per = np.bincount(cell_of, minlength=len(start) - 1)
        assert np.array_equal(start, np.concatenate([[0], np.cumsum(per)]))
        cells = np.flatnonzero(per)
        assert np.array_equal(b.cells.cpu().numpy()[:len(cells)], cells)
        assert np.array_equal(b.perm.cpu().numpy()[:n], np.argsort(cell_of, kind="stable"))
        rows = np.zeros(len(slice_off[1:]) * 64, dtype=np.int64)
        rows[:n] = counts
        rows = rows.reshape(-1, 64)
        assert np.array_equal(slice_off, np.concatenate([[0], np.cumsum(64 * rows.max(1))]))
        assert loc.nnz == rows.sum()


@pytest.mark.parametrize("nf,nw", [(130, 3), (65536, 40), (65600, 200)])
def test_paired_slices_match_numpy(gpu, nf, nw):
    from pysph_amd.base import api as base
    from pysph_amd.base.nnps import update_together
    f, w = _arrays(nf, 40.0, 1), _arrays(nw, 40.0, 2)
    w.set_name("w")
    particles = base.Particles([f, w])
    man = particles.nnps_manager
    locs = [man.get_neighbor_particle_locator(s, f, 2.0) for s in (f, w)]
    for _ in range(3):
        for a in (f, w):
            a.set_dirty(True)
        particles.update()
        update_together(locs)
        for loc in locs:
            rows = np.zeros((nf + 63) // 64 * 64, dtype=np.int64)
            rows[:nf] = loc.counts.cpu().numpy()
            rows = rows.reshape(-1, 64)
            off = loc.slice_off.cpu().numpy()
            assert np.array_equal(off, np.concatenate([[0], np.cumsum(64 * rows.max(1))]))
            assert loc.nnz == rows.sum()
