"""The bound of h that a variable-h build takes: the grid's, and a fresh one
when h was written after the binning (rows against the oracle on the binning's
cells) or the grid covers another array with larger h."""
import numpy as np
import pytest

from oracle import cpu_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("factor", [1.0, 0.6, 2.5])
@pytest.mark.parametrize("other", [False, True])
def test_rows_after_writing_h(gpu, factor, other):
    from pysph_amd.base import api as base
    rng = np.random.default_rng(3)
    n = 1500
    p = rng.uniform(0.0, 1.0, (n, 3))
    d = dict(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(),
             h=0.04 * rng.uniform(0.5, 1.5, n))
    pa = base.get_particle_array(name="f", m=np.ones(n), **d)
    arrays = [pa]
    if other:
        q = rng.uniform(0.0, 1.0, (50, 3))
        arrays.append(base.get_particle_array(name="o", x=q[:, 0].copy(), y=q[:, 1].copy(),
                                              z=q[:, 2].copy(), h=np.full(50, 0.2),
                                              m=np.ones(50)))
    particles = base.Particles(arrays, variable_h=True)
    loc = particles.nnps_manager.get_neighbor_particle_locator(pa, pa, 2.0)
    loc.get_csr()
    if factor != 1.0:
        d["h"] = d["h"] * factor
        pa.set(h=d["h"])
    loc.is_dirty = True
    off, idx = (t.cpu().numpy() for t in loc.get_csr())
    want = cpu_ref.nnps_varh(d, d, 2.0, particles.cell_manager.cell_size)
    assert np.array_equal(off, want[0]) and np.array_equal(idx, want[1])
