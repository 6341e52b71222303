"""The operators' short square roots and divisions (uniform_h = 2) against
the IEEE ones (uniform_h = 1): the same bits, over the range of h they are
taken for, with coincident and nearly coincident particles and pairs on the
spline's breaks (q = 1 and 2), in 2D and 3D, below and above the size where
the momentum and XSPH launches change form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _particles(dim, h, n, seed=5):
    rng = np.random.default_rng(seed)
    # a lattice of h/2 (pairs at exactly q = 1 and 2 sit in the lists only as
    # far as rounding puts them there), half of it disturbed, and some copies
    # of its points: exactly coincident, and closer than any power of two that
    # matters relative to h
    m = int(round(n ** (1.0 / dim)))
    g = np.arange(m) * 0.5
    p = np.stack(np.meshgrid(*([g] * dim), indexing="ij"), -1).reshape(-1, dim)
    p = np.concatenate([p, np.zeros((len(p), 3 - dim))], 1)
    k = len(p) // 2
    p[:k, :dim] += rng.uniform(-0.2, 0.2, (k, dim))
    same = p[rng.integers(0, len(p), 40)].copy()
    near = p[rng.integers(0, len(p), 40)].copy()
    near[:, 0] += np.float64(2.0) ** rng.integers(-52, -20, 40)
    origin = np.zeros((4, 3))
    origin[:, 0] = [0.0, 1e-320, 2.0 ** -300, 2.0 ** -700]
    p = np.concatenate([p, same, near, origin]) * h
    n = len(p)
    d = dict(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(), h=np.full(n, h),
             m=rng.uniform(0.5, 1.5, n), rho=rng.uniform(0.9, 1.1, n),
             p=rng.uniform(-1.0, 1.0, n), cs=rng.uniform(9.0, 11.0, n))
    for k in ("u", "v") + (("w",) if dim == 3 else ()):
        d[k] = rng.normal(0.0, 1.0, n)
    return d


def _results(dim, d, monkeypatch, mode):
    from pysph_amd.base import api as base
    from pysph_amd.base.nnps import CellManager
    from pysph_amd.sph import api as sph
    took, h_mode = [], CellManager.h_mode

    def told(self):
        took.append(h_mode(self))
        return min(took[-1], mode)
    monkeypatch.setattr(CellManager, "h_mode", told)
    pa = base.get_particle_array(name="f", **d)
    for k in ("ax", "ay", "az", "dt_fac"):
        pa.add_property({"name": k})
    particles = base.Particles([pa])
    kernel = base.CubicSplineKernel(dim=dim)
    out = {}
    calls = [("rho2", sph.SPHRho.withargs(), ("ax",)),
             ("rate", sph.SPHDensityRate.withargs(), ("ax",)),
             ("mom", sph.MomentumEquation.withargs(alpha=0.3, beta=0.2), ("ax", "ay", "az")),
             ("xsph", sph.XSPHCorrection.withargs(eps=0.5), ("ax", "ay", "az")),
             ("pgrad", sph.SPHPressureGradient.withargs(), ("ax", "ay", "az")),
             ("avisc", sph.MonaghanArtificialViscosity.withargs(alpha=0.3, beta=0.2),
              ("ax", "ay", "az"))]
    for name, f, props in calls:
        calc = sph.SPHCalc(particles, [pa], pa, kernel, [f.get_func(pa, pa)], list(props))
        calc.sph(*props)
        out[name] = np.concatenate([pa.get(k) for k in props])
    out["dt_fac"] = pa.get("dt_fac")
    monkeypatch.undo()
    return out, took


@pytest.mark.parametrize("dim,h,n,mode", [
    (2, 1.0, 900, 2), (3, 1.0, 1700, 2), (3, 0.013, 1700, 2), (2, 2.0 ** -99, 900, 2),
    (2, 2.0 ** 99, 900, 2), (2, 2.0 ** -101, 400, 1), (3, 1.0, 280000, 2)])
def test_same_bits_as_the_ieee_forms(gpu, monkeypatch, dim, h, n, mode):
    d = _particles(dim, h, n)
    want, _ = _results(dim, d, monkeypatch, 1)
    got, took = _results(dim, d, monkeypatch, 2)
    assert took == [mode] * 6
    for k in want:
        assert np.array_equal(want[k], got[k]), k
        assert np.isfinite(got[k]).all() or h < 2.0 ** -90 or h > 2.0 ** 90, k
