"""Single precision: density from the compact 16-byte rows against the same sum
from the records, and the scatter that writes both (wide stores where the
destinations are adjacent and aligned) against numpy."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,jitter,two", [(1, 0.0, False), (65, 0.0, True), (5000, 0.0, True),
                                          (5000, 0.2, False)])
def test_density_rows_equal_records(gpu, n, jitter, two):
    from pysph_amd.base import api as base
    from pysph_amd.sph import api as sph
    rng = np.random.default_rng(n)
    side = (n / 50.0) ** (1.0 / 3.0)

    def arr(name, k):
        p = rng.uniform(0.0, side, (k, 3))
        return base.get_particle_array(
            name=name, cl_precision="single", x=p[:, 0].copy(), y=p[:, 1].copy(),
            z=p[:, 2].copy(), h=0.3 * (1.0 + jitter * rng.uniform(-1, 1, k)),
            m=rng.uniform(0.5, 1.5, k))

    arrays = [arr("f", n)] + ([arr("w", n // 3 + 1)] if two else [])
    particles = base.Particles(arrays)
    f = arrays[0]
    f.add_property({"name": "one"})
    f.add_property({"name": "all"})
    kernel = base.CubicSplineKernel(dim=3)
    funcs = [sph.SPHRho.withargs().get_func(a, f) for a in arrays]
    calc = sph.SPHCalc(particles, arrays, f, kernel, funcs, ["all"])
    calc.sph("all")  # the compact rows
    assert particles.cell_manager.posmass(f).dtype == torch.float32
    tmp = [f.get_carray(k) for k in ("one", "_tmpx", "_tmpy")]
    for k, fn in enumerate(funcs):  # one source at a time: the records
        fn.eval(kernel, *tmp, accumulate=k > 0)
        if k == 0:
            f.touch("one")
    assert np.array_equal(f.get("one"), f.get("all"))


@pytest.mark.parametrize("n", [1, 257])
@pytest.mark.parametrize("fields,shift", [
    ((0, 1, 2, 3), 0), ((0, 1, 2, 3), 1), ((0, 1, 2, 3), 2), ((0, 2, 3, 7), 0),
    ((1, 2, 3, 4, 5, 6), 0), ((0,), 0), ((8, 9, 10, 11), 0)])
def test_scatter_float_rows(gpu, n, fields, shift):
    from pysph_amd import _lib
    ctx = _lib.context()
    rng = np.random.default_rng(n + shift)
    src = torch.tensor(rng.normal(size=(len(fields), n)), device="cuda")
    rank = torch.tensor(rng.permutation(n).astype(np.int32), device="cuda")
    rec = torch.zeros(12 * n + 4, dtype=torch.float32, device="cuda")
    pm = torch.zeros(4 * n + 4, dtype=torch.float32, device="cuda")
    a, b = _lib.PropListF32(), _lib.PropListF32()
    a.nprops, a.dst_stride = len(fields), 12
    b.nprops, b.dst_stride = min(4, len(fields)), 4
    for k, q in enumerate(fields):
        a.src[k], a.dst[k] = src[k].data_ptr(), rec.data_ptr() + 4 * (q + shift)
    for k in range(b.nprops):
        b.src[k], b.dst[k] = src[k].data_ptr(), pm.data_ptr() + 4 * (k + shift)
    ctx.check(ctx.lib.sph_scatter_sorted2_f32(ctx.handle, n, rank.data_ptr(), ctypes.byref(a),
                                              ctypes.byref(b)))
    want, wpm = np.zeros(12 * n + 4, np.float32), np.zeros(4 * n + 4, np.float32)
    r, v = rank.cpu().numpy().astype(np.int64), src.cpu().numpy().astype(np.float32)
    for k, q in enumerate(fields):
        want[12 * r + q + shift] = v[k]
        if k < b.nprops:
            wpm[4 * r + k + shift] = v[k]
    assert np.array_equal(rec.cpu().numpy(), want)
    assert np.array_equal(pm.cpu().numpy(), wpm)
