"""A batch's cell counts are cleared in the bounding-box kernel or, with more
cells than a few blocks clear in passing, by a launch of their own: the same
steps on both sides of that line (32 blocks of 256 threads and 256 cells a
simulation, for one or two of them)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LINE = 32 * 256 * 256


@pytest.mark.parametrize("nsims,key_cap", [(1, LINE - 1), (1, LINE), (1, 4 * LINE + 5),
                                           (2, 2 * LINE - 1), (2, 2 * LINE), (3, 4 * LINE)])
def test_steps_do_not_depend_on_the_key_space(gpu, nsims, key_cap):
    from pysph_amd.batch import BatchedSimulation
    from pysph_amd.solver.generators import elliptical_drop
    sims = [elliptical_drop(dx=0.08 + 0.01 * k, vel=80.0 + k) for k in range(nsims)]
    out = []
    for cap in (None, key_cap):
        b = BatchedSimulation(sims, key_cap=cap)
        assert (b.key_cap == key_cap) == (cap is not None)
        for _ in range(3):
            b.step(1e-5)
        b.check()
        out.append({k: b.get(k) for k in ("x", "y", "u", "v", "rho", "p")})
    for k, v in out[0].items():
        assert np.array_equal(v, out[1][k]), k
