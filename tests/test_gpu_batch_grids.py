"""The grids of a batch at the number of simulations where they change from one
launch to two, and past one wavefront of them: every simulation of a batch
against the same simulation alone, empty ones included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _drop(k):
    from pysph_amd.solver.generators import elliptical_drop
    if k % 7 == 3:
        e = np.zeros(0)
        return dict(x=e, y=e, u=e, v=e, h=e, m=e, rho=e, cs=e)
    d = elliptical_drop(dx=0.1 + 0.01 * (k % 3), radius=0.3 + 0.05 * (k % 5), vel=60.0 + k)
    return {q: np.asarray(v)[:1] if k % 7 == 5 else np.asarray(v) for q, v in d.items()
            if np.ndim(v) == 1}


@pytest.mark.parametrize("nsims", [2, 15, 16, 17, 70])
def test_batch_equals_single_simulations(gpu, nsims):
    from pysph_amd.batch import BatchedSimulation
    sims = [_drop(k) for k in range(nsims)]
    both = BatchedSimulation(sims)
    both.step(1e-5)
    both.check()
    got = {q: both.get(q) for q in ("x", "y", "u", "v", "rho", "p")}
    off = both.sim_off_host
    for k in {0, 3, 5, nsims // 2, nsims - 1} & set(range(nsims)):
        if len(sims[k]["x"]) == 0:
            continue
        one = BatchedSimulation([sims[k]])
        one.step(1e-5)
        one.check()
        for q, v in got.items():
            assert np.array_equal(v[off[k]:off[k + 1]], one.get(q)), (k, q)
