"""What the reverse of a whole RK2 step does not take."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_per_simulation_time_steps_are_refused(gpu):
    """The forward step multiplies dt by each simulation's own; the reverse
    knows one dt, and must not return another step's gradient."""
    from pysph_amd import _lib
    from pysph_amd.adjoint import Rollout
    g = np.arange(4) * 0.1
    pos = np.stack(np.meshgrid(g, g, indexing="ij"), -1).reshape(-1, 2)
    n = len(pos)
    roll = Rollout(pos, np.full(n, 0.01), 0.13, nsteps=2, dt=1e-5, checkpoint=2)
    dev = roll.sim.device
    zero, one = (torch.full((n,), v, dtype=torch.float64, device=dev) for v in (0.0, 1.0))
    roll.forward(zero, zero, 0.1)
    assert torch.isfinite(roll.backward(one, zero)[0]).all()
    steps = torch.full((1,), 0.5, dtype=torch.float64, device=dev)
    roll.forward(zero, zero, 0.1)
    roll.sim.desc.dt_sim = steps.data_ptr()
    with pytest.raises(_lib.SphError, match="one time step"):
        roll.backward(one, zero)
    roll.sim.synchronize()
