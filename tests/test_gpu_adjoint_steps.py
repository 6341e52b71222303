"""The reverse of whole RK2 steps (sph_batch_rk2_vjp over the evaluations of
sph_batch_rk2_step_kept, the last segment kept from the forward pass) against
the same reverse composed of single evaluations (sph_batch_eval and
sph_batch_vjp), and the 3D kernels against torch.autograd."""
import ctypes

import numpy as np
import pytest
import torch

from tests import sph_torch_ref as ref

pytestmark = pytest.mark.gpu


def _block(dim, n, seed):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / dim)))
    g = np.stack(np.meshgrid(*([np.arange(m) * 0.1] * dim), indexing="ij"), -1)
    pos = (g.reshape(-1, dim)[:n] + rng.uniform(-0.02, 0.02, (n, dim)))
    vel = rng.normal(0.0, 5.0, (n, dim))
    return pos, vel, np.full(n, 0.1 ** dim), 0.13


def _composed(roll, vel, alpha, bars, nsteps, dt):
    """The reverse with one evaluation per call: every state kept, evaluations
    recomputed one at a time, cotangents combined by torch."""
    s, d, n = roll.sim, roll.dim, roll.n
    keys = roll._state_keys()
    call = roll._call

    def eval_at(x):
        for q in keys:
            s.t[q].copy_(x[q])
        call("sph_batch_eval")

    def vjp(fbar):
        out = {q: torch.zeros(n, dtype=torch.float64, device=s.device) for q in keys}
        al = torch.zeros(1, dtype=torch.float64, device=s.device)
        p = [fbar[q].data_ptr() for q in keys[d:]] + [None] * (3 - d)
        x = [out[q].data_ptr() for q in keys[:d]] + [None] * (3 - d)
        u = [out[q].data_ptr() for q in keys[d:]] + [None] * (3 - d)
        call("sph_batch_vjp", *p, *x, *u, al.data_ptr())
        for c in range(d):
            out[keys[d + c]] = out[keys[d + c]] + fbar[keys[c]]
        return out, al

    s.stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s.stream):
        x0 = {q: (roll.pos0[q] if q in roll.pos0 else vel[keys.index(q) - d].clone())
              for q in keys}
        starts, mids = [], []
        for q in keys:
            s.t[q].copy_(x0[q])
        for _ in range(nsteps):
            starts.append({q: s.t[q].clone() for q in keys})
            call("sph_batch_save_initial")
            call("sph_batch_eval")
            call("sph_batch_stage", dt / 2)
            mids.append({q: s.t[q].clone() for q in keys})
            call("sph_batch_eval")
            call("sph_batch_stage", dt)
        final = [s.t[q].clone() for q in keys[:d]]
        bar = {q: torch.zeros(n, dtype=torch.float64, device=s.device) for q in keys}
        for c in range(d):
            bar[keys[c]].copy_(bars[c])
        total = torch.zeros(1, dtype=torch.float64, device=s.device)
        for k in reversed(range(nsteps)):
            eval_at(mids[k])
            x1, al = vjp({q: dt * bar[q] for q in keys})
            total += al
            eval_at(starts[k])
            x2, al = vjp({q: (0.5 * dt) * x1[q] for q in keys})
            total += al
            bar = {q: bar[q] + x1[q] + x2[q] for q in keys}
    s.check()
    return final, [bar[q] for q in keys[d:]] + [total]


@pytest.mark.parametrize("dim,n,nsteps,checkpoint", [
    (2, 1, 2, 2), (2, 33, 7, 3), (2, 257, 6, 3), (3, 500, 5, 8), (3, 31, 4, 1)])
def test_steps_match_single_evaluations(gpu, dim, n, nsteps, checkpoint):
    from pysph_amd.adjoint import Rollout
    dt = 1e-5
    pos, vel, m, h = _block(dim, n, 3 + n)
    roll = Rollout(pos, m, h, nsteps=nsteps, dt=dt, checkpoint=checkpoint, dim=dim, beta=0.1)
    dev = roll.sim.device
    v = [torch.tensor(vel[:, c], device=dev) for c in range(dim)]
    bars = [torch.linspace(-1, 1, n, dtype=torch.float64, device=dev) * (c + 1)
            for c in range(dim)]
    out = roll.forward(v[0], v[1], 0.2, w0=v[2] if dim == 3 else None)
    got = roll.backward(*bars)
    again = roll.backward(*bars)  # the last segment recomputed this time
    final, want = _composed(roll, v, 0.2, bars, nsteps, dt)
    # the same operations in the same order throughout
    for a, b in zip(out, final):
        assert torch.equal(a, b)
    for a, b, c in zip(got, want, again):
        assert torch.equal(a.reshape(-1), b.reshape(-1))
        assert torch.equal(a, c)


@pytest.mark.parametrize("n", [60, 343])
def test_vjp_3d_matches_torch_autograd(gpu, n):
    from pysph_amd.batch import BatchedSimulation
    pos, vel, m, h = _block(3, n, n)
    d = dict(x=pos[:, 0], y=pos[:, 1], z=pos[:, 2], u=vel[:, 0], v=vel[:, 1], w=vel[:, 2],
             m=m, h=np.full(n, h), rho=np.ones(n), p=np.zeros(n), cs=np.full(n, 1400.0))
    sim = BatchedSimulation([d], dim=3, alpha=0.3, beta=0.2)
    sim.ctx.check(sim.ctx.lib.sph_batch_eval(sim.ctx.handle, ctypes.byref(sim.desc)))
    abar = torch.tensor(np.random.default_rng(4).normal(0.0, 1.0, (3, n)), device=sim.device)
    out = torch.zeros((6, n), dtype=torch.float64, device=sim.device)
    al = torch.zeros(1, dtype=torch.float64, device=sim.device)
    sim.stream.wait_stream(torch.cuda.current_stream())
    sim.ctx.check(sim.ctx.lib.sph_batch_vjp(
        sim.ctx.handle, ctypes.byref(sim.desc), *[abar[c].data_ptr() for c in range(3)],
        *[out[c].data_ptr() for c in range(6)], al.data_ptr()))
    sim.check()
    tp, tv = (torch.tensor(a, requires_grad=True) for a in (pos, vel))
    alpha = torch.tensor(0.3, dtype=torch.float64, requires_grad=True)
    pairs = ref.pairs_bruteforce(*pos.T[:2], h, z=pos[:, 2])
    acc, _, _ = ref.accelerations(tp, tv, torch.tensor(m), h, pairs, alpha, beta=0.2)
    gx, gu, ga = torch.autograd.grad(acc, (tp, tv, alpha), grad_outputs=abar.cpu().T)
    # the bound of the 2D comparison
    for got, want in ((out[:3].T, gx), (out[3:].T, gu), (al, ga.reshape(1))):
        assert float((got.cpu() - want).abs().max()) <= 1e-9 * float(want.abs().max())
