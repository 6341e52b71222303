"""Reverse mode of a simulation rollout, for fitting initial velocities or the
artificial viscosity to a target end state.

``Rollout`` advances one simulation (the same kernels as the batched path:
SPHRho, Tait, MomentumEquation + Monaghan viscosity, PositionStepping, RK2
of solver/integrator.py:467-498) for ``nsteps`` steps, keeping the positions
and velocities every ``checkpoint`` steps, and each evaluation's neighbour
lists and sorted records in the last segment.  ``Rollout.backward`` walks the
segments in reverse: it recomputes a segment from its checkpoint (all but the
one whose evaluations are kept), keeping them likewise, and then applies the
hand-written vector-Jacobian kernels (``sph_batch_rk2_vjp``) over those frozen
lists, step by step.  For RK2, X1 = X0 + dt/2 F(X0), X2 = X0 + dt F(X1):

    X1bar = J_F(X1)^T (dt X2bar);  X0bar = X2bar + X1bar + J_F(X0)^T (dt/2 X1bar)

``rollout`` wraps this in a ``torch.autograd.Function`` so that the final
positions are differentiable with respect to the initial velocities and
alpha.  The stage arithmetic x0 + a*dt is differentiated as exact; the
neighbour lists are piecewise constant in the positions (the kernel and its
gradient vanish at the support radius), so they are held fixed.
"""
import ctypes

import numpy as np
import torch

from .batch import BatchedSimulation


class Rollout:
    """One simulation of n particles (2D or 3D) with fixed physics except
    alpha; initial positions fixed, initial velocities and alpha free."""

    def __init__(self, pos, m, h, nsteps, dt, checkpoint=20, dim=2, co=1400.0, ro=1.0,
                 gamma=7.0, beta=0.0, eta=0.1, device=None):
        pos = np.asarray(pos, dtype=np.float64)
        n = pos.shape[0]
        self.n, self.dim = n, dim
        self.nsteps, self.dt = int(nsteps), float(dt)
        self.checkpoint = max(1, int(checkpoint))
        d = dict(x=pos[:, 0], y=pos[:, 1], z=pos[:, 2] if dim == 3 else np.zeros(n),
                 h=np.broadcast_to(np.asarray(h, dtype=np.float64), (n,)).copy(),
                 m=np.broadcast_to(np.asarray(m, dtype=np.float64), (n,)).copy(),
                 rho=np.full(n, ro), p=np.zeros(n), cs=np.full(n, co))
        if np.ptp(d["h"]) != 0.0:
            raise NotImplementedError("the reverse mode needs one h for all particles")
        self.sim = BatchedSimulation([d], dim=dim, co=co, ro=ro, gamma=gamma, alpha=0.0,
                                     beta=beta, eta=eta, device=device)
        s = self.sim
        with torch.cuda.stream(s.stream):
            self.pos0 = {k: s.t[k].clone() for k in ("x", "y", "z")}
            # one workspace per evaluation of a segment (lists + records kept)
            nb = s.work.numel()
            self.seg_work = [torch.empty(nb, dtype=torch.uint8, device=s.device)
                             for _ in range(2 * self.checkpoint)]
        self.main_work = (s.desc.work, s.desc.work_bytes)
        for wk in self.seg_work:
            self._use(wk)
            self._call("sph_batch_init_workspace")
        self._use(None)
        self.checkpoints = []
        self.kept = None  # the segment whose evaluations seg_work holds
        self.alpha = 0.0

    # -- pieces ---------------------------------------------------------
    def _call(self, name, *args):
        s = self.sim
        s.ctx.check(getattr(s.ctx.lib, name)(s.ctx.handle, ctypes.byref(s.desc), *args))

    def _use(self, work):
        if work is None:
            self.sim.desc.work, self.sim.desc.work_bytes = self.main_work
        else:
            self.sim.desc.work, self.sim.desc.work_bytes = work.data_ptr(), work.numel()

    def _state_keys(self):
        return ("x", "y", "z", "u", "v", "w") if self.dim == 3 else ("x", "y", "u", "v")

    def _set_initial(self, u0, v0, w0, alpha):
        s = self.sim
        with torch.cuda.stream(s.stream):
            for k in ("x", "y", "z"):
                s.t[k].copy_(self.pos0[k])
            s.t["u"].copy_(u0)
            s.t["v"].copy_(v0)
            if w0 is not None:
                s.t["w"].copy_(w0)
        self.alpha = float(alpha)
        s.desc.alpha = self.alpha

    def _step(self, j=None):
        """One RK2 step; with j, its evaluations are kept in the workspaces of
        step j of a segment."""
        if j is None:
            self._call("sph_batch_rk2_step", self.dt)
            return
        self._use(self.seg_work[2 * j])
        self._call("sph_batch_rk2_step_kept", self.dt, self.seg_work[2 * j + 1].data_ptr())
        self._use(None)

    # -- forward / backward ---------------------------------------------
    def forward(self, u0, v0, alpha, w0=None):
        """Final positions (device tensors) from initial velocities u0, v0
        (w0 in 3D) and alpha; keeps the checkpoints for backward."""
        s = self.sim
        s.stream.wait_stream(torch.cuda.current_stream(s.device))
        self._set_initial(u0, v0, w0, alpha)
        self.checkpoints, self.kept = [], None
        keys = self._state_keys()
        last = (self.nsteps - 1) // self.checkpoint
        for k in range(self.nsteps):
            seg, j = divmod(k, self.checkpoint)
            if j == 0:
                with torch.cuda.stream(s.stream):
                    self.checkpoints.append({q: s.t[q].clone() for q in keys})
            # the last segment is the first that backward needs: keep it now
            self._step(j if seg == last else None)
        s.check()
        self.kept = last
        with torch.cuda.stream(s.stream):
            out = tuple(s.t[q].clone() for q in keys[:self.dim])
        s.synchronize()
        return out

    def backward(self, *pos_bar):
        """Gradients of sum(pos_bar . final positions) with respect to the
        initial velocities (one tensor per component) and alpha."""
        s = self.sim
        s.stream.wait_stream(torch.cuda.current_stream(s.device))
        keys = self._state_keys()
        d = self.dim
        with torch.cuda.stream(s.stream):  # every tensor op below is ordered with the kernels
            # adjoints of the state, one row per component in the order of keys
            bar = torch.zeros((2 * d, self.n), dtype=torch.float64, device=s.device)
            for c in range(d):
                bar[c].copy_(pos_bar[c])
            x1bar = torch.empty_like(bar)
            alpha_total = torch.zeros(1, dtype=torch.float64, device=s.device)
            for seg in reversed(range(len(self.checkpoints))):
                first = seg * self.checkpoint
                nseg = min(self.checkpoint, self.nsteps - first)
                if self.kept != seg:
                    self.kept = None
                    for q in keys:
                        s.t[q].copy_(self.checkpoints[seg][q])
                    for j in range(nseg):
                        self._step(j)
                    self.kept = seg
                for j in reversed(range(nseg)):
                    # X1bar = J_F(X1)^T (dt X2bar);  X0bar = X2bar + X1bar + J_F(X0)^T (dt/2 X1bar)
                    self._use(self.seg_work[2 * j])
                    self._call("sph_batch_rk2_vjp", self.dt, self.seg_work[2 * j + 1].data_ptr(),
                               bar.data_ptr(), x1bar.data_ptr(), alpha_total.data_ptr())
                    self._use(None)
            res = tuple(bar[d + c].clone() for c in range(d)) + (alpha_total,)
        s.check()
        return res


class _RolloutFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, roll, alpha, *vel0):
        out = roll.forward(*[v.detach() for v in vel0[:2]], float(alpha),
                           w0=vel0[2].detach() if len(vel0) > 2 else None)
        ctx.roll = roll
        return out

    @staticmethod
    def backward(ctx, *pos_bar):
        pos_bar = [g if g is not None else torch.zeros(ctx.roll.n, dtype=torch.float64,
                                                       device=ctx.roll.sim.device)
                   for g in pos_bar]
        res = ctx.roll.backward(*pos_bar)
        vel_bar, alpha_bar = res[:-1], res[-1]
        return (None, alpha_bar.reshape(())) + tuple(vel_bar)


def rollout(roll, alpha, *vel0):
    """Differentiable final positions: rollout(roll, alpha, u0, v0[, w0])."""
    return _RolloutFn.apply(roll, alpha, *vel0)
