"""Discrete adjoint of one explicit Runge-Kutta step of the residual, for the
gradient of a wall force with respect to the state and the wall shape.

Problem (codens_amd.configs.adjoint_wall): one curvilinear viscous block,
laminar Navier-Stokes, Roe flux with unlimited MUSCL, wall and far-field
ghosts.  With u(v; sn, vol) the residual of sch_roe (net outgoing flux of
every real cell after zpres, zvismo, the ghosts and zvisqc), the step is the
4-stage scheme

    v_s = v_0 - alpha_s (dt / vol) u(v_{s-1}),   alpha = 1/4, 1/3, 1/2, 1,

with the local steps dt of chronos at the initial state held fixed, and the
objective is the x force of the wall pressure, J = sum over the j = 1 faces
of p(v_4) S_x (the pressure of the wall ghost, clpara.f90, is that of the
adjacent cell).  The mesh moves through the normal (y) displacement delta of
a seeded set of wall nodes; the far-field normals stay those of the
undisplaced mesh.

Pieces, each a torch.autograd.Function over the C-ABI:

* Residual: forward = the production kernels (codens_zpres, codens_zvismo,
  codens_bc_wall, codens_bc_farfield, codens_zvisqc, codens_bc_tq_copy,
  codens_sch_roe); backward = codens_adj_residual_vjp; jvp =
  codens_adj_residual_jvp.
* Metrics: forward = the mesh metrics of the displaced nodes on the device
  (codens_mesh_metrics: extmhg ghost nodes, norm.f90, svol.f90); backward =
  codens_adj_metric_vjp plus the transposed ghost-node extrapolation; jvp =
  exact polynomial differences of the metrics (sn is bilinear and vol cubic
  in the nodes, so a central difference is exact for sn and a Richardson
  pair of central differences is exact for vol).

torch.autograd keeps the four stage states v_0..v_3 (and the mesh metrics)
as the checkpoints of the reverse sweep.
"""
from __future__ import annotations

import numpy as np
import torch

from . import abi
from . import layout as L
from .solver import Solver

RK_ALPHA = (0.25, 1.0 / 3.0, 0.5, 1.0)


def _dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device="cuda")


def _fold_ghost_nodes(b: L.Block, bar: np.ndarray) -> np.ndarray:
    """Transpose of layout.extrapolate_ghost_nodes on a [k, j, i] view:
    adjoints of the ghost nodes added to the nodes they copy, in the reverse
    order of the copies (j layers, then i layers, then k layers).  A numpy
    array or a torch tensor."""
    a = bar.clone() if isinstance(bar, torch.Tensor) else bar.copy()
    i1, i2, j1, j2 = b.ii1 - b.id1, b.ii2 - b.id1, b.jj1 - b.jd1, b.jj2 - b.jd1
    k1, k2 = b.kk1 - b.kd1, b.kk2 - b.kd1
    a[:, j1, :] += a[:, j1 - 1, :]; a[:, j1 - 1, :] = 0.
    a[:, j2, :] += a[:, j2 + 1, :]; a[:, j2 + 1, :] = 0.
    a[:, j1:j2 + 1, i1] += a[:, j1:j2 + 1, i1 - 1]; a[:, j1:j2 + 1, i1 - 1] = 0.
    a[:, j1:j2 + 1, i2] += a[:, j1:j2 + 1, i2 + 1]; a[:, j1:j2 + 1, i2 + 1] = 0.
    a[k1, j1:j2 + 1, i1:i2 + 1] += a[k1 - 1, j1:j2 + 1, i1:i2 + 1]; a[k1 - 1, j1:j2 + 1, i1:i2 + 1] = 0.
    a[k2, j1:j2 + 1, i1:i2 + 1] += a[k2 + 1, j1:j2 + 1, i1:i2 + 1]; a[k2 + 1, j1:j2 + 1, i1:i2 + 1] = 0.
    return a


class AdjointProblem:
    """Buffers, boundary lists and frozen data of the differentiated step."""

    def __init__(self, case):
        if case.scheme.get("ilim", 0) != 0 or not case.ns or len(case.layout.blocks) != 1:
            raise ValueError("the adjoint covers one viscous block with unlimited MUSCL (ilim = 0)")
        self.case = case
        self.lay = case.layout
        self.b = self.lay.blocks[0]
        self.blk = abi.block(self.b)
        self.ph = abi.phys(**case.phys)
        self.sc = abi.scheme(**case.scheme)
        self.S = Solver(case)
        i64 = lambda a: _dev(a, torch.int64)
        w, fa = case.wall, case.farfield
        self.bcs = (i64(w.ghost), i64(w.inner), i64(fa.ghost), i64(fa.inner), _dev(fa.normals))
        self.winf = _dev(case.winf)
        n = self.lay.ip11
        self.real = torch.zeros(n, dtype=torch.float64, device="cuda")
        self.real[_dev(self.lay.interior(), torch.int64)] = 1.0
        # frozen local steps of the initial state (chronos)
        self.S.thermo()
        self.S.time_step()
        self.dt = self.S.dt.clone()
        self.x0, self.y0, self.z0 = (np.ascontiguousarray(a).copy() for a in case.nodes)
        self.xyz0 = tuple(_dev(a) for a in (self.x0, self.y0, self.z0))
        self.wall_nodes = np.asarray(case.wall_nodes)
        self.wall_nodes_d = i64(self.wall_nodes)
        self.wall_local = i64(self.wall_nodes - self.b.npc)
        self.wall_cells = i64(w.inner)
        self.wall_sx = i64(self.b.nnn + (w.inner - self.b.npc))  # sn(m, d = j, c = x) of the wall faces
        self.sg = self._orientation()

    def _orientation(self):
        """+-0.5 of each face family, as norm.f90's orientation test gives."""
        b, sn = self.b, self.case.sn
        X, Y, Z = b.view(self.x0), b.view(self.y0), b.view(self.z0)
        k, j, i = b.kk1 - b.kd1, b.jj1 - b.jd1, b.ii1 - b.id1
        P = lambda di, dj, dk: np.array([A[k + dk, j + dj, i + di] for A in (X, Y, Z)])
        diag = {2: ((1, 1, 0), (0, 1, 0), (1, 0, 0)), 1: ((1, 0, 1), (0, 0, 1), (1, 0, 0)),
                0: ((0, 1, 1), (0, 0, 1), (0, 1, 0))}
        m = (k * b.njd + j) * b.nid + i
        out = []
        for d in range(3):
            e1, e2, e3 = diag[d]
            t = np.cross(P(*e1) - P(0, 0, 0), P(*e2) - P(*e3))
            s = np.array([sn[9 * b.npc + (c * 3 + d) * b.nnn + m] for c in range(3)])
            out.append(0.5 if float(np.dot(s, t)) > 0 else -0.5)
        return out

    # -- mesh ----------------------------------------------------------------
    def nodes(self, delta):
        """Node coordinates with the wall nodes moved by delta (y only), as
        fresh device arrays."""
        x, y, z = (a.clone() for a in self.xyz0)
        y.index_add_(0, self.wall_nodes_d, torch.as_tensor(delta, dtype=torch.float64, device="cuda"))
        return x, y, z

    def metrics(self, delta):
        """(sn of the block (9 nnn), vol (ip11), the nodes with their ghost
        layer) of the mesh moved by delta, on the device."""
        x, y, z = self.nodes(delta)
        sn = torch.empty(9 * self.b.nnn, dtype=torch.float64, device="cuda")
        vol = torch.zeros(self.lay.ip11, dtype=torch.float64, device="cuda")
        abi.mesh_metrics(self.blk, x, y, z, sn, vol)
        return sn, vol, (x, y, z)

    def metric_jvp(self, delta, ddot):
        """Exact derivative of (sn, vol) along the wall displacement ddot."""
        sp, vp, _ = self.metrics(delta + ddot)
        sm, vm, _ = self.metrics(delta - ddot)
        _, vh, _ = self.metrics(delta + 0.5 * ddot)
        _, vl, _ = self.metrics(delta - 0.5 * ddot)
        snd = 0.5 * (sp - sm)
        d1 = 0.5 * (vp - vm)
        d2 = vh - vl
        return snd, (4.0 * d2 - d1) / 3.0

    def metric_vjp(self, snbar, volbar, xyz):
        """(snbar, volbar) -> adjoint of the wall displacements, at the nodes
        xyz (with their ghost layer) the metrics were formed from."""
        nnn = self.b.nnn
        bars = [torch.empty(nnn, dtype=torch.float64, device="cuda") for _ in range(3)]
        abi.adj_metric_vjp(self.blk, *xyz, self.sg, snbar.contiguous(), volbar.contiguous(), *bars)
        yb = _fold_ghost_nodes(self.b, bars[1].view(self.b.nkd, self.b.njd, self.b.nid))
        return yb.reshape(-1)[self.wall_local]

    # -- residual ------------------------------------------------------------
    def residual(self, v, sn_blk, vol):
        """u(v) of the production kernels (real cells; zero elsewhere), a copy
        that later calls of the solver leave alone."""
        S = self.S
        S.v.copy_(v)
        S.sn_blk = [sn_blk.contiguous()]
        S.vol = vol.contiguous()
        S.thermo()
        S.ghosts()
        S.stresses()
        S.residual()
        return S.u[:5].clone()

    def jvp(self, v, sn_blk, vol, vd, snd, vold):
        z = lambda t, like: torch.zeros_like(like) if t is None else t.contiguous()
        u = torch.zeros_like(v[:5]); ud = torch.zeros_like(v[:5])
        abi.adj_residual_jvp(self.blk, self.ph, self.sc, v.contiguous(), z(vd, v), sn_blk.contiguous(),
                             z(snd, sn_blk), vol.contiguous(), z(vold, vol), self.winf, self.bcs, u, ud)
        return u, ud

    def vjp(self, v, sn_blk, vol, ubar):
        # the call overwrites every entry of a one-block layout (planes past
        # the fifth aside) and reads 5 x ip11 doubles of ubar, on the real cells
        ub = ubar[:5]
        if ub.shape != (5, v.shape[-1]) or ub.dtype != torch.float64 or not ub.is_contiguous():
            ub = torch.empty((5, v.shape[-1]), dtype=torch.float64, device=v.device).copy_(ub)
        vb = torch.empty_like(v, memory_format=torch.contiguous_format)
        vb[5:] = 0.
        snb = torch.empty_like(sn_blk, memory_format=torch.contiguous_format)
        volb = torch.empty_like(vol, memory_format=torch.contiguous_format)
        abi.adj_residual_vjp(self.blk, self.ph, self.sc, v.contiguous(), sn_blk.contiguous(), vol.contiguous(),
                             self.winf, self.bcs, ub, vb[:5], snb, volb)
        return vb, snb, volb

    # -- the step and the objective -----------------------------------------
    def rk_step(self, v0, sn_blk, vol):
        c = torch.where(self.real > 0, self.dt / torch.where(self.real > 0, vol, torch.ones_like(vol)),
                        torch.zeros_like(vol))
        v = v0
        for a in RK_ALPHA:
            u = Residual.apply(v, sn_blk, vol, self)
            v = torch.addcmul(v0, c, u, value=-a)
        return v

    def objective(self, v, sn_blk):
        w = v[:, self.wall_cells]
        p = self.ph.gam1 * (w[4] - 0.5 * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]) / w[0] - self.ph.pinfl)
        return (p * sn_blk[self.wall_sx]).sum()

    def J(self, v0, delta):
        """Objective of the step from v0 on the mesh with wall displacement
        delta (torch tensors; differentiable in both)."""
        sn_blk, vol = Metrics.apply(delta, self)
        return self.objective(self.rk_step(v0, sn_blk, vol), sn_blk)

    def J_value(self, v0, delta):
        """Forward only, for finite differences (production kernels, device
        metrics); delta a numpy array or a device tensor."""
        with torch.no_grad():
            sn_blk, vol, _ = self.metrics(delta)
            return float(self.objective(self.rk_step(v0, sn_blk, vol), sn_blk))


class Residual(torch.autograd.Function):
    @staticmethod
    def forward(ctx, v, sn_blk, vol, prob):
        ctx.prob = prob
        ctx.save_for_backward(v, sn_blk, vol)
        ctx.save_for_forward(v, sn_blk, vol)
        return prob.residual(v, sn_blk, vol)

    @staticmethod
    def backward(ctx, ubar):
        v, sn_blk, vol = ctx.saved_tensors
        vb, snb, volb = ctx.prob.vjp(v, sn_blk, vol, ubar)
        return vb, snb, volb, None

    @staticmethod
    def jvp(ctx, vd, snd, vold, _):
        v, sn_blk, vol = ctx.saved_tensors
        _, ud = ctx.prob.jvp(v, sn_blk, vol, vd, snd, vold)
        return ud


class Metrics(torch.autograd.Function):
    @staticmethod
    def forward(ctx, delta, prob):
        d = delta.detach()
        sn, vol, xyz = prob.metrics(d)
        ctx.prob = prob
        ctx.delta = d
        ctx.xyz = xyz
        return sn, vol

    @staticmethod
    def backward(ctx, snbar, volbar):
        prob = ctx.prob
        if snbar is None:
            snbar = torch.zeros(9 * prob.b.nnn, dtype=torch.float64, device="cuda")
        if volbar is None:
            volbar = torch.zeros(prob.lay.ip11, dtype=torch.float64, device="cuda")
        return prob.metric_vjp(snbar, volbar, ctx.xyz), None

    @staticmethod
    def jvp(ctx, ddot, _):
        return ctx.prob.metric_jvp(ctx.delta, ddot.detach())


def gradient(prob: AdjointProblem, v0, delta):
    """(dJ/dv0, dJ/ddelta) by the reverse sweep."""
    v = v0.detach().clone().requires_grad_(True)
    d = delta.detach().clone().requires_grad_(True)
    J = prob.J(v, d)
    gv, gd = torch.autograd.grad(J, [v, d])
    return float(J.detach()), gv, gd


def directional(prob: AdjointProblem, v0, delta, vdir, ddir):
    """dJ along (vdir, ddir) by the tangent-linear sweep (forward mode)."""
    import torch.autograd.forward_ad as fwAD
    with fwAD.dual_level():
        v = fwAD.make_dual(v0.detach(), vdir)
        d = fwAD.make_dual(delta.detach(), ddir)
        J = prob.J(v, d)
        return float(fwAD.unpack_dual(J).tangent)
