"""The adjoint of the block residual where its inputs are not those of a plain
gradient call: a solver used between the forward and the reverse sweep."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def problem(dims=(7, 6, 5), **phys):
    from codens_amd import configs
    from codens_amd.adjoint import AdjointProblem
    case = configs.adjoint_wall(*dims, nwall_nodes=6)
    case.phys.update(phys)
    return AdjointProblem(case), case


def test_solver_used_before_backward():
    """The saved residuals are the forward sweep's, whatever the solver
    computes afterwards, and its own buffer stays where it is."""
    P, case = problem()
    leaf = lambda a: torch.as_tensor(a, device="cuda").clone().requires_grad_(True)
    grads = []
    at = P.S.u.data_ptr()
    for used in (False, True):
        v, d = leaf(case.v0), leaf(np.zeros(len(case.wall_nodes)))
        J = P.J(v, d)
        if used:
            P.S.v[0] *= 1.1
            P.S.residual()
        grads.append(torch.autograd.grad(J, [v, d]))
        assert P.S.u.data_ptr() == at
    scale = [float(g.abs().max()) for g in grads[0]]
    # two reverse sweeps differ by the order of the ghosts' atomic sums only
    for a, b, s in zip(*grads, scale):
        assert s > 0 and float((a - b).abs().max()) <= 1e-12 * s
