"""What AdjointProblem.vjp hands to the library (on the CPU, the library's call
recorded): the kernels read 5 x ip11 doubles of the residual's adjoint, whatever
form the caller's has."""
import types

import pytest
import torch


@pytest.mark.parametrize("form", ["plain", "single", "column", "transposed", "seven"])
def test_adjoint_of_u_as_the_kernels_read_it(monkeypatch, form):
    from codens_amd import adjoint
    n = 11
    full = torch.arange(5 * n, dtype=torch.float64).view(5, n)
    ubar = {"plain": full, "single": full.float(), "column": full[:, :1],
            "transposed": full.t().contiguous().t(), "seven": torch.cat([full, -full[:2]])}[form]
    want = ubar[:5].double().expand(5, n)
    got = []
    monkeypatch.setattr(adjoint, "abi", types.SimpleNamespace(
        adj_residual_vjp=lambda b, ph, sc, v, sn, vol, winf, bcs, ub, vb, snb, volb: got.append(ub)))
    P = object.__new__(adjoint.AdjointProblem)
    P.blk = P.ph = P.sc = P.winf = P.bcs = None
    vb, snb, volb = P.vjp(torch.ones(5, n, dtype=torch.float64), torch.ones(9 * n, dtype=torch.float64),
                          torch.ones(n, dtype=torch.float64), ubar)
    ub, = got
    assert ub.dtype == torch.float64 and ub.shape == (5, n) and ub.is_contiguous() and torch.equal(ub, want)
    assert vb.shape == (5, n) and snb.shape == (9 * n,) and volb.shape == (n,)
