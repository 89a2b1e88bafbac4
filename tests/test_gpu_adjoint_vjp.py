"""The reverse sweep of the block residual against its tangent-linear sweep
(dual numbers of the restated residual, an independent path) on states whose
faces take every branch of the Roe flux: sub- and supersonic both ways, with
pinfl and without MUSCL.  <J xdot, ubar> = <xdot, J^T ubar> over state,
metrics and volumes: both sides are sums of the same products in other
orders, so they differ by rounding of the terms' magnitudes (1e-11 of the sum
of their absolute values)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 3, 2), (5, 4, 3), (17, 9, 6), (65, 3, 5)])
@pytest.mark.parametrize("pinfl,muscl,speed", [(0.0, 1, 0.5), (0.2, 1, 3.0), (0.0, 0, 3.0)])
def test_vjp_against_jvp(dims, pinfl, muscl, speed):
    from codens_amd import configs
    from codens_amd.adjoint import AdjointProblem
    case = configs.adjoint_wall(*dims, nwall_nodes=3)
    case.phys["pinfl"], case.scheme["muscl"] = pinfl, muscl
    P = AdjointProblem(case)
    b, n = case.layout.blocks[0], case.layout.ip11
    rng = np.random.default_rng(hash((dims, muscl, int(10 * speed))) % 2**31)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")
    rho, q, p = rng.uniform(0.5, 1.5, n), rng.uniform(-speed, speed, (3, n)), rng.uniform(0.5, 1.5, n)
    v = dev(np.stack([rho, *(rho * q), (p - pinfl) / 0.4 + pinfl + 0.5 * rho * (q * q).sum(0)]))
    sn, vol = dev(case.sn[9 * b.npc: 9 * (b.npc + b.nnn)]), dev(case.vol)
    vd, snd = dev(rng.standard_normal((5, n))), dev(rng.standard_normal(9 * b.nnn)) * sn.abs().max()
    vold = dev(rng.standard_normal(n)) * vol
    ub = dev(rng.standard_normal((5, n))) * P.real
    _, ud = P.jvp(v, sn, vol, vd, snd, vold)
    vb, snb, volb = P.vjp(v, sn, vol, ub)
    terms = [ud * ub, vd * vb, snd * snb, vold * volb]
    lhs, rhs = float(terms[0].sum()), sum(float(t.sum()) for t in terms[1:])
    scale = sum(float(t.abs().sum()) for t in terms)
    assert np.isfinite(scale) and scale > 0
    assert abs(lhs - rhs) <= 1e-11 * scale, (lhs, rhs, scale)
