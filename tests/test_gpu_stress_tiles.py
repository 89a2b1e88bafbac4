"""Stresses and heat flux (zvisqc) on extents around its three tile shapes
(64 x 4, 32 x 8, 16 x 16) and slabs of 8 planes, against the oracle.  Bar: the
same 12 sums of six products and a handful of products as the oracle's, 1e-12
of the largest value."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

import cpu_ref as C
from randcase import all_thermo, random_mesh, random_state, relerr

TOL = 1e-12


def T(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda", dtype=torch.float64)


# whole tiles, one cell past a tile, rows shorter than any tile, one plane past a slab
@pytest.mark.parametrize("dims", [(64, 4, 8), (65, 5, 9), (32, 8, 3), (33, 9, 17), (16, 16, 2), (17, 15, 4), (3, 2, 2)])
def test_zvisqc_tiles(dims):
    from codens_amd import abi
    lay, sn, vol = random_mesh([dims], seed=29)
    n, b = lay.ip11, lay.blocks[0]
    rng = np.random.default_rng(3)
    v = random_state(n, rng)
    _, t, _ = all_thermo(v)
    mu, mut = 1e-3 * (1 + .1 * rng.random(n)), 1e-3 * rng.random(n)
    O = C.Orc(lay, C.orc_phys())
    tq, g = np.zeros((9, n)), T(np.zeros((9, n)))
    O.zfluto(0, mu, mut, tq, O.zgrad2(0, sn, vol, v, t))
    abi.zvisqc(abi.block(b), abi.phys(), T(sn[9 * b.npc: 9 * (b.npc + b.nnn)]), T(vol), T(v), T(t), T(mu), T(mut), g)
    h = g.cpu().numpy()
    for q in range(9):
        assert relerr(h[q], tq[q]) <= TOL, q
