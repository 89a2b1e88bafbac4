"""The FP64 implicit phase of all blocks in one launch per pass against
implimf_3d block by block on curvilinear blocks (no face normal has a zero
component, so that every product of a face sum counts) of more planes than a
slab: the same bits, whichever of their kernels (small blocks', single
sub-iterations, pairs) the two take."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from randcase import all_thermo, random_mesh, random_state


def T(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda", dtype=torch.float64)


# single sub-iterations in the all-blocks launch, and pairs
@pytest.mark.parametrize("dims", [[(29, 13, 17), (5, 3, 2), (20, 20, 12), (16, 16, 33), (33, 40, 20)],
                                  [(29, 13, 17), (60, 40, 20), (160, 128, 48), (2, 40, 33)]])
@pytest.mark.parametrize("lmx,ityprk", [(1, 0), (2, 1), (3, 0), (4, 0), (5, 1)])
def test_batched_implicit_bits(dims, lmx, ityprk):
    from codens_amd import abi
    lay, sn, vol = random_mesh(dims, seed=23)
    n, rng = lay.ip11, np.random.default_rng(5)
    v = random_state(n, rng)
    ps, _, c = (T(a) for a in all_thermo(v))
    u, ff = T(1e-3 * rng.standard_normal((5, n))), T(1e-4 * rng.standard_normal((5, n)))
    dt, mu, mut = T(.01 * (1 + rng.random(n))), T(1e-3 * (1 + .1 * rng.random(n))), T(1e-4 * rng.random(n))
    ph, gsn, gvol = abi.phys(), T(sn), T(vol)
    blocks = [abi.block(b) for b in lay.blocks]
    (va, da), (vb, db) = [(T(v), T(np.full_like(v, 5.))) for _ in range(2)]
    abi.implimf_3d_batch(abi.block_array(blocks), len(blocks), ph, u, dt, va, da, ff, mu, mut, lmx, gsn, gvol, c,
                         ityprk=ityprk)
    for b, cb in zip(lay.blocks, blocks):
        abi.implimf_3d(cb, ph, u, dt, vb, db, ff, mu, mut, lmx, gsn[9 * b.npc: 9 * (b.npc + b.nnn)], gvol, ps, c,
                       ityprk=ityprk)
    assert torch.equal(da, db) and torch.equal(va, vb)
    assert float(da[:, T(lay.interior()).long()].abs().min()) < 1.
