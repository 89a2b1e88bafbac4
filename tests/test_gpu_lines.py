"""The line-implicit phase of the transport equations at line lengths and
counts around the kernels' batches of 15 steps, waves of 32 and 64 lines and
tiles of 16 cells, block by block and all blocks in one launch, against the
oracle.  The increments are read off v(6:7) = 0.  Bar: the systems are
diagonally dominant, so six sweeps of at most 46 steps of a few rounding
errors stay below 6 x 46 x 4 x 1.1e-16 = 1.2e-13 of the largest; 1e-12."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

import cpu_ref as C
from randcase import random_mesh, random_state, relerr

TOL = 1e-12


def T(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda", dtype=torch.float64)


@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("dims", [[(15, 16, 30)], [(31, 14, 2), (33, 29, 46)], [(2, 3, 45), (16, 17, 15), (32, 2, 16)]])
def test_impli2_line_shapes(dims, batched):
    from codens_amd import abi
    from oracle import ptr
    lay, sn, vol = random_mesh(dims, seed=17)
    n = lay.ip11
    rng = np.random.default_rng(19)
    v = np.zeros((7, n))
    v[:5] = random_state(n, rng)
    u = np.zeros((7, n))
    u[5:] = 1e-3 * rng.standard_normal((2, n))
    mu, mut = 1e-3 * (1 + .1 * rng.random(n)), 1e-3 * rng.random(n)
    dt, cfke = .01 * (1 + rng.random(n)), rng.random(n)
    O, vo, gv = C.Orc(lay, C.orc_phys()), v.copy(), T(v)
    g = [T(x) for x in (u, dt, mu, mut, cfke, vol)]
    if batched:
        abi.impli2_eqt_3d_batch(abi.block_array([abi.block(b) for b in lay.blocks]), len(lay.blocks), g[0], g[1], gv,
                                g[2], g[3], g[4], T(sn), g[5], 2.0)
    for b in lay.blocks:
        snb = np.ascontiguousarray(sn[9 * b.npc: 9 * (b.npc + b.nnn)])
        O.lib.orc_impli2_eqt_3d(ctypes.byref(C.orc_block(b)), ptr(u), C.L_(n), ptr(dt), ptr(vo), ptr(mu), ptr(mut),
                                ptr(cfke), ptr(snb), ptr(vol), C.D(2.0))
        if not batched:
            abi.impli2_eqt_3d(abi.block(b), g[0], g[1], gv, g[2], g[3], g[4], T(snb), g[5], 2.0)
    hv = gv.cpu().numpy()
    inner = lay.interior()
    for e in (5, 6):
        assert relerr(hv[e, inner], vo[e, inner]) <= TOL, e
    other = np.ones(n, dtype=bool)
    other[inner] = False
    assert np.array_equal(hv[:5], v[:5]) and not hv[5:, other].any()
