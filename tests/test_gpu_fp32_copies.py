"""The FP32 form of the implicit phase on extents around the coefficient pass's
tiles of 64 x 4 columns, whose workgroups also write the FP32 copies of what the
sub-iterations read (a tile's high faces by another thread than the others),
against the FP64 oracle.  Bar: the increment within 2e-5 relative, as for small
blocks (FP32 sub-iterations of about 1e-7 per operation, grown over 4 sweeps)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

import cpu_ref as C
from randcase import all_thermo, random_mesh, random_state, relerr

TOL = 2e-5


def T(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda", dtype=torch.float64)


# whole tiles in i and in j, one cell past one, one cell short, several slabs
@pytest.mark.parametrize("dims", [(64, 4, 9), (128, 8, 3), (65, 5, 10), (63, 3, 17), (64, 5, 2), (66, 12, 33)])
@pytest.mark.parametrize("ityprk", [0, 1])
def test_fp32_tile_edges(dims, ityprk):
    from codens_amd import abi
    lay, sn, vol = random_mesh([dims], seed=37)
    n, b, rng = lay.ip11, lay.blocks[0], np.random.default_rng(41)
    v = random_state(n, rng)
    ps, _, c = all_thermo(v)
    mu, mut = 1e-3 * (1 + .1 * rng.random(n)), 1e-4 * rng.random(n)
    u, ff = 1e-3 * rng.standard_normal((5, n)), 1e-4 * rng.standard_normal((5, n))
    dt = .01 * (1 + rng.random(n))
    O = C.Orc(lay, C.orc_phys())
    vo, do = v.copy(), np.zeros((5, n))
    O.implimf_3d(0, u, dt, vo, do, ff, mu, mut, 4, sn, vol, ps, c, ityprk=ityprk)

    def run(v, u, ff, snb):
        gv, gd = T(v), T(np.full((5, n), 7.))
        abi.implimf_3d_f32(abi.block(b), abi.phys(), T(u), T(dt), gv, gd, T(ff), T(mu), T(mut), 4, snb, T(vol), T(ps),
                           T(c), ityprk=ityprk)
        return gv.cpu().numpy(), gd.cpu().numpy()
    snb = T(sn[9 * b.npc: 9 * (b.npc + b.nnn)])
    nan = np.full((5, n), np.nan)
    run(nan, nan, nan, torch.full_like(snb, float("nan")))  # a copy left out would be NaN below
    hv, hd = run(v, u, ff, snb)
    inner = lay.interior()
    for e in range(5):
        assert relerr(hd[e], do[e]) <= TOL, e
        assert relerr((hv[e] - v[e])[inner], (vo[e] - v[e])[inner]) <= TOL, e
    out = np.ones(n, dtype=bool)
    out[inner] = False
    assert not hd[:, out].any()
