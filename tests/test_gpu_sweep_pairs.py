"""The FP64 sub-iterations two to a launch, and those of small blocks, against
the tiled kernel's, one to a launch: the same operations on every cell, so the
same bits."""
import numpy as np
import pytest
import torch

from randcase import all_thermo, random_mesh, random_state

pytestmark = pytest.mark.gpu


def T(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda", dtype=torch.float64)


def fields(lay, near=False):
    rng = np.random.default_rng(11)
    n = lay.ip11
    v = random_state(n, rng)
    if near:  # densities a few units of the last place off 1, where a reciprocal rounds with least room
        v[0] = 1. + 2. ** -52 * rng.integers(-8, 8, n)
    ps, _, c = all_thermo(v)
    return dict(v=v, u=1e-3 * rng.standard_normal((5, n)), ff=1e-4 * rng.standard_normal((5, n)),
                dt=.01 * (1 + rng.random(n)), mu=1e-3 * (1 + .1 * rng.random(n)), mut=1e-4 * rng.random(n), ps=ps, c=c)


def pair_launches(abi, call):
    """call() in the default mode, and with one sub-iteration to a launch
    forced; launches of pairs (but a first one) and of single sub-iterations
    in the former"""
    abi.timing_enable(True)
    for name in ("implimf_sweep", "implimf_sweep2"):
        abi.timing_read(name, reset=True)
    try:
        two = call()
        launches = abi.timing_read("implimf_sweep2", reset=True)[1], abi.timing_read("implimf_sweep", reset=True)[1]
        prev = abi.sweep_tile(0)
        try:
            one = call()
        finally:
            abi.sweep_tile(prev)
        assert abi.timing_read("implimf_sweep2", reset=True)[1] == 0
    finally:
        abi.timing_enable(False)
    return two, one, launches


# tiles of 28 x 12 cells (30 x 14 of the first pair of an even number) and slabs of
# 1 to 6 planes: whole and partial tiles, one cell past a tile, two planes, a
# block narrower than the rings
@pytest.mark.parametrize("dims", [(56, 60, 37), (57, 61, 40), (60, 70, 37), (61, 57, 40), (2, 300, 60), (200, 200, 2), (300, 121, 3),
                                  (600, 240, 2), (113, 49, 33)])
@pytest.mark.parametrize("lmx,ityprk", [(2, 0), (3, 0), (4, 1)])
def test_pairs_match_singles(dims, lmx, ityprk):
    from codens_amd import abi
    lay, sn, vol = random_mesh([dims], seed=7)
    b = lay.blocks[0]
    f = fields(lay, near=lmx == 4)
    snb, g = T(sn[9 * b.npc: 9 * (b.npc + b.nnn)]), {k: T(a) for k, a in f.items()}

    def call():
        v, d = T(f["v"]), T(np.full_like(f["v"], 5.))
        abi.implimf_3d(abi.block(b), abi.phys(), g["u"], g["dt"], v, d, g["ff"], g["mu"], g["mut"], lmx, snb,
                       T(vol), g["ps"], g["c"], ityprk=ityprk)
        return v.cpu().numpy(), d.cpu().numpy()

    two, one, launches = pair_launches(abi, call)
    assert launches == ((lmx - 1) // 2, 0), "the shape is one that runs in pairs"
    assert np.array_equal(two[0], one[0]) and np.array_equal(two[1], one[1])


@pytest.mark.parametrize("lmx,ityprk", [(2, 1), (3, 1), (4, 0)])
@pytest.mark.parametrize("full", [False, True])
def test_batched_pairs_match_singles(lmx, ityprk, full):
    """Small blocks alone take single sweeps; with a block that fills the chip all run in pairs."""
    from codens_amd import abi
    dims = [(29, 13, 17), (56, 60, 37), (5, 3, 2), (28, 12, 16), (2, 40, 33)]
    lay, sn, vol = random_mesh(dims + [(160, 128, 48)] * full, seed=9)
    f = fields(lay)
    g, gsn, gvol = {k: T(a) for k, a in f.items()}, T(sn), T(vol)
    arr = abi.block_array([abi.block(b) for b in lay.blocks])

    def call():
        v, d = T(f["v"]), T(np.full_like(f["v"], 5.))
        abi.implimf_3d_batch(arr, len(lay.blocks), abi.phys(), g["u"], g["dt"], v, d, g["ff"], g["mu"], g["mut"], lmx,
                             gsn, gvol, g["c"], ityprk=ityprk)
        return v.cpu().numpy(), d.cpu().numpy()

    two, one, launches = pair_launches(abi, call)
    assert launches == (((lmx - 1) // 2, 0) if full else (0, lmx - 1))
    assert np.array_equal(two[0], one[0]) and np.array_equal(two[1], one[1])


# eight cells to a wave: fewer, a row's end inside a wave, the largest block
@pytest.mark.parametrize("dims", [(2, 2, 2), (5, 3, 2), (17, 9, 7), (32, 32, 16), (2, 90, 2)])
@pytest.mark.parametrize("lmx,ityprk", [(2, 0), (3, 1), (4, 0)])
def test_small_block_matches_tiles(dims, lmx, ityprk):
    from codens_amd import abi
    lay, sn, vol = random_mesh([dims], seed=13)
    b = lay.blocks[0]
    f = fields(lay, near=lmx == 3)
    snb, g = T(sn[9 * b.npc: 9 * (b.npc + b.nnn)]), {k: T(a) for k, a in f.items()}

    def call():
        v, d = T(f["v"]), T(np.full_like(f["v"], 5.))
        abi.timing_read("implimf_sweep1", reset=True)
        abi.implimf_3d(abi.block(b), abi.phys(), g["u"], g["dt"], v, d, g["ff"], g["mu"], g["mut"], lmx, snb,
                       T(vol), g["ps"], g["c"], ityprk=ityprk)
        return v.cpu().numpy(), d.cpu().numpy(), abi.timing_read("implimf_sweep1", reset=True)[1]

    here, tiled, _ = pair_launches(abi, call)
    assert (here[2], tiled[2]) == (0, 1), "the small block's kernel forms the first increment"
    assert np.array_equal(here[0], tiled[0]) and np.array_equal(here[1], tiled[1])
