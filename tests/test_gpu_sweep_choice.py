"""What implimf_3d decides on the host for a block: quickly, and by a rule that
holds for narrow blocks too."""
import time

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def call(dims, lmx=5, batched=False):
    """a call of the implicit phase on blocks of the given sizes"""
    from codens_amd import abi
    from codens_amd import layout as L
    lay = L.Layout(dims)
    n = lay.ip11
    R = lambda *s: torch.rand(*s, device="cuda", dtype=torch.float64)
    v = .1 * R(5, n)
    v[0] += 1.
    v[4] += 2.5
    u, ff, d, sn = 1e-3 * R(5, n), R(5, n), R(5, n), 1e-2 * R(9 * n)
    vol, dt, mu, mut, ps, c = (R(n) + .5 for _ in range(6))
    blocks, ph = [abi.block(b) for b in lay.blocks], abi.phys()
    arr = abi.block_array(blocks)
    if batched:
        return lambda: abi.implimf_3d_batch(arr, len(dims), ph, u, dt, v, d, ff, mu, mut, lmx, sn, vol, c)
    return lambda: abi.implimf_3d(blocks[0], ph, u, dt, v, d, ff, mu, mut, lmx, sn, vol, ps, c)


def host_time(f):
    """the shortest of 30 calls, until they return"""
    f()
    best = 1.
    for _ in range(30):
        torch.cuda.synchronize()
        t = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t)
    return best


def pair_launches(f):
    """the number of pairs of sub-iterations (but a first one) that a call launches"""
    from codens_amd import abi
    abi.timing_enable(True)
    try:
        abi.timing_read("implimf_sweep2", reset=True)
        f()
        return abi.timing_read("implimf_sweep2", reset=True)[1]
    finally:
        abi.timing_enable(False)


def test_host_time_of_long_blocks():
    """The slab depths are found in about the square root of the plane count:
    a block of 40,000 planes takes the host no more than 3 times what one of 40
    takes (6 times with a look at every depth)."""
    assert host_time(call([(2, 2, 40000)])) <= 3. * host_time(call([(64, 64, 40)]))


# measured on MI355X, two single sub-iterations / a pair (us)
@pytest.mark.parametrize("dims,pairs", [((16, 16, 400), False),  # 19 / 33
                                        ((4, 64, 400), False),  # 47 / 60
                                        ((3, 63, 128), False), ((5, 231, 17), False), ((8, 30, 202), False),
                                        ((2, 2, 12000), False),  # 128 / 180
                                        ((40, 40, 20), False), ((24, 24, 64), False),
                                        ((20, 20, 2000), True),  # 139 / 90
                                        ((17, 33, 300), True), ((65, 33, 129), True), ((130, 96, 66), True)])
def test_pairs_where_they_are_faster(dims, pairs):
    assert bool(pair_launches(call([dims]))) == pairs


@pytest.mark.parametrize("dims,pairs", [([(16, 16, 192)] * 16, False),  # 136 / 176
                                        ([(28, 12, 64)] * 16, False),  # 61 / 86
                                        ([(4, 4, 3000)] * 3, False), ([(12, 17, 40), (25, 33, 18), (37, 14, 22)], False),
                                        ([(16, 192, 16)] * 32, True),  # 273 / 171
                                        ([(56, 24, 32)] * 32, True)])  # 168 / 102
def test_batched_pairs_where_they_are_faster(dims, pairs):
    assert bool(pair_launches(call(dims, batched=True))) == pairs
