"""The cells that bench.py divides a sweep launch's time by: those of the blocks
that launch the kernel."""
import pytest

import bench


def test_mean_cells_of_a_launch():
    # blocks of 1000, 50,000 and 90,000 cells, lmax = 10, 5 stages
    n, stages, lmax = 141000, 5, 10
    assert bench.cells_per_sweep_launch([50000, 90000], 2 * 4 * stages, stages, n, lmax, False) == 70000
    assert bench.cells_per_sweep_launch([], 4 * stages, stages, n, lmax, True) == n
    assert bench.cells_per_sweep_launch(None, 3 * 9 * stages, stages, n, lmax, False) == n / 3
    assert bench.cells_per_sweep_launch(None, 9 * stages, stages, n, lmax, True) == n


@pytest.mark.gpu
def test_blocks_that_run_in_pairs():
    """As many blocks as a stage launches pairs for, none of at most 16384 cells;
    the solver's state stays as it is."""
    import torch
    from codens_amd import abi, configs
    from codens_amd.solver import Solver
    case = configs.multiblock_sa(4, 8, 110, None, seed=71)
    cells = [b.ncells for b in case.layout.blocks]
    assert min(cells) <= 16384 and max(cells) > 200000 and case.lmax == 10
    s = Solver(case)
    abi.timing_enable(True)
    abi.timing_read("implimf_sweep2", reset=True)
    s.stage()
    launches = abi.timing_read("implimf_sweep2", reset=True)[1]
    abi.timing_enable(False)
    v, d = s.v.clone(), s.d.clone()
    pairs = bench.pair_cells(s)
    assert torch.equal(s.v, v) and torch.equal(s.d, d)
    assert launches == 4 * len(pairs) > 0 and all(c in cells and c > 16384 for c in pairs)
