"""Order of the Spalart-Allmaras source launches of several blocks on several
streams.  met_smsa reads fd at the block-local index (met_smsa.f90:216-217),
that is, entries of the blocks stored first; the result is that of one stream
only if those blocks' flux densities are formed before and their next
gradients after.  On the CPU: the launches and the streams' waits recorded, and
each launch's predecessors compared; on the GPU: the same bits as one stream."""
import types

import pytest

from codens_amd import layout as L


class FakeStream:
    """The launches ordered before whatever comes next on the stream."""

    def __init__(self):
        self.seen = set()

    def wait_stream(self, other):
        self.seen |= other.seen


class FakeAbi:
    """Records (entry point, block) -> its predecessors, per turbulence stage."""

    def __init__(self, blocks):
        self.at = {b.npc: l for l, b in enumerate(blocks)}
        self.before, self.stage = {}, 0

    def workspace_set(self, k):
        pass

    def __getattr__(self, name):
        def launch(b, *args, stream):
            op = (self.stage, name, self.at[b.npc])
            self.before[op] = frozenset(stream.seen)
            stream.seen.add(op)
        return launch


# blocks that reach into none, one and several of those stored before them
@pytest.mark.parametrize("dims", [[(8, 6, 5), (5, 4, 3), (6, 6, 6), (20, 8, 6)],
                                  [(3, 3, 3), (2, 2, 2), (4, 3, 2), (2, 2, 2), (24, 12, 9), (2, 3, 2), (30, 12, 9)]])
@pytest.mark.parametrize("lanes", [(0, 1, 2), (2, 0, 1), (0, 0, 1)])
def test_smsa_after_the_densities_it_reads(monkeypatch, dims, lanes):
    from codens_amd import solver
    lay = L.Layout(dims)
    n = len(dims)
    none = types.SimpleNamespace(numel=lambda: 0)
    abi = FakeAbi(lay.blocks)
    monkeypatch.setattr(solver, "abi", abi)
    S = object.__new__(solver.Solver)
    S.case = types.SimpleNamespace(turb=types.SimpleNamespace(model="1SA", tc=None, kfludis=2, klroe=2, kparoi=0,
                                                              cmt=1., epsk=0., epse=0.))
    S.lay, S.blocks, S.batch = lay, lay.blocks, set()
    S.stream, S.side = FakeStream(), [FakeStream() for _ in range(3)]
    S.lane = [lanes[l % 3] for l in range(n)]
    S.coin = S.tq_copy = (none,) * 3
    S.wall = S.far = S.sym = (none,)
    for f in ("v", "u", "d", "dt", "fd", "mu", "mut", "vol", "dist", "cfke", "ts6", "ts7"):
        setattr(S, f, None)
    S.sn_blk = S.g9 = S.tprod = [None] * n
    for abi.stage in range(2):
        S.turb_stage()
    for st in range(2):
        for l, b in enumerate(lay.blocks):
            before = abi.before[(st, "met_smsa", l)]
            for j, other in enumerate(lay.blocks):
                if j == l or other.npc >= b.nnn:
                    continue
                # this stage's densities of a block stored before
                assert j < l and (st, "met_flud", j) in before
                # and no gradients of the next stage
                if st == 0:
                    assert (0, "met_smsa", l) in abi.before[(1, "met_gradtr", j)]


@pytest.mark.gpu
@pytest.mark.parametrize("streams", [2, 3, 4])
def test_spalart_allmaras_streams_match_serial(streams):
    """The source Jacobian cfke, the state and the eddy viscosity over 3
    stages, eager and replayed, bit for bit."""
    import torch
    from codens_amd import configs
    from codens_amd.solver import Solver
    case = configs.multiblock_sa(9, 4, 11, None, seed=7, ilim=1, lmax=4)
    ref, eager, graph = Solver(case), Solver(case, streams=streams), Solver(case, streams=streams)
    graph.capture()
    ref.stage(); eager.stage()
    for _ in range(2):
        ref.stage(); eager.stage(); graph.stage()
    torch.cuda.synchronize()
    for s in (eager, graph):
        for x, y in ((s.cfke, ref.cfke), (s.v, ref.v), (s.mut, ref.mut)):
            assert torch.equal(x.cpu(), y.cpu())
