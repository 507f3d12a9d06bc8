"""The branching network at the limits of its kernels: the incidence graph's largest launch, and
layers of exactly one workgroup's rows (8 wavefronts of 16) and one tile more."""
import numpy as np
import pytest

import gpupsat_amd as G
import test_gpu_gnn_shapes as S
from gpupsat_amd import learned as Lr
from gpupsat_amd.formula import Batch, Formula
from oracle import gnn_ref as R

pytestmark = pytest.mark.gpu


def test_graph_at_the_limits_of_its_kernel():
    """1,984 variables (63,488 bytes of counters), 65,536 edges and clauses of 64 literals, three
    such instances: the most that is built on the GPU (see test_dispatch_rules.py).  One variable
    more in another instance, and the same graph is built on the host."""
    print("[gnn limits] graph of 1,984 variables, 65,536 edges", flush=True)
    rng = np.random.default_rng(8)

    def instance():
        lens = np.append(np.full(900, 64), rng.multinomial(65536 - 900 * 64 - 400, np.full(400, 1 / 400)) + 1)
        assert lens.sum() == 65536 and lens.max() == 64
        rng.shuffle(lens)
        lits = rng.integers(0, 2 * 1984, 65536).astype(np.int32)
        lits[::7] = 3967                                   # one literal thousands of times
        return Formula(1984, lits, np.concatenate([[0], np.cumsum(lens)]).astype(np.int64))

    fs = [instance() for _ in range(3)]
    other = Formula(1985, np.arange(4, dtype=np.int32), np.array([0, 2, 4], dtype=np.int64))
    theta = R.init_params(13)
    got = []
    for x in (fs, fs + [other]):
        with G.GpuBatch(Batch.from_formulas(x)) as gb:
            g = Lr.GnnGraph(gb)
            got.append(g.forward(Lr.GnnModel(theta))[: 3 * 1984])
            g.close()
    np.testing.assert_array_equal(got[0], got[1])


@pytest.mark.parametrize("sizes", [[(64, 128)], [(65, 129)], [(64, 127), (64, 129)], [(63, 112), (66, 145)]])
@pytest.mark.parametrize("rounds", [1, 2])
def test_one_workgroup_of_rows(sizes, rounds):
    """128 literal and clause rows, 130 and 129, and twice as many over two instances."""
    S.test_forward_and_gradient(sizes, (2, 4), rounds)
