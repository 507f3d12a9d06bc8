"""The packed kernel's wide words, made on the GPU when a batch is created: clauses of 0 to 4
literals at the edges of a workgroup's 256, over many instances of different sizes."""
import numpy as np
import pytest

import gpupsat_amd as G
from gpupsat_amd import workloads as W
from gpupsat_amd.formula import Batch, Formula

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shortest,longest", [(0, 4), (1, 1), (2, 3), (4, 4)])
def test_words_of_every_length(orc, shortest, longest):
    print("[wide words]", shortest, longest, flush=True)
    rng = np.random.default_rng([shortest, longest])
    fs = [Formula(1, np.zeros(0, np.int32), np.zeros(1, np.int64))]
    for n, m in [(497, 256), (2016, 257), (30, 255), (700, 1), (600, 513), (1000, 0)] * 6:
        lens = rng.integers(shortest, longest + 1, m)
        off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
        fs.append(Formula(n, rng.integers(0, 2 * n, off[-1]).astype(np.int32), off))
    b = Batch.from_formulas(fs)
    rows = W.random_assignments(b, 9, 0.3, seed=longest)
    with G.GpuBatch(b) as gb:
        assert gb.eval_kernel() == "packed"
        got = gb.clause_eval(rows, 9), *gb.bcp_fixpoint(rows, 9)
    for g, w in zip(got, (orc.eval_batch(b, rows, 9), *orc.bcp_batch(b, rows, 9))):
        np.testing.assert_array_equal(g, w)
