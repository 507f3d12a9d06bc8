"""The packed evaluation kernel's forms: wide slots (n above 496) and 10-bit ones, at the sizes
where the rule changes form, at the edges of their 64-clause groups and at the lengths where rows
are read another way -- equal to the oracle and to the CSR kernel."""
import numpy as np
import pytest

import gpupsat_amd as G
from gpupsat_amd import workloads as W
from gpupsat_amd.formula import Batch, Formula

pytestmark = pytest.mark.gpu


def formula(rng, n, lens):
    """One clause per entry of lens, in that order, over distinct variables."""
    cl = [2 * rng.choice(n, size=k, replace=False) + rng.integers(0, 2, size=k) for k in lens]
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    return Formula(n, np.concatenate([c for c in cl if len(c)] or [[]]).astype(np.int32), off)


# (variables, clauses of more than 2 literals, of at most 2, longest) and the kernel that takes it
CASES = [
    (496, 64, 128, 6, "packed"), (496, 63, 66, 4, "packed"), (300, 0, 70, 2, "packed"), (100, 1, 63, 5, "packed"),
    (497, 64, 200, 4, "packed"), (600, 65, 127, 4, "packed"), (512, 200, 0, 3, "packed"), (1024, 0, 900, 2, "packed"),
    (2016, 130, 1500, 4, "packed"), (2017, 130, 1500, 4, "csr"), (497, 64, 64, 5, "csr"),
]


@pytest.mark.parametrize("n,long_,short,longest,kernel", CASES)
def test_forms(orc, n, long_, short, longest, kernel):
    print("[packed forms]", n, long_, short, longest, flush=True)
    rng = np.random.default_rng([n, long_, short])
    lens = np.concatenate([rng.integers(3, max(4, longest + 1), size=long_), rng.integers(1, 3, size=short)])
    lens = np.minimum(lens, longest)
    if long_ and longest > 3:
        lens[0] = longest
    rng.shuffle(lens)
    # a second, smaller instance of another shape in the same batch
    b = Batch.from_formulas([formula(rng, n, lens), formula(rng, 33, [3] * 20 + [2] * 100 + [1])])
    for A, p in ((64, 0.02), (37, 0.3)):
        rows = W.random_assignments(b, A, p, seed=n + A)
        want = orc.eval_batch(b, rows, A), *orc.bcp_batch(b, rows, A)
        with G.GpuBatch(b) as gb:
            assert gb.eval_kernel() == kernel
            for over in ({}, {"eval_pkk_waves": 1}, {"eval_pkk": 0}):
                with G.tuned(**over):
                    got = gb.clause_eval(rows, A), *gb.bcp_fixpoint(rows, A)
                for g, w in zip(got, want):
                    np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("n_nodes", [100, 140, 300])
def test_colorings(orc, n_nodes):
    """Long implication chains (and the 32-bit handoff) on 4-colourings."""
    print("[packed forms] colourings", n_nodes, flush=True)
    b = W.coloring_batch(6, n_nodes=n_nodes, seed=n_nodes)
    for p in (0.01, 0.05):
        rows = W.random_assignments(b, 64, p, seed=n_nodes)
        with G.GpuBatch(b) as gb:
            assert gb.eval_kernel() == "packed"
            for over in ({}, {"eval_pkk_compact": 0}):
                with G.tuned(**over):
                    for g, w in zip(gb.bcp_fixpoint(rows, 64), orc.bcp_batch(b, rows, 64)):
                        np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("n", [1, 16, 17, 127, 128, 129, 192, 193, 496, 511, 512, 513, 1024, 2016])
def test_row_lengths(orc, n):
    """Rows copied in and out a word at a time over all wavefronts: rows of 1 word, of the words
    one batch of transposes takes (8, 16, 24 or 32, by the wavefronts) and one more, of the 12
    that are read without a copy and one more, of the most a table holds; beside an instance without variables."""
    print("[packed forms] rows", n, flush=True)
    rng = np.random.default_rng(n)
    k = min(n, 4)
    none = Formula(0, np.zeros(0, np.int32), np.zeros(1, np.int64))
    b = Batch.from_formulas([formula(rng, n, [k] * 30 + [min(n, 2)] * (2 * n)), none, formula(rng, n, [1] * 3)])
    for A, p in ((1, 0.2), (33, 0.02), (64, 0.1)):
        rows = W.random_assignments(b, A, p, seed=n)
        want = orc.eval_batch(b, rows, A), *orc.bcp_batch(b, rows, A)
        with G.GpuBatch(b) as gb:
            assert gb.eval_kernel() == "packed"
            for nw in (1, 2, 3, 4):
                with G.tuned(eval_pkk_waves=nw):
                    got = gb.clause_eval(rows, A), *gb.bcp_fixpoint(rows, A)
                for g, w in zip(got, want):
                    np.testing.assert_array_equal(g, w)
