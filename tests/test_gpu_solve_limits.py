"""Solves at the limits of the search's id sizes and of its memory, against verdicts known by
construction or from the oracle."""
import numpy as np
import pytest

import gpupsat_amd as G
from gpupsat_amd.formula import Batch, Formula

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length", [65535, 65536, 65537, 65602])
def test_clause_length_beyond_16_bits(length):
    """A clause (a, b repeated, c) beside the units not-a and not-b holds by c alone, its last
    literal; with not-c as well nothing is left of it."""
    a, b, c = 1, 3, 5
    cl = [[a] + [b] * (length - 2) + [c], [a ^ 1], [b ^ 1]]
    batch = Batch.from_formulas([Formula.from_clauses(4, cl), Formula.from_clauses(4, cl + [[c ^ 1]])])
    with G.GpuBatch(batch) as gb:
        for mem in (0, 1, 2, 3, 4):
            print("[solve limits] clause of", length, "clause_mem", mem, flush=True)
            r = gb.solve(G.SolveOpts.default(clause_mem=mem))
            assert r["status"].tolist() == [G.SAT, G.UNSAT]
            assert r["verified"].tolist() == [1, 0]
