"""The solver's alternative paths against the oracle: every placement of the job state, watch
lists longer than a wavefront, current levels longer than a wavefront, clauses that name a
variable twice, clauses of more than 8 literals, 32-bit ids, instances without clauses."""
import numpy as np
import pytest

import gpupsat_amd as G
from gpupsat_amd import workloads as W
from gpupsat_amd.formula import Batch, Formula

pytestmark = pytest.mark.gpu


def _chain(n, long_end):
    """x0 -> x1 -> ... -> x(n-1), and x(n-1) contradicts two clauses over a last variable: with
    every phase true the first decision implies the whole chain and a conflict at its end."""
    pos, neg = (lambda v: 2 * v + 1), (lambda v: 2 * v)
    cl = [[neg(i), pos(i + 1)] for i in range(n - 1)]
    cl += [[neg(n - 1), pos(n)], [neg(n - 1), neg(n)]]
    if long_end:
        cl.append([pos(v) for v in range(n)])        # one clause of n literals: x(n-1) never true
    return Formula.from_clauses(n + 1, cl)


def _hub(rng, n, m):
    """Random clauses of which every other one holds one of two hub literals."""
    cl = W.random_ksat_clauses(rng, 1, n, m, 3)[0]
    cl[::2, 0] = rng.integers(0, 2, size=len(cl[::2]))
    return Formula(n, cl.reshape(-1).copy(), np.arange(0, 3 * m + 1, 3, dtype=np.int64))


def _mixed(rng, n, repeat):
    cl = []
    for _ in range(int(4.5 * n)):
        k = int(rng.choice([2, 3, 4, 9, 20], p=[.15, .45, .3, .05, .05]))
        v = rng.integers(0, n, k) if repeat else rng.choice(n, min(k, n), replace=False)
        cl.append([int(2 * x + rng.integers(0, 2)) for x in v])
    return Formula.from_clauses(n, cl)


def _formulas(kind):
    rng = np.random.default_rng(len(kind))
    if kind == "chain":
        return [_chain(n, e) for n in (30, 62, 63, 64, 65, 130, 200) for e in (False, True)]
    if kind == "hub3":
        return [_hub(rng, 40, m) for m in (60, 126, 130, 160, 170, 180)] + [Formula.from_clauses(3, [])]
    if kind == "repeat3":
        return [Formula.from_clauses(20, [[int(2 * x + rng.integers(0, 2)) for x in rng.integers(0, 20, 3)]
                                          for _ in range(90)]) for _ in range(12)]
    return [_mixed(rng, 30, i % 2 == 0) for i in range(12)] + [W.pigeonhole_formula(5, 4), Formula.from_clauses(4, [])]


@pytest.mark.parametrize("kind", ["chain", "hub3", "repeat3", "mixed"])
def test_paths_agree_with_the_oracle(orc, kind):
    b = Batch.from_formulas(_formulas(kind))
    want = [orc.solve_cdcl(b.instance(i))[0] for i in range(b.n_inst)]
    ref = None
    with G.GpuBatch(b) as gb:
        for mem in (1, 2, 3, 4):
            print(f"[solve paths] {kind} clause_mem={mem}", flush=True)
            r = gb.solve(G.SolveOpts.default(clause_mem=mem, phase_init=1, max_conflicts=200000), want_bumps=True)
            assert r["info"]["clause_mem"] == mem
            assert r["status"].tolist() == want
            assert int(r["verified"].sum()) == want.count(G.SAT)
            if mem < 4:      # one search, wherever its state sits
                got = (r["model_rows"], r["job_stats"][:, :7], r["var_bumps"])
                ref = ref or got
                for x, y in zip(got, ref):
                    np.testing.assert_array_equal(x, y)


def test_ids_beyond_16_bits(orc):
    """66,000 clauses: clause ids no longer fit 16 bits (planted solutions, one flipped clause
    set unsatisfiable by two complementary unit chains)."""
    print("[solve paths] 66,000 clauses", flush=True)
    rng = np.random.default_rng(5)
    n, m = 400, 66000
    sol = rng.integers(0, 2, n)
    cl = W.random_ksat_clauses(rng, 1, n, m, 3)[0]
    bad = (((cl & 1) == sol[cl >> 1]).sum(1) == 0)
    cl[bad, 0] ^= 1
    sat = [list(map(int, c)) for c in cl]
    fs = [Formula.from_clauses(n, sat), Formula.from_clauses(n, sat + [[0, 2], [0, 3], [1, 2], [1, 3]])]
    b = Batch.from_formulas(fs)
    with G.GpuBatch(b) as gb:
        r = gb.solve(G.SolveOpts.default(max_conflicts=20000))
    assert r["info"]["clause_mem"] in (2, 4)
    assert r["status"].tolist() == [G.SAT, G.UNSAT] and r["verified"].tolist() == [1, 0]
