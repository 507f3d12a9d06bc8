"""Solves at the limits of the search's id sizes and of its memory, against verdicts known by
construction or from the oracle."""
import numpy as np
import pytest

import gpupsat_amd as G
from gpupsat_amd import workloads as W
from gpupsat_amd.formula import Batch, Formula
from test_gpu_solve_paths import _formulas
from test_zz_no_alloc import _call

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


@pytest.mark.parametrize("kind", ["chain", "hub3", "repeat3", "mixed"])
def test_32_bit_ids_run_the_same_search(kind):
    """The search with 32-bit ids (a cap of 66,000 learned clauses asks for them; its clauses'
    literals are the batch's, not the wavefront's) against the one with 16-bit ids: neither fills
    its cap, so models and counters are equal.  With the whole state in HBM (placement 4) only the
    verdicts are: lanes that move a watch to the same literal in one step append to its list in
    the order that their atomics reach the cache, which is not the lanes' order as in LDS, and the
    order of a list decides which of several conflicts is met first."""
    batch = Batch.from_formulas(_formulas(kind))
    ref = None
    with G.GpuBatch(batch) as gb:
        for cap, mem in ((20000, 1), (20000, 2), (66000, 2), (66000, 4)):
            print("[solve limits]", kind, "learnt_cap", cap, "clause_mem", mem, flush=True)
            r = gb.solve(G.SolveOpts.default(clause_mem=mem, phase_init=1, learnt_cap=cap, larena_cap=300000,
                                             max_conflicts=4000), want_bumps=True)
            got = r["status"], r["model_rows"], r["job_stats"][:, :7], r["var_bumps"]
            ref = ref or got
            for x, y in list(zip(got, ref))[: 1 if mem == 4 else 4]:
                np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("decision", [0, 1])
def test_branching_variable_with_the_state_in_hbm(decision):
    """The next variable to branch on, found eight at a time per lane (512 a step) where the
    state is in HBM: the same as in LDS, ties included.  Clauses of two literals that share no
    variable: the model shows which of the two was decided first, and no watch list holds two
    clauses (with two, their order could differ, as above)."""
    rng = np.random.default_rng(3)
    fs = [Formula.from_clauses(n, [[2 * int(x) + 1 for x in v] for v in rng.permutation(n)[: n // 2 * 2].reshape(-1, 2)])
          for n in (1, 63, 64, 65, 511, 512, 513, 575, 576, 577, 1100)]
    batch = Batch.from_formulas(fs)
    act = rng.integers(0, 4, int(batch.n_vars.sum())).astype(np.float32)
    got = []
    with G.GpuBatch(batch) as gb:
        for mem in (2, 4):
            print("[solve limits] branching, decision", decision, "clause_mem", mem, flush=True)
            r = gb.solve(G.SolveOpts.default(clause_mem=mem, decision=decision, max_conflicts=1000), act_init=act)
            assert r["info"]["clause_mem"] == mem
            got.append((r["status"], r["model_rows"], r["job_stats"][:, :7]))
    for x, y in zip(*got):
        np.testing.assert_array_equal(x, y)


def test_workspace_larger_than_the_gpu(orc):
    """64 jobs with room for 1.9e9 learned literals each (7.6 GB a wavefront, 486 GB in all) share
    as many wavefronts as there is memory for."""
    print("[solve limits] 7.6 GB a wavefront", flush=True)
    batch = W.random_3sat_batch(64, 20, 85, seed=4)
    with G.GpuBatch(batch) as gb:
        r = gb.solve(G.SolveOpts.default(larena_cap=1900000000))
    assert 1 <= r["info"]["waves"] <= 32
    assert r["status"].tolist() == [orc.solve_cdcl(batch.instance(i))[0] for i in range(64)]


def test_noalloc_with_the_scratch_region_full():
    """4,000 jobs whose cubes (their literals repeated) leave 8 KB of the 64 MiB scratch region,
    less than one wavefront's learned literals: the job state goes to LDS, which needs none."""
    f = W.random_3sat_batch(1, 10, 20, seed=5).instance(0)
    batch = Batch.from_formulas([f, W.pigeonhole_formula(4, 3)])
    J, N = 4000, 2
    up = lambda n: (n + 255) // 256 * 256                                 # noqa: E731
    words = 2
    table = [16 * J, 4, 8, 8 * N, 4 * N, 4 * N, 4 * N, 4 * N, 8 * (N + 1), 8 * len(G.JOB_STAT_FIELDS) * J, 4 * words, 12 * N]
    total = ((64 << 20) - sum(up(x) for x in table) - 8192) // 256 * 256 // 4
    per = np.full(J, total // J)
    per[: total - per.sum()] += 1
    ji = np.repeat(np.arange(2, dtype=np.int32), J // 2)
    co = np.concatenate([[0], np.cumsum(per)]).astype(np.int32)
    assert co[-1] == total
    cl = (np.repeat(np.arange(J), per) % 2 + 2 * np.repeat(np.arange(J) // 2 % 10, per)).astype(np.int32)
    with G.GpuBatch(batch) as gb:
        assert gb.row_words(1) == words
        print("[solve limits] scratch region full", flush=True)
        rc, status, *_, info = _call("gpsat_solve_noalloc", gb, G.SolveOpts.default(), jobs=(ji, co, cl))
        assert rc == 0, G.lib().gpsat_last_error()
    assert status.tolist() == [G.SAT, G.UNSAT]
    assert info.clause_mem == 1 and info.workspace_bytes == 0
