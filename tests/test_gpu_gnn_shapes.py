"""The branching network's layers at the edges of their tiles (16 rows a wavefront, 128 or, in the
first round backward, 64 a workgroup, neighbours read in fours) and for every form of the first and last round, against
the CPU FP64 oracle with the same BF16 rounding points."""
import numpy as np
import pytest

import gpupsat_amd as G
from gpupsat_amd import learned as Lr
from gpupsat_amd.formula import Batch, Formula
from oracle import gnn_ref as R

pytestmark = pytest.mark.gpu


def formula(rng, n, m, lo, hi):
    """m clauses of lo..hi distinct variables, all over the lower three quarters of the n
    variables but for one (literals without and with many occurrences)."""
    top = max(hi, 3 * n // 4)
    cl = []
    for _ in range(m):
        k = int(rng.integers(lo, hi + 1))
        v = rng.choice(top, size=k, replace=False)
        v[0] = 0 if 0 not in v else v[0]              # variable 0 in every clause
        cl.append(2 * v + rng.integers(0, 2, size=k))
    off = np.concatenate([[0], np.cumsum([len(c) for c in cl])]).astype(np.int64)
    return Formula(n, np.concatenate(cl).astype(np.int32), off)


# (variables, clauses) of the instances; clause lengths; rounds.  Rows in all: 2 literals a
# variable, one a clause: below, at and above one tile, one wavefront's and one workgroup's.
CASES = [
    ([(7, 1)], (1, 1), 1),
    ([(8, 16)], (2, 5), 2),
    ([(9, 17)], (1, 5), 3),
    ([(32, 64)], (3, 3), 1),
    ([(33, 65), (5, 3)], (2, 4), 3),
    ([(64, 127), (16, 31), (31, 130)], (1, 9), 4),
    ([(260, 1100)], (3, 3), 2),
]


@pytest.mark.parametrize("sizes,lens,rounds", CASES)
def test_forward_and_gradient(sizes, lens, rounds):
    print("[gnn shapes]", sizes, lens, rounds, flush=True)
    rng = np.random.default_rng([len(sizes), rounds, sizes[0][0]])
    b = Batch.from_formulas([formula(rng, n, m, lens[0], min(lens[1], n)) for n, m in sizes])
    g = R.Graph(b)
    theta = R.init_params(11)
    target, phase = rng.random(g.V), (rng.random(g.V) < 0.5).astype(float)
    mask = (rng.random(g.V) < 0.6).astype(float)
    with G.GpuBatch(b) as gb:
        m = Lr.GnnModel(theta)
        gg = Lr.GnnGraph(gb, rounds)
        gg.labels(target, phase, mask)
        y = gg.forward(m)
        loss, grad, y2 = gg.loss_grad(m, alpha=0.7)
        again = gg.loss_grad(m, alpha=0.7)
    np.testing.assert_array_equal(y, y2)
    np.testing.assert_array_equal(grad, again[1])     # the same bit for bit
    rl, ry, rgrad = R.backward(theta.astype(np.float64), g, target, phase, mask, quant=True, rounds=rounds, alpha=0.7)
    # as in test_gpu_gnn.py: FP32 instead of FP64 sums flip an occasional BF16 rounding
    assert np.linalg.norm(y - ry) <= 2e-3 * np.linalg.norm(ry)
    assert abs(loss - rl) <= 1e-3 * max(1.0, abs(rl))
    o = 0
    for name, shp in R.PARAM_SHAPES:
        k = int(np.prod(shp))
        a, r = grad[o:o + k], rgrad[o:o + k]
        o += k
        assert np.linalg.norm(a - r) <= 5e-3 * max(np.linalg.norm(r), 1e-12), name


@pytest.mark.parametrize("m,lo,hi", [(0, 1, 1), (1, 1, 1), (63, 1, 1), (64, 1, 1), (65, 1, 1), (128, 2, 2), (85, 3, 3),
                                     (86, 3, 3), (400, 1, 8), (1300, 3, 3), (40, 40, 64)])
def test_graph_built_on_device_and_host(m, lo, hi):
    """The incidence structure built on the GPU against the host's: an instance above its size
    limits sends the whole batch to the host.  Sums over neighbours are in edge order, so equal
    structures give equal bits."""
    print("[gnn graph]", m, lo, hi, flush=True)
    rng = np.random.default_rng([m, hi])
    n = max(hi + 3, m // 4)
    empty = Formula(3, np.zeros(0, np.int32), np.zeros(1, np.int64))
    f = formula(rng, n, m, lo, hi) if m else empty
    small = [f, formula(rng, 5, 9, 2, 2), empty, f]
    big = Formula(2000, np.arange(4, dtype=np.int32), np.array([0, 2, 4], dtype=np.int64))
    theta = R.init_params(13)
    got = []
    for fs in (small, small + [big]):
        with G.GpuBatch(Batch.from_formulas(fs)) as gb:
            g = Lr.GnnGraph(gb)
            V = sum(x.n_vars for x in small)
            got.append(g.forward(Lr.GnnModel(theta))[:V])
            g.close()
    np.testing.assert_array_equal(got[0], got[1])


def test_gradient_of_many_copies():
    """A batch whose gradient rows exceed the last-level cache (576,000 rows of 512 bytes; they
    pass the caches), as 512 copies of one formula: the loss is a mean over variables, and 512 a
    power of two, so every row's gradient is the single formula's scaled exactly and only the
    order of the FP32 sums differs (each a sum of the same terms, 2^-24 per addition over about
    40 levels and runs, with some cancellation: 1e-4 of the block's norm)."""
    print("[gnn shapes] 512 copies", flush=True)
    rng = np.random.default_rng(5)
    f = formula(rng, 180, 765, 3, 3)
    theta = R.init_params(17)
    lab = rng.random(180), (rng.random(180) < 0.5).astype(float), (rng.random(180) < 0.6).astype(float)
    out = []
    for k in (1, 512):
        with G.GpuBatch(Batch.from_formulas([f] * k)) as gb:
            g = Lr.GnnGraph(gb)
            g.labels(*(np.tile(x, k) for x in lab))
            out.append(g.loss_grad(Lr.GnnModel(theta)))
            g.close()
    (l1, g1, y1), (lk, gk, yk) = out
    np.testing.assert_array_equal(np.tile(y1, (512, 1)), yk)
    assert abs(l1 - lk) <= 1e-5 * abs(l1)
    o = 0
    for name, shp in R.PARAM_SHAPES:
        k = int(np.prod(shp))
        a, r = gk[o:o + k], g1[o:o + k]
        o += k
        assert np.linalg.norm(a - r) <= 1e-4 * max(np.linalg.norm(r), 1e-12), name
