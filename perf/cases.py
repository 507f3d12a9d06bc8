"""The work that users of this engine have it do, as performance cases over its public
entry points: batched clause evaluation and BCP fixpoints, CDCL solves, and the branching
network's inference and training pass.

Assignment rows and outputs of the device-buffer calls live in torch tensors (a caller's own
device memory); everything else goes through gpupsat_amd as in tests/ and bench.py.  Outputs
are integers (compared for equality), except the network's.
"""
import ctypes
import math

import numpy as np
import torch

import gpupsat_amd as G
from gpupsat_amd import learned as LB
from gpupsat_amd import workloads as W
from gpupsat_amd.formula import Batch, Formula

A = 64                                   # assignment rows per instance, the most a call takes
RATIO3 = 4.26                            # clauses per variable of hard random 3-SAT
HID = 64                                 # the network's hidden size


def listed():
    return [
        # the smallest call: a handful of small formulas on buffers already on the GPU, where the
        # launch and the binding are what is paid for (an online service checking a few trails)
        {"name": "eval_bcp_small", "kind": "eval_bcp", "family": "3sat", "inst": 16, "n": 50, "p": 0.2, "rows": A},
        # bench.py's headline step: 10,000 random 3-SAT under dense trails (most rows conflict)
        {"name": "eval_bcp_3sat_dense", "kind": "eval_bcp", "family": "3sat", "inst": 10000, "n": 200, "p": 0.3,
         "rows": A},
        # the same batch under sparse trails, where BCP has long implication chains to follow
        {"name": "eval_bcp_3sat_sparse", "kind": "eval_bcp", "family": "3sat", "inst": 10000, "n": 200, "p": 0.05,
         "rows": A},
        # mixed random 3/4/5-SAT with n 100-400, ragged instance sizes (the cube workload's batch)
        {"name": "eval_bcp_mixed", "kind": "eval_bcp", "family": "mixed", "inst": 2048, "n": 400, "p": 0.1, "rows": A},
        # structured formulas: 4-colourings of sparse graphs, 600 variables, clauses of 2 and 4
        {"name": "eval_bcp_coloring", "kind": "eval_bcp", "family": "coloring", "inst": 1000, "n": 600, "p": 0.05,
         "rows": A},
        # a caller with rows in host memory and fewer of them (the host-buffer form, PCIe included)
        {"name": "bcp_host", "kind": "bcp_host", "family": "3sat", "inst": 1000, "n": 200, "p": 0.1, "rows": 37},
        # one formula solved alone, what the command-line tool does per file: latency of one search
        {"name": "solve_one", "kind": "solve", "family": "3sat", "inst": 1, "n": 150},
        # bench.py's solve leg: many small random 3-SAT, one wavefront each
        {"name": "solve_3sat", "kind": "solve", "family": "3sat", "inst": 20000, "n": 50},
        # structured solves: colourings (satisfiable, long propagations) and pigeonhole principles
        # (unsatisfiable, learning-bound; clauses of 2, 4 and 6 literals) in one batch
        {"name": "solve_structured", "kind": "solve", "family": "structured", "inst": 500, "n": 600},
        # cube-and-conquer: harder 3-SAT split by the MaxClause chooser into 16 cubes each
        {"name": "solve_cubes", "kind": "cubes", "family": "3sat", "inst": 128, "n": 175, "depth": 4},
        # network inference on formulas never seen before (graph construction included)
        {"name": "gnn_infer", "kind": "gnn_infer", "family": "3sat", "inst": 256, "n": 300},
        # the network's training pass: loss and gradient of a batch whose graph is kept
        {"name": "gnn_train", "kind": "gnn_train", "family": "3sat", "inst": 512, "n": 300},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eval_bcp", "eval_bcp", "eval_bcp", "bcp_host", "solve", "solve", "cubes", "gnn_infer",
                       "gnn_train"])
    if kind == "eval_bcp":
        fam = rng.choice(["3sat", "mixed", "coloring"])
        p = round(math.exp(rng.uniform(math.log(0.02), math.log(0.3))), 4)
        rows = rng.choice([A, A, rng.randint(1, A)])
        if fam == "3sat":
            n = _log_int(rng, 50, 450)
            return {"kind": kind, "family": fam, "inst": _log_int(rng, 8, 1.6e6 / n), "n": n, "p": p, "rows": rows}
        if fam == "mixed":
            return {"kind": kind, "family": fam, "inst": _log_int(rng, 16, 2048), "n": rng.randint(150, 400), "p": p,
                    "rows": rows}
        n = 4 * _log_int(rng, 30, 400)
        return {"kind": kind, "family": fam, "inst": _log_int(rng, 8, 4e5 / n), "n": n, "p": p, "rows": rows}
    if kind == "bcp_host":
        return {"kind": kind, "family": "3sat", "inst": _log_int(rng, 4, 1000), "n": _log_int(rng, 50, 250),
                "p": round(rng.uniform(0.02, 0.3), 4), "rows": rng.randint(1, A)}
    if kind == "solve":
        fam = rng.choice(["3sat", "structured"])
        if fam == "3sat":
            n = _log_int(rng, 40, 150)
            return {"kind": kind, "family": fam, "inst": _log_int(rng, 1, 20000 * (40 / n) ** 3), "n": n}
        return {"kind": kind, "family": fam, "inst": _log_int(rng, 10, 500), "n": 4 * rng.randint(60, 150)}
    if kind == "cubes":
        return {"kind": kind, "family": "3sat", "inst": _log_int(rng, 4, 128), "n": rng.randint(120, 170),
                "depth": rng.randint(2, 5)}
    return {"kind": kind, "family": "3sat", "inst": _log_int(rng, 4, 256 if kind == "gnn_infer" else 512),
            "n": rng.randint(100, 300)}


# ---------------------------------------------------------------------------------------------
# inputs

def _ksat(rng, N, n, m, k):
    """int32[N, m, k]: uniform random clauses of k distinct variables, either sign (the family of
    workloads.random_ksat_clauses, drawn without retries)."""
    v = np.empty((N, m, k), dtype=np.int32)
    for j in range(k):
        x = rng.integers(0, n - j, size=(N, m), dtype=np.int32)
        for q in np.moveaxis(np.sort(v[..., :j], axis=-1), -1, 0):
            x += x >= q                          # the x-th variable not among the first j
        v[..., j] = x
    return 2 * v + rng.integers(0, 2, size=v.shape, dtype=np.int32)


def _formulas(case, seed):
    fam, N, n = case["family"], case["inst"], case["n"]
    if fam == "3sat":
        rng = np.random.default_rng([seed, 11])
        m = int(round(RATIO3 * n))
        return Batch.uniform(_ksat(rng, N, n, m, 3), n)
    if fam == "mixed":
        rng = np.random.default_rng([seed, 12])
        fs = []
        for k, v, m in _mixed_sizes(case):
            cl = _ksat(rng, 1, v, m, k)[0]
            fs.append(Formula(v, cl.reshape(-1), np.arange(0, m * k + 1, k, dtype=np.int64)))
        return Batch.from_formulas(fs)
    if fam == "coloring":
        return _colorings(N, n // 4, seed)
    # structured: colourings, plus one pigeonhole principle of each size 4..7 per 25 of them
    col = _colorings(N, n // 4, seed)
    php = [W.pigeonhole_formula(p + 1, p) for p in (4, 5, 6, 7)] * max(1, N // 25)
    return Batch.from_formulas([col.instance(i) for i in range(N)] + php)


def _mixed_sizes(case):
    """(literals per clause, variables, clauses) of every instance: the same for every seed."""
    rng = np.random.default_rng([case["inst"], case["n"]])
    ks, ns = rng.integers(3, 6, size=case["inst"]), rng.integers(100, case["n"] + 1, size=case["inst"])
    return [(k, v, int(round({3: RATIO3, 4: 9.9, 5: 21.1}[k] * v))) for k, v in zip(ks.tolist(), ns.tolist())]


def _colorings(N, nodes, seed):
    """4-colourings of Erdos-Renyi graphs of average degree 4.2-4.8 (workloads.coloring_batch's
    family; its formulas, built with array operations)."""
    rng = np.random.default_rng([seed, 13])
    u = np.repeat(np.arange(nodes), 4).reshape(nodes, 4)
    c = np.tile(np.arange(4), (nodes, 1))
    alo = 2 * (4 * u + c) + 1                                             # at least one colour
    pa, pb = np.array([(a, b) for a in range(4) for b in range(a + 1, 4)]).T
    base = np.arange(nodes)[:, None]
    amo = np.stack([2 * (4 * base + pa), 2 * (4 * base + pb)], axis=-1).reshape(-1, 2)
    fs = []
    for _ in range(N):
        e = W.er_graph(rng, nodes, rng.uniform(4.2, 4.8))
        k = np.arange(4)
        dif = np.stack([2 * (4 * e[:, :1] + k), 2 * (4 * e[:, 1:] + k)], axis=-1).reshape(-1, 2)
        lits = np.concatenate([alo.reshape(-1), amo.reshape(-1), dif.reshape(-1)]).astype(np.int32)
        off = np.concatenate([np.arange(0, 4 * nodes, 4), np.arange(4 * nodes, len(lits) + 1, 2)]).astype(np.int64)
        fs.append(Formula(4 * nodes, lits, off))
    return Batch.from_formulas(fs)


def _rows(batch, rows, p, seed):
    """Partial assignments: every variable assigned with probability p, either polarity, packed
    as literal bitmaps (16 variables a word), int32[sum of rows * W_i] on the GPU."""
    n = torch.as_tensor(batch.n_vars.astype(np.int64), device="cuda")
    w = (2 * n + 31) // 32
    per = torch.repeat_interleave(n, rows * w)                            # variables, by word
    first = torch.repeat_interleave(torch.cumsum(rows * w, 0) - rows * w, rows * w)
    j = (torch.arange(per.numel(), device="cuda") - first) % torch.repeat_interleave(w, rows * w)
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)
    out = torch.zeros(per.numel(), dtype=torch.int64, device="cuda")
    for k in range(16):
        u = torch.rand(per.numel(), generator=gen, device="cuda")
        pol = torch.rand(per.numel(), generator=gen, device="cuda") < 0.5
        on = (u < p) & (16 * j + k < per)
        out |= torch.where(on, torch.where(pol, 2, 1), 0) << (2 * k)
    return torch.where(out >= 2 ** 31, out - 2 ** 32, out).to(torch.int32)


class _Mem:
    """A torch tensor's memory as the device-buffer calls take it."""

    def __init__(self, t):
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    kind = case["kind"]
    batch = _formulas(case, seed)
    s = {"kind": kind, "gb": G.GpuBatch(batch)}
    N = batch.n_inst
    if kind in ("eval_bcp", "bcp_host"):
        R = case["rows"]
        rows = _rows(batch, R, case["p"], seed)
        s["R"] = R
        if kind == "bcp_host":
            s["rows"] = rows.cpu().numpy().view(np.uint32)
            return s
        new = lambda n: torch.empty(n, dtype=torch.int32, device="cuda")  # noqa: E731
        s["rows"] = _Mem(rows)
        s["counts"], s["out"], s["conflict"], s["props"] = (
            _Mem(new((N, R, 3))), _Mem(torch.empty_like(rows)), _Mem(new((N, R))), _Mem(new((N, R))))
        torch.cuda.synchronize()
    elif kind == "solve":
        s["opts"] = G.SolveOpts.default()
    elif kind == "cubes":
        s["opts"] = G.SolveOpts.default()
        f = [batch.instance(i) for i in range(N)]
        s["jobs"] = G.cube_jobs(batch, [G.cube_vars(x, strategy=0)[: case["depth"]] for x in f])
    else:
        s["model"] = LB.GnnModel(np.load(_weights()))
        if kind == "gnn_train":
            rng = np.random.default_rng([seed, 14])
            V = int(batch.n_vars.sum())
            s["labels"] = _labels(rng, V)
            s["graph"] = LB.GnnGraph(s["gb"])
            s["graph"].labels(*s["labels"])
    return s


def _weights():
    return LB.__file__.replace("learned.py", "branching_weights.npy")


def _labels(rng, V):
    """Targets as generate_labels makes them: scores in [0, 1], phases, phases known for some."""
    return (rng.random(V, dtype=np.float32), (rng.random(V) < 0.5).astype(np.float32),
            (rng.random(V) < 0.4).astype(np.float32))


# ---------------------------------------------------------------------------------------------
# one pass

def run(s):
    kind, gb = s["kind"], s["gb"]
    if kind == "eval_bcp":
        gb.eval_bcp_dev(s["rows"], s["R"], s["counts"], s["out"], s["conflict"], s["props"])
        return [s[k].t for k in ("counts", "out", "conflict", "props")]
    if kind == "bcp_host":
        return list(gb.bcp_fixpoint(s["rows"], s["R"]))
    if kind == "solve":
        r = gb.solve(s["opts"])
        # every counter of a job (the other fields are clock readings)
        return {"status": r["status"], "verified": r["verified"], "models": r["model_rows"],
                "counters": r["job_stats"][:, :7]}
    if kind == "cubes":
        # a caller after verdicts: which cube's model comes first is not determined
        r = gb.solve(s["opts"], jobs=s["jobs"], want_models=False)
        return {"status": r["status"], "verified": r["verified"]}
    if kind == "gnn_infer":
        g = LB.GnnGraph(gb)
        y = g.forward(s["model"])
        g.close()
        return y
    loss, grad, y = s["graph"].loss_grad(s["model"])
    return {"loss": loss, "grad": grad, "y": y}


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without

def _sizes(case):
    """(literals, clauses, variables, row words) of the whole batch (a colouring's edges on
    average)."""
    fam, N, n = case["family"], case["inst"], case["n"]
    if fam == "3sat":
        m = int(round(RATIO3 * n))
        return 3 * m * N, m * N, n * N, (2 * n + 31) // 32 * N
    if fam == "mixed":
        z = _mixed_sizes(case)
        return (sum(k * m for k, _, m in z), sum(m for _, _, m in z), sum(v for _, v, _ in z),
                sum((2 * v + 31) // 32 for _, v, _ in z))
    nodes = n // 4
    m2 = nodes * 6 + 4 * (4.5 * nodes / 2)
    L, M = N * (4 * nodes + 2 * m2), N * (nodes + m2)
    V, words = N * n, N * ((2 * n + 31) // 32)
    if fam == "structured":
        for p in (4, 5, 6, 7):
            c = max(1, N // 25)
            am = p * (p + 1) * p // 2
            L, M, V = L + c * ((p + 1) * p + 2 * am), M + c * (p + 1 + am), V + c * (p + 1) * p
            words += c * ((2 * (p + 1) * p + 31) // 32)
    return L, M, V, words


def work(case):
    """Formulas as 4-byte literals and clause offsets, rows, and outputs, each once.  A search's
    own work is not known beforehand: a solve counts its formulas and its models only."""
    kind, N = case["kind"], case["inst"]
    L, M, V, words = _sizes(case)
    arena = 4 * (L + M + N)
    if kind in ("eval_bcp", "bcp_host"):
        R = case["rows"]
        return {"bytes": arena + 8 * R * words + N * R * (20 if kind == "eval_bcp" else 8), "flops": 0}
    if kind in ("solve", "cubes"):
        return {"bytes": arena + 4 * words + 8 * N, "flops": 0}
    # per node and round: a 128- or 192-wide input times 64 outputs (clauses, literals); per
    # variable the 128-wide readout and the two outputs; the backward pass is twice that
    f = LB.ROUNDS * (M * 2 * 128 * HID + 2 * V * 2 * 192 * HID) + V * 2 * (128 * HID + 2 * HID)
    if kind == "gnn_infer":
        return {"bytes": arena + 4 * LB.param_count() + 8 * V, "flops": f}
    return {"bytes": arena + 8 * LB.param_count() + (12 + 8) * V, "flops": 3 * f}


# ---------------------------------------------------------------------------------------------
# 64-bit values

def exact(case, seed):
    """The network's outputs in 64 bits (plain torch; its weights are taken as they are, without
    the rounding to BF16).  Everything else is whole numbers."""
    if not case["kind"].startswith("gnn"):
        return None
    b = _formulas(case, seed)
    dev = "cuda"
    V = int(b.n_vars.sum())
    base = np.concatenate([[0], np.cumsum(b.n_vars.astype(np.int64))])[:-1]
    lens = np.diff(b.clause_off)
    cl = torch.as_tensor(np.repeat(np.arange(len(lens)), lens), device=dev)
    inst = np.repeat(np.arange(b.n_inst), np.diff(b.clause_off[b.inst_clause_off]))
    ln = torch.as_tensor(b.lits.astype(np.int64) + 2 * base[inst], device=dev)
    C, L = len(lens), 2 * V
    theta = torch.tensor(np.load(_weights()).astype(np.float64), device=dev, requires_grad=True)
    parts, o = [], 0
    for shp in ((HID,),) * 4 + ((HID, 2 * HID), (HID,), (HID, 3 * HID), (HID,), (HID, 2 * HID), (HID,), (2, HID), (2,)):
        k = math.prod(shp)
        parts.append(theta[o:o + k].reshape(shp))
        o += k
    u_l, v_l, u_c, v_c, W_c, b_c, W_l, b_l, W_o, b_o, W_y, b_y = parts
    occ = torch.bincount(ln, minlength=L).double()[:, None]
    size = torch.as_tensor(lens, device=dev).double()[:, None]
    other = torch.arange(L, device=dev) ^ 1
    with torch.set_grad_enabled(case["kind"] == "gnn_train"):
        Hl, Hc = occ / 8 * u_l + v_l, size / 4 * u_c + v_c
        for _ in range(LB.ROUNDS):
            Mc = torch.zeros(C, HID, dtype=torch.float64, device=dev).index_add(0, cl, Hl[ln]) / 4
            Hc = torch.relu(torch.cat([Hc, Mc], 1) @ W_c.T + b_c)
            Ml = torch.zeros(L, HID, dtype=torch.float64, device=dev).index_add(0, ln, Hc[cl]) / 8
            Hl = torch.relu(torch.cat([Hl, Ml, Hl[other]], 1) @ W_l.T + b_l)
        y = torch.relu(torch.cat([Hl[1::2], Hl[0::2]], 1) @ W_o.T + b_o) @ W_y.T + b_y
        if case["kind"] == "gnn_infer":
            return y
        t, ph, mask = (torch.as_tensor(x, device=dev).double() for x in _labels(np.random.default_rng([seed, 14]), V))
        bce = torch.nn.functional.softplus(y[:, 1]) - y[:, 1] * ph
        loss = ((y[:, 0] - t) ** 2 + mask * bce).mean()
        loss.backward()
    return {"loss": float(loss), "grad": theta.grad, "y": y.detach()}
