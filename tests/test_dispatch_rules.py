"""Host rules that choose a path, compiled from the library's headers (no GPU needed)."""
import os
import shutil
import subprocess

import pytest

import gpupsat_amd as G

ROOT = os.path.dirname(G._HERE)


def run_rules(tmp_path, body):
    """Compile `body` (statements that print) against the internal headers, host pass only."""
    hipcc = next((c for c in ("/opt/rocm/bin/hipcc", shutil.which("hipcc")) if c and os.path.exists(c)), None)
    if hipcc is None:
        pytest.skip("no hipcc")
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text('#include <stdio.h>\n#include "gpsat_internal.hpp"\n#include "solver.hpp"\n'
                   "using namespace gpsat;\nint main()\n{\n" + body + "\n}\n")
    subprocess.run([hipcc, "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-O1",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(G._HERE, "csrc"), str(src), "-o", str(exe),
                    "-L" + G._HERE, "-lgpsat", "-Wl,-rpath," + G._HERE], check=True, capture_output=True, text=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()


def test_gnn_graph_is_built_where_its_batch_is(tmp_path):
    """A graph on another device than its batch is built from the host's copies."""
    got = run_rules(tmp_path, """
    DeviceBatch d;
    d.n_inst = 4; d.max_n = 100; d.max_len = 3; d.max_lits = 1278; d.n_lits = 4 * 1278;
    for (int batch : {0, 1})
        for (int dev : {0, 1}) {
            d.device = batch;
            printf("%d ", (int)gnn_graph_on_device(d, dev));
        }""")
    assert got == ["1", "0", "0", "1"]


def test_large_formulas_keep_their_memory_per_wavefront(tmp_path):
    """Bytes of a wavefront's state with 32-bit ids: 63 a variable, two watch list entries of 4
    for each learned-clause slot of its literals, 4 a literal and 8 a clause (4 where all have
    three literals: the one that is not watched), 53 a learned clause besides the
    literals it may hold, and at most 1 KB of rounding (each of 19 arrays to 16 bytes, 64 entries
    read past two of them)."""
    got = run_rules(tmp_path, """
    SolveOptsDev o{};
    for (int all3 : {0, 1})
        for (int n : {17, 5000, 100000})
            for (int m : {66000, 1000001}) {
                o.learnt_cap = 256; o.larena_cap = 32 * 256 + n; o.watch_slack = 8;
                const long L = 3l * m + (all3 ? 0 : 12345);
                const SolveLayout lay = solve_layout(n, m, L, all3, 4, o);
                const long most = 63l * n + 2l * n * 8 * 4 + 4 * L + (all3 ? 4l : 8l) * m + 53l * o.learnt_cap + 4l * o.larena_cap + 1024;
                printf("%d ", (int)(lay.state_bytes + lay.watch_bytes + lay.arena_bytes <= most));
            }""")
    assert got == ["1"] * 12


def test_gnn_graph_of_one_large_instance_is_built_on_the_host(tmp_path):
    """(edges of each instance, instances) on either side of the line, and the kernel's limits:
    variables, clause length, edges."""
    got = run_rules(tmp_path, """
    struct { long lits; int inst, n, len; } c[] = {
        {300, 1, 100, 3}, {8000, 1, 600, 3}, {12500, 1, 900, 3}, {12501, 1, 900, 3}, {32000, 1, 1900, 3}, {32000, 2, 1900, 3},
        {32000, 3, 1900, 3}, {65000, 2, 1900, 3}, {65536, 3, 1984, 64}, {65537, 3, 1984, 64}, {65536, 3, 1985, 64},
        {65536, 3, 1984, 65}};
    for (auto& x : c) {
        DeviceBatch d;
        d.n_inst = x.inst; d.max_n = x.n; d.max_len = x.len; d.max_lits = x.lits; d.n_lits = x.lits * x.inst;
        printf("%d ", (int)gnn_graph_on_device(d, d.device));
    }""")
    assert got == list("111000101000")
