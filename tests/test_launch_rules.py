"""The rules that choose a batch's launch shape (launch_rules.hpp), compiled
for the CPU."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "launch_rules.hpp"
using namespace mtk;
extern "C" void layer_rows_of(int n, const long *j, int *rows) {  // j: matched, tuned, fits2, fits, nodes
    std::vector<LayerJob> v;
    for (int i = 0; i < n; i++, j += 5) v.push_back(LayerJob{j[0] != 0, (int)j[1], j[2] != 0, j[3] != 0, j[4]});
    const std::vector<int> r = layer_rows(v);
    for (int i = 0; i < n; i++) rows[i] = r[i];
}
extern "C" int pick_cs_of(int n, const long *wg, const int *ns, int cmax, int thresh, int thresh4) {
    std::vector<std::pair<long, int>> v;
    for (int i = 0; i < n; i++) v.push_back({wg[i], ns[i]});
    return pick_cs(v, cmax, thresh, thresh4);
}
extern "C" void descent_of(int fits2, int fits, double (*timed)(const int *), int *best) {
    group_descent(fits2 != 0, fits != 0, timed, best);
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(SRC)
    so = str(d / "librules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I" + os.path.join(ROOT, "maos_amd", "csrc", "hip"), str(d / "rules.cpp"), "-o", so], check=True)
    return C.CDLL(so)


def rows_of(rules, jobs):
    flat = [int(v) for j in jobs for v in j]
    out = (C.c_int * len(jobs))()
    rules.layer_rows_of(len(jobs), (C.c_long * len(flat))(*flat), out)
    return list(out)


def job(nodes, tuned=0, fits2=True, fits=True, matched=True):
    return (matched, tuned, fits2, fits, nodes)


L30, M20, S8 = 55296, 16384, 3136  # layer nodes of one 30 m, 20 m and 8 m system


@pytest.mark.parametrize("jobs,rows", [
    ([job(L30)], [16]),                                        # one system
    ([job(2 * L30)], [32]),                                    # two of one plan
    ([job(L30)] * 2, [32] * 2),                                # two plans of one each: the same launch
    ([job(M20)] * 6, [16] * 6),                                # 98 304 nodes
    ([job(M20)] * 7, [32] * 7),                                # 114 688
    ([job(L30)] * 32, [32] * 32),
    ([job(L30), job(L30, matched=False)], [16, 16]),           # the generic kernel's nodes are another launch's
    ([job(L30, 16), job(12 * L30)], [16, 32]),                 # a tuned choice stays
    ([job(L30, 16), job(L30)], [16, 16]),
    ([job(L30, 32), job(L30)], [32, 32]),
    ([job(L30, 64), job(L30, 64, fits=False)], [64, 16]),
    ([job(M20, 32), job(S8, 32, fits2=False)], [32, 16]),
    # members whose layers are too small for 32 rows need a launch of their
    # own beside them, which large members have to repay
    ([job(L30)] * 8 + [job(S8, fits2=False, fits=False)] * 8, [16] * 16),
    ([job(L30)] * 16 + [job(S8, fits2=False, fits=False)] * 8, [32] * 16 + [16] * 8),
])
def test_layer_rows(rules, jobs, rows):
    assert rows_of(rules, jobs) == rows


@pytest.mark.parametrize("jw,cmax,cs", [
    # (workgroups per system, systems) per job; 512 workgroups for 2, 1100 for 4
    ([(96, 1)], 4, 1),
    ([(96, 10)], 4, 1),
    ([(96, 11)], 4, 2),
    ([(96, 45)], 4, 4),
    ([(96, 45)], 2, 2),
    ([(36, 29)], 4, 2),
    # jobs of one system fill one slot however many there are
    ([(96, 1)] * 6, 4, 1),
    ([(96, 1)] * 32, 4, 1),
    ([(96, 2)] * 16, 4, 2),
    ([(96, 3)] * 16, 4, 1),
    ([(96, 4)] * 16, 4, 4),
    # a few of them beside a large job leave its choice
    ([(96, 48), (36, 1)], 4, 4),
    ([(96, 4)] + [(96, 1)] * 20, 4, 1),
])
def test_systems_per_workgroup(rules, jw, cmax, cs):
    wg = (C.c_long * len(jw))(*[w for w, _ in jw])
    ns = (C.c_int * len(jw))(*[n for _, n in jw])
    assert rules.pick_cs_of(len(jw), wg, ns, cmax, 512, 1100) == cs


@pytest.mark.parametrize("fits2,fits", [(1, 1), (1, 0), (0, 0)])
@pytest.mark.parametrize("rows", [0, 16, 32, 64])
@pytest.mark.parametrize("col", [0, 2])
def test_group_descent_finds_the_fastest(rules, rows, col, fits2, fits):
    """The search times every layer tile shape that fits and both column
    kernels, and keeps the fastest (0: the built-in choice)."""
    tried = []

    def timed(c):
        tried.append(list(c[:6]))
        return 1.0 + 0.1 * (c[3] != rows) + 0.1 * (c[4] != col) + 0.1 * (c[0] != 2) + 0.01 * (c[1] != 1)

    best = (C.c_int * 6)()
    rules.descent_of(fits2, fits, C.CFUNCTYPE(C.c_double, C.POINTER(C.c_int))(timed), best)
    shapes = {0, 16} | ({32} if fits2 else set()) | ({64} if fits else set())
    assert tried[0] == [0, 0, 0, 0, 0, 1]
    assert {t[3] for t in tried} == shapes
    assert list(best) == [2, 0, 0, rows if rows in shapes else 0, col, 1]
