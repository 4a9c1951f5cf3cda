"""The block plan, its unit streams and their CPU replay under AddressSanitizer and UndefinedBehaviorSanitizer
(g++, host code only): grids whose tail is dense, grids whose tail lacks blocks (the tail is the top chain of the
elimination tree, which need not be dense), radial grids without a tail and a lone slack bus without unknowns."""
import os
import subprocess

import numpy as np
import pytest
import scipy.sparse as sp

from conftest import ROOT, load_fixture, zero_diagonal_grid
from test_sanitize import _write

BUILD = os.path.join(ROOT, "tests", "cpp", "_build")
EXE = os.path.join(BUILD, "block_sanitize")
CSRC = os.path.join(ROOT, "lightsim2grid_amd", "csrc")
SOURCES = [os.path.join(ROOT, "tests", "cpp", f) for f in ("block_sanitize.cpp", "block_replay.cpp")] + \
          [os.path.join(CSRC, f) for f in ("blocks.cpp", "analysis.cpp")]


@pytest.fixture(scope="module")
def exe():
    os.makedirs(BUILD, exist_ok=True)
    newest = max(os.path.getmtime(s) for s in SOURCES + [os.path.join(CSRC, h) for h in ("blocks.hpp", "analysis.hpp")])
    if not os.path.exists(EXE) or os.path.getmtime(EXE) < newest:
        tmp = "%s.%d.tmp" % (EXE, os.getpid())
        subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-fno-omit-frame-pointer",
                               "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-o", tmp] + SOURCES)
        os.replace(tmp, EXE)
    return EXE


def tree(parent, load=0.002):
    """A radial grid: bus k joined to bus parent[k] (< k), bus 0 the slack, small loads everywhere."""
    n = len(parent)
    k = np.arange(1, n)
    p = np.asarray(parent)[1:]
    y = np.full(n - 1, 1 / (0.01 + 0.05j))
    Y = sp.csc_matrix(sp.coo_matrix((np.r_[y, y, -y, -y], (np.r_[k, p, k, p], np.r_[k, p, p, k])), shape=(n, n))) \
        if n > 1 else sp.csc_matrix(np.ones((1, 1), complex))
    Y.sort_indices()
    S = np.full(n, -load * (1 + 0.3j))
    w = np.zeros(n)
    w[0] = 1.0
    return {"Ybus": Y, "Sbus": S, "V0": np.ones(n, complex), "slack_ids": np.zeros(1, np.int32), "slack_weights": w,
            "pv": np.zeros(0, np.int32), "pq": np.arange(1, n, dtype=np.int32)}


def _grid(name):
    from lightsim2grid_amd import gridgen
    kind, _, size = name.partition(" ")
    if kind == "feeder":  # laterals of 20 buses on a trunk of 20
        n = int(size)
        return tree([0] + [0 if k % 20 == 1 and k <= 20 else k - 20 if k <= 20 * 20 and k % 20 == 1 else k - 1
                           for k in range(1, n)], 2e-5)
    if kind == "star":
        return tree([0] * int(size))
    if kind == "alone":
        return tree([0])
    if kind == "zero":
        return zero_diagonal_grid()
    return gridgen.make(name).solver_inputs() if name.endswith("_synth") else load_fixture(name)


# tail: whether the plan has one, and whether blocks of it are absent
@pytest.mark.parametrize("name,tail,absent", [("case14_synth", True, True), ("case118_synth", True, True),
                                              ("case300", True, None), ("case2000_synth", True, True),
                                              ("feeder 401", None, None), ("star 300", False, False),
                                              ("zero diagonal", None, None), ("alone", False, False)])
def test_block_plan_under_asan_ubsan(exe, tmp_path, name, tail, absent):
    path = str(tmp_path / "grid")
    _write(path, _grid(name))
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=1:verify_asan_link_order=0",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1")
    r = subprocess.run([exe, path, "0" if name.startswith("zero") else "1"], capture_output=True, text=True, env=env,
                       timeout=600)
    assert r.returncode == 0 and r.stdout.endswith("OK\n"), (name, r.stdout[-2000:], r.stderr[-4000:])
    _, m, _, lacks, _ = r.stdout.split()
    assert tail is None or (int(m) > 0) == tail
    assert absent is None or (int(lacks) > 0) == absent
