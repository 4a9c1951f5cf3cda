"""The block plan of the factorisation (lightsim2grid_amd/csrc/blocks.cpp) replayed on the CPU, unit by
unit of its lane streams, against the oracle: same converged flag and iteration count, |V - V_oracle| <=
1e-8, and no two tasks of a level that touch the same place. Values start as NaN, so a read of a place
that nothing wrote fails the solve. Grids from 3 buses (no dense tail) over PV-heavy and PQ-only ones
to the largest fixture; launch shapes from 1 to 32 instances per workgroup, 4 and 16 waves."""
import ctypes
import os
import subprocess

import numpy as np
import pytest
import scipy.sparse as sp

from conftest import FIXTURES, ROOT, load_fixture

SO = os.path.join(ROOT, "tests", "cpp", "libblockreplay.so")
SRC = [os.path.join(ROOT, "tests", "cpp", "block_replay.cpp"),
       os.path.join(ROOT, "lightsim2grid_amd", "csrc", "blocks.cpp"),
       os.path.join(ROOT, "lightsim2grid_amd", "csrc", "analysis.cpp")]


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(SO) or os.path.getmtime(SO) < max(os.path.getmtime(s) for s in SRC):
        subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", SO] + SRC)
    return ctypes.CDLL(SO)


def _grid(name):
    if name in FIXTURES:
        return load_fixture(name)
    from lightsim2grid_amd import gridgen
    if name.endswith("_synth"):
        return gridgen.make(name).solver_inputs()
    n, npv, seed, dist = {"3 buses": (3, 1, 1, False), "5 buses, no pv": (5, 0, 2, False),
                          "40 buses, 30 pv": (40, 30, 3, True), "333 buses": (333, 80, 5, True)}[name]
    return gridgen.generate(n, n + n // 4 if n > 3 else 3, npv, seed, distributed_slack=dist,
                            loading=0.3 if n > 5 else 0.5).solver_inputs()


def replay(lib, d, single, G, waves, by_life):
    Y = sp.csc_matrix(d["Ybus"])
    Y.sort_indices()
    n = Y.shape[0]
    i32 = lambda a: np.ascontiguousarray(np.atleast_1d(a), np.int32)  # noqa: E731
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    Yp, Yi, Yx = i32(Y.indptr), i32(Y.indices), np.ascontiguousarray(Y.data, np.complex128)
    S, V = np.ascontiguousarray(d["Sbus"], np.complex128), np.array(d["V0"], np.complex128)
    sl, w, pv, pq = i32(d["slack_ids"]), np.ascontiguousarray(d["slack_weights"], float), i32(d["pv"]), i32(d["pq"])
    st, info = ctypes.c_int(), np.zeros(6, np.int32)
    it = lib.block_replay_solve(n, p(Yp), p(Yi), p(Yx), p(S), p(sl), len(sl), p(w), p(pv), len(d["pv"]), p(pq),
                                len(d["pq"]), int(single), p(V), 10, ctypes.c_double(1e-8), G, waves, by_life,
                                ctypes.byref(st), p(info))
    return it, st.value, V, info


@pytest.mark.parametrize("name", ["3 buses", "5 buses, no pv", "40 buses, 30 pv", "333 buses", "case14_synth",
                                  "case118_synth", "case2000_synth"] + list(FIXTURES))
def test_block_plan_solves_as_the_oracle(lib, oracle_mod, name):
    d = _grid(name)
    for single in ([False, True] if len(np.atleast_1d(d["slack_ids"])) == 1 else [False]):
        o = oracle_mod.OracleNR(single)
        conv = o.compute_pf(d["Ybus"], d["V0"], d["Sbus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], 10, 1e-8)
        for G, waves in ((1, 16), (1, 4), (2, 4), (4, 16), (32, 16)):
            it, st, V, info = replay(lib, d, single, G, waves, int(G != 1))
            assert info[5] == 0
            assert (st == 0) == conv and it == o.get_nb_iter()
            assert np.max(np.abs(V - o.get_V())) <= 1e-8
