"""The block plan of launches that keep a part of the values outside LDS (lightsim2grid_amd/csrc/blocks.cpp), on the
CPU: at cuts from the fewest pairs in LDS to one pair short of all, every address that the kernel forms on the units
lies in its part, every unit that reaches outside LDS is marked, no block straddles the cut, and the tail is in LDS.
Also with a constant J, the plan of fast-decoupled grids."""
import ctypes
import os
import subprocess

import numpy as np
import pytest
import scipy.sparse as sp

from conftest import ROOT
from test_block_plan import _grid

CPP = os.path.join(ROOT, "tests", "cpp")
CSRC = os.path.join(ROOT, "lightsim2grid_amd", "csrc")
SO = os.path.join(CPP, "libblockspill.so")
SRC = [os.path.join(CPP, "block_spill.cpp"), os.path.join(CSRC, "blocks.cpp"), os.path.join(CSRC, "analysis.cpp")]


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(SO) or os.path.getmtime(SO) < max(os.path.getmtime(s) for s in SRC + [os.path.join(CSRC, "blocks.hpp")]):
        tmp = "%s.%d.tmp" % (SO, os.getpid())
        subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", tmp] + SRC)
        os.replace(tmp, SO)
    return ctypes.CDLL(SO)


def check(lib, d, single, const, G, waves, fsize, rooms):
    Y = sp.csc_matrix(d["Ybus"])
    Y.sort_indices()
    i32 = lambda a: np.ascontiguousarray(np.atleast_1d(a), np.int32)  # noqa: E731
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    Yp, Yi, sl, pv, pq, rooms = map(i32, (Y.indptr, Y.indices, d["slack_ids"], d["pv"], d["pq"], rooms))
    w, info = np.ascontiguousarray(d["slack_weights"], float), np.zeros(6, np.int32)
    bad = lib.block_spill_check(Y.shape[0], p(Yp), p(Yi), p(sl), len(sl), p(w), p(pv), len(d["pv"]), p(pq), len(d["pq"]),
                                int(single), int(const), G, waves, fsize, len(rooms), p(rooms), p(info))
    return bad, info


@pytest.mark.parametrize("name", ["3 buses", "5 buses, no pv", "40 buses, 30 pv", "333 buses", "case118_synth",
                                  "case2000_synth", "case300"])
@pytest.mark.parametrize("const", [False, True])
@pytest.mark.parametrize("G,waves,fsize", [(1, 16, 8), (1, 4, 4), (4, 16, 8), (8, 4, 4)])
def test_units_reach_what_is_there(lib, name, const, G, waves, fsize):
    d = _grid(name)
    single = const  # a fast-decoupled J has no slack unknown
    _, info = check(lib, d, single, const, G, waves, fsize, [])
    n, fixed = int(info[0]), int(info[1])
    # every cut near both ends (where two of three neighbours split a block of two pairs), some between
    rooms = sorted({r for r in list(range(fixed, fixed + 4)) + list(range(n - 5, n + 1)) +
                    np.linspace(fixed, n, 6).astype(int).tolist() if r >= fixed})
    bad, info = check(lib, d, single, const, G, waves, fsize, rooms)
    assert bad == 0 and info[5] == 0
    assert info[2] >= min(len(rooms) - 1, 4) or n - fixed < 5
    if n > 1000:
        assert info[3] > 0 and info[4] > 0
