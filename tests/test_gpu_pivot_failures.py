"""Pivot failures on grids without a dense tail (a top chain of fewer than 8 unknowns), met by lanes of every wave
of the workgroup: the statuses of the oracle's failing factorisations (5 on a fresh solver, then 6) and the re-pivot
that status 5 starts. One wave reads what another one found, with no tail's barrier between them."""
import sys

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


def _inputs(f, t, y, load, pv=()):
    f, t, y = np.array(f), np.array(t), np.array(y, complex)
    n = int(max(f.max(), t.max())) + 1
    Y = sp.csc_matrix(sp.coo_matrix((np.r_[y, y, -y, -y], (np.r_[f, t, f, t], np.r_[f, t, t, f])), shape=(n, n)))
    Y.sort_indices()
    w = np.zeros(n)
    w[0] = 1.0
    pv = np.array(pv, np.int32)
    return {"Ybus": Y, "Sbus": np.full(n, -load * (1 + 0.3j)), "V0": np.ones(n, complex),
            "slack_ids": np.zeros(1, np.int32), "slack_weights": w, "pv": pv,
            "pq": np.setdiff1d(np.arange(1, n), pv).astype(np.int32)}


def star(n, dc=False):
    """Bus 0, the slack, joined to each of the others: every pivot has nothing to eliminate."""
    return _inputs([0] * (n - 1), range(1, n), [16.0 if dc else 4 - 16j] * (n - 1), 1e-3)


def tailless_zero_diagonal_grid():
    """100 hubs of 6 leaves at the slack bus, three PV buses in a ring and a PQ bus whose three lines to them add up
    to an admittance of 0: its diagonal J block is exactly 0 at a flat start, and eliminated before its neighbours."""
    f, t, y = [], [], []
    n = 1
    for _ in range(100):
        f += [0] + [n] * 6
        t += range(n, n + 7)
        n += 7
    y = [4 - 16j] * len(f)
    a, b, c, z = range(n, n + 4)
    f += [a, b, a, 0, z, z, z]
    t += [b, c, c, a, a, b, c]
    y += [4 - 16j] * 4 + [2 - 8j, 1 - 3j, -3 + 11j]
    d = _inputs(f, t, y, 1e-4, (a, b, c))
    d["Sbus"][[a, b, c]] = -1e-3
    d["Sbus"][z] = 0
    assert d["Ybus"][z, z] == 0
    return d


@pytest.mark.parametrize("bus", [1, 70, 150, 299])
@pytest.mark.parametrize("prec,G", [(0, 1), (2, 1), (0, 2), (0, 4)])
def test_zero_pivot_in_any_wave_without_a_tail(gpu_ctx, oracle_mod, bus, prec, G):
    from lightsim2grid_amd import abi
    d = star(300)
    Y = d["Ybus"].copy()
    Y.data[(Y.indices == bus) | (np.repeat(np.arange(300), np.diff(Y.indptr)) == bus)] = 0
    _say("zero pivot, no tail", bus, prec, G)
    o = oracle_mod.OracleNR(False)
    e = []
    for _ in range(2):
        assert not o.compute_pf(Y, d["V0"], d["Sbus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], 10, 1e-8)
        e.append(o.get_error())
    assert e == [5, 6]
    gr = abi.Grid(gpu_ctx, Y, d["slack_ids"], d["slack_weights"], d["pv"], d["pq"])
    V0 = np.repeat(d["V0"][None, :], 3, axis=0)
    for want in e:
        r = gr.solve(gr.ybus_values(Y), d["Sbus"], V0, 10, 1e-8, precision=prec, instances_per_wg=G)
        assert np.all(r["status"] == want)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("single", [False, True])
def test_repivot_without_a_tail(gpu_ctx, oracle_mod, prec, single):
    from lightsim2grid_amd import abi
    d = tailless_zero_diagonal_grid()
    _say("repivot, no tail", prec, single)
    o = oracle_mod.OracleNR(single)
    assert o.compute_pf(d["Ybus"], d["V0"], d["Sbus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], 10, 1e-8)
    gr = abi.Grid(gpu_ctx, d["Ybus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], single_slack=single)
    V0 = np.repeat(d["V0"][None, :], 3, axis=0)
    r = gr.solve(gr.ybus_values(d["Ybus"]), d["Sbus"], V0, 10, 1e-8, precision=prec)
    assert r["stats"]["repivot_rows"] == 3
    assert np.all(r["status"] == 0) and np.all(r["iters"] == o.get_nb_iter())
    assert np.max(np.abs(r["V"] - o.get_V()[None, :])) <= 1e-8


@pytest.mark.parametrize("bus", [1, 70, 150, 297])
def test_dc_zero_pivot_of_the_walk_without_a_tail(gpu_ctx, oracle_mod, bus):
    """Two buses cut off from the slack: the second one's pivot is 16 - 16 * 16 / 16 = 0 after the first."""
    from lightsim2grid_amd import abi
    d = star(300, dc=True)
    f, t = list(range(300)), [0] * 300
    f[bus + 1], t[bus + 1] = bus + 1, bus
    keep = [k for k in range(1, 300) if k != bus]
    d["Ybus"] = _inputs([f[k] for k in keep], [t[k] for k in keep], [16.0] * len(keep), 0)["Ybus"]
    _say("dc zero pivot, no tail", bus)
    _, err = oracle_mod.dc_pf(d["Ybus"], d["V0"], d["Sbus"], d["slack_ids"], d["pv"], d["pq"])
    assert err != 0
    gr = abi.Grid(gpu_ctx, d["Ybus"], d["slack_ids"], None, d["pv"], d["pq"], dc=True)
    V0 = np.repeat(d["V0"][None, :], 2, axis=0)
    for want in (5, 6):
        r = gr.solve(gr.ybus_values(d["Ybus"]), d["Sbus"], V0, 10, 1e-8, precision=abi.FP64, instances_per_wg=1)
        assert np.all(r["status"] == want)
