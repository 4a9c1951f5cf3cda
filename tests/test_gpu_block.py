"""The block-plan kernel at the edges of its launch shapes and phases, against the oracle: no dense tail, tails
of each code size of the wave that factors them, tails cut at the largest,
V beside the values, over them and in memory, values spilled, several instances per workgroup in both block
sizes, Ybus edits inside and beyond the eight kept in LDS, one and two batches of rows per lane.
Bar: the FP64 form the oracle's flags and iterations and |V - V_oracle| <= 1e-8; the FP32 form the same flags,
iterations within one and 5e-8."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


def _grid(n, per_bus, seed, loading):
    from lightsim2grid_amd import gridgen
    return gridgen.generate(n, int(n * per_bus), max(1, n // 4), seed, distributed_slack=n > 60, loading=loading)


def _check(oracle_mod, ctx, g, conts, prec, G, block=None):
    from lightsim2grid_amd import abi
    d = g.solver_inputs()
    o = oracle_mod.OracleNR(False)
    assert o.compute_pf(d["Ybus"], d["V0"], d["Sbus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], 10, 1e-8)
    Vb = o.get_V()
    deltas = g.ybus_deltas(conts)
    Vr, itr, _, conv, conn, _ = oracle_mod.contingency(d["Ybus"], d["Sbus"], d["slack_ids"], d["slack_weights"], d["pv"],
                                                       d["pq"], Vb, deltas, 10, 1e-8, False, False, 4)
    gr = abi.Grid(ctx, d["Ybus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"])
    r = gr.solve(gr.ybus_values(d["Ybus"]), d["Sbus"], Vb, 10, 1e-8, precision=prec, deltas=deltas, instances_per_wg=G)
    ok = conv & conn
    assert np.array_equal((r["status"] == 0)[conn], ok[conn])
    assert np.max(np.abs(r["iters"][ok] - itr[ok])) <= (0 if prec == abi.FP64 else 1)
    assert np.max(np.abs(r["V"][ok] - Vr[ok])) <= (1e-8 if prec == abi.FP64 else 5e-8)
    return r["stats"]


# buses, branches per bus, seed, loading: top chains of 0, 8, 17, 30, 38, 51, 84 and 70 unknowns (the tail takes
# at most 48 of them), the last one with more than 64 levels (two words of the waves' level masks)
TAILS = [(6, 1.2, 3, 0.3), (12, 1.3, 1, 0.5), (250, 1.7, 4, 0.2), (400, 1.9, 4, 0.15), (500, 2.4, 6, 0.12),
         (400, 3.3, 1, 0.15), (700, 3.3, 1, 0.12), (1200, 3.3, 2, 0.1)]


@pytest.mark.parametrize("n,per_bus,seed,loading", TAILS)
@pytest.mark.parametrize("prec", [0, 2])
@pytest.mark.parametrize("G", [1, 2, 4])
def test_block_kernel_tails_and_shapes(gpu_ctx, oracle_mod, n, per_bus, seed, loading, prec, G):
    g = _grid(n, per_bus, seed, loading)
    _say("block", n, per_bus, prec, G)
    rng = np.random.default_rng(seed)
    conts = [[int(k)] for k in rng.choice(g.nbr, min(g.nbr, 11), replace=False)]
    _check(oracle_mod, gpu_ctx, g, conts, prec, G)


@pytest.mark.parametrize("k", [1, 2, 3, 5])
@pytest.mark.parametrize("prec", [0, 2])
def test_block_kernel_edits_per_instance(gpu_ctx, oracle_mod, k, prec):
    """4 k edits per instance, 8 of them kept in LDS; outages that share a bus edit one row several times."""
    from lightsim2grid_amd import gridgen
    g = gridgen.make("case118_synth")
    _say("block edits", k, prec)
    lines = np.nonzero(~gridgen.bridges(g))[0]
    rng = np.random.default_rng(k)
    conts = [sorted(int(x) for x in rng.choice(lines, k, replace=False)) for _ in range(9)]
    _check(oracle_mod, gpu_ctx, g, conts, prec, 1)


@pytest.mark.parametrize("n,prec", [(1023, 0), (1025, 0), (1400, 0), (2049, 2), (1900, 2), (2300, 2), (3100, 2)])
def test_block_kernel_where_v_and_values_lie(gpu_ctx, oracle_mod, n, prec):
    """From V beside the values over V laid over them and V in memory to values spilled; rows of one batch, of
    one batch and a row, of several."""
    g = _grid(n, 1.35, 7, 0.2)
    _say("block memory", n, prec)
    rng = np.random.default_rng(n)
    conts = [[int(k)] for k in rng.choice(g.nbr, 5, replace=False)]
    _check(oracle_mod, gpu_ctx, g, conts, prec, 1)


@pytest.mark.parametrize("prec", [0, 1])
def test_shortest_time_launch_with_and_without_a_block_form(gpu_ctx, oracle_mod, prec):
    """instances_per_wg = -1: on the block plan bit-equal to one workgroup of 1024 lanes per instance; on the plan
    of a re-pivoted grid, which has no block form, the wide kernel, equal to the oracle."""
    from conftest import zero_diagonal_grid
    from lightsim2grid_amd import abi
    _say("shortest time", prec)
    g = _grid(900, 1.5, 3, 0.3)
    d = g.solver_inputs()
    gr = abi.Grid(gpu_ctx, d["Ybus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"])
    a = (gr.ybus_values(d["Ybus"]), d["Sbus"], d["V0"], 10, 1e-8)
    r = gr.solve(*a, precision=prec, instances_per_wg=-1)
    gr.reset()
    r1 = gr.solve(*a, precision=prec, instances_per_wg=1)
    assert r["stats"]["instances_per_wg"] == -1 and r1["stats"]["instances_per_wg"] == 1
    assert r["status"][0] == 0 and np.max(np.abs(r["V"] - r1["V"])) <= (1e-9 if prec == abi.FP64 else 5e-8)
    if r1["stats"]["block_size"] == r["stats"]["block_size"]:
        assert np.array_equal(r["V"], r1["V"])

    d = zero_diagonal_grid()
    o = oracle_mod.OracleNR(False)
    assert o.compute_pf(d["Ybus"], d["V0"], d["Sbus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], 10, 1e-8)
    gr = abi.Grid(gpu_ctx, d["Ybus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"])
    Yx = gr.ybus_values(d["Ybus"])
    for _ in range(2):  # the plan is kept: the second solve runs on it alone
        r = gr.solve(Yx, d["Sbus"], d["V0"], 10, 1e-8, precision=prec, instances_per_wg=-1)
        assert r["stats"]["instances_per_wg"] == -1
        assert r["status"][0] == 0 and r["iters"][0] == o.get_nb_iter()
        assert np.max(np.abs(r["V"][0] - o.get_V())) <= 1e-8
    assert r["stats"]["workgroups"] > 1  # the wide kernel's


@pytest.mark.parametrize("n,rows,prec,more", [(60, 600, 0, False), (118, 1100, 0, True), (118, 2000, 2, True),
                                              (10000, 800, 0, True), (10000, 600, 0, False)])
def test_default_launch_shape_equals_one_instance_per_workgroup(gpu_ctx, n, rows, prec, more):
    """The shape that a launch takes by itself (`more`: several instances per workgroup) against G = 1: equal
    statuses, FP64 equal iterations and |dV| <= 1e-9, FP32 the bound of the FP32 form."""
    from lightsim2grid_amd import abi, gridgen
    _say("default shape", n, rows, prec)
    g = gridgen.make(f"case{n}_synth") if n in (118, 10000) else gridgen.generate(n, n + n // 3, n // 4, 3, loading=0.3)
    d = g.solver_inputs()
    gr = abi.Grid(gpu_ctx, d["Ybus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"])
    Yx = gr.ybus_values(d["Ybus"])
    base = gr.solve(Yx, d["Sbus"], d["V0"], 10, 1e-8)
    assert base["status"][0] == 0
    lines = np.nonzero(~gridgen.bridges(g))[0]
    deltas = g.ybus_deltas([[int(lines[k % len(lines)])] for k in range(rows)])
    r0, r1 = (gr.solve(Yx, d["Sbus"], base["V"][0], 10, 1e-8, precision=prec, deltas=deltas, instances_per_wg=G)
              for G in (0, 1))
    assert (r0["stats"]["instances_per_wg"] > 1) == more
    assert np.array_equal(r0["status"], r1["status"])
    ok = r1["status"] == 0
    if prec == abi.FP64:
        assert np.array_equal(r0["iters"][ok], r1["iters"][ok])
    assert np.max(np.abs(r0["V"][ok] - r1["V"][ok])) <= (1e-9 if prec == abi.FP64 else 5e-8)
