"""Batches in contexts whose HBM budget holds less than the launch would take by itself: they run with fewer instances
side by side, with the results of an ample budget bit for bit where the launch shape is the same."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


def _solve(ctx, g, base, rows, prec, G):
    from lightsim2grid_amd import abi, gridgen
    d = g.solver_inputs()
    gr = abi.Grid(ctx, d["Ybus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"])
    lines = np.nonzero(~gridgen.bridges(g))[0]
    deltas = g.ybus_deltas([[int(lines[k % len(lines)])] for k in range(rows)])
    try:
        return gr.solve(gr.ybus_values(d["Ybus"]), d["Sbus"], base, 10, 1e-8, precision=prec, deltas=deltas,
                        instances_per_wg=G)
    finally:
        gr.close()


def _base(ctx, g):
    from lightsim2grid_amd import abi
    d = g.solver_inputs()
    gr = abi.Grid(ctx, d["Ybus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"])
    r = gr.solve(gr.ybus_values(d["Ybus"]), d["Sbus"], d["V0"], 10, 1e-8)
    gr.close()
    assert r["status"][0] == 0
    return r["V"][0]


@pytest.mark.parametrize("prec", [0, 2])
@pytest.mark.parametrize("budget,rows", [(1 << 20, 64), (1 << 19, 3), (4 << 20, 300)])
def test_shortest_time_launches_in_a_small_budget(gpu_ctx, prec, budget, rows):
    """instances_per_wg = -1 needs the workspace of one instance, however many there are."""
    from lightsim2grid_amd import abi, gridgen
    _say("small budget, -1", budget, rows, prec)
    g = gridgen.make("case2000_synth")
    V = _base(gpu_ctx, g)
    want = _solve(gpu_ctx, g, V, rows, prec, -1)
    ctx = abi.Context(0, budget)
    got = _solve(ctx, g, V, rows, prec, -1)
    ctx.close()
    assert got["stats"]["resident_workgroups"] <= want["stats"]["resident_workgroups"]
    for k in ("V", "iters", "status"):
        assert np.array_equal(got[k], want[k])


def test_large_fp64_batch_in_a_smaller_budget(gpu_ctx):
    """10 000 buses in FP64 take four instances per workgroup where the budget holds them, else one."""
    from lightsim2grid_amd import abi, gridgen
    _say("small budget, 10 000 buses")
    g = gridgen.make("case10000_synth")
    V, rows = _base(gpu_ctx, g), 1100
    r4 = _solve(gpu_ctx, g, V, rows, 0, 0)
    ctx = abi.Context(0, 800 << 20)
    r1 = _solve(ctx, g, V, rows, 0, 0)
    ctx.close()
    assert (r4["stats"]["instances_per_wg"], r1["stats"]["instances_per_wg"]) == (4, 1)
    assert np.array_equal(r4["status"], r1["status"]) and np.array_equal(r4["iters"], r1["iters"])
    ok = r1["status"] == 0
    assert np.max(np.abs(r4["V"][ok] - r1["V"][ok])) <= 1e-9


@pytest.mark.parametrize("name,rows,prec,G,budget", [("case10000_synth", 1100, 0, 8, 720e6), ("case10000_synth", 1100, 0, 1, 337e6),
                                                     ("case2000_synth", 600, 0, 1, 37.5e6), ("case118_synth", 9000, 0, 32, 95e6)])
def test_shapes_asked_for_in_a_budget_of_the_scalar_plans(gpu_ctx, name, rows, prec, G, budget):
    """What the scalar plan of a grid took for a launch shape is enough for the block plan's, at the most with fewer
    instances or workgroups side by side."""
    from lightsim2grid_amd import abi, gridgen
    _say("small budget, shapes", name, rows, prec, G)
    g = gridgen.make(name)
    V = _base(gpu_ctx, g)
    want = _solve(gpu_ctx, g, V, rows, prec, G)
    ctx = abi.Context(0, int(budget))
    got = _solve(ctx, g, V, rows, prec, G)
    ctx.close()
    assert np.array_equal(got["status"], want["status"]) and np.array_equal(got["iters"], want["iters"])
    ok = want["status"] == 0
    assert np.max(np.abs(got["V"][ok] - want["V"][ok])) <= 1e-9
    if G in (1, 32):
        assert got["stats"]["instances_per_wg"] == G and np.array_equal(got["V"], want["V"])


def test_autotune_in_a_budget_of_the_scalar_plans(gpu_ctx):
    from lightsim2grid_amd import abi, gridgen
    _say("small budget, autotune")
    g = gridgen.make("case10000_synth")
    d = g.solver_inputs()
    V, rows = _base(gpu_ctx, g), 520
    lines = np.nonzero(~gridgen.bridges(g))[0]
    deltas = g.ybus_deltas([[int(k)] for k in lines[:rows]])
    out = []
    for ctx in (gpu_ctx, abi.Context(0, 720_000_000)):
        gr = abi.Grid(ctx, d["Ybus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"])
        dev = ctx.to_device
        a = (dev(gr.ybus_values(d["Ybus"])), 0, dev(np.ascontiguousarray(d["Sbus"])), 0, dev(V), 0,
             ctx.empty((rows, g.n), np.complex128), rows, ctx.empty(rows, np.int32), ctx.empty(rows, np.int32))
        dd = tuple(dev(x) for x in deltas)
        if ctx is not gpu_ctx:
            gr.autotune_device(*a, precision=0, deltas=dd)
        gr.solve_device(*a, precision=0, deltas=dd)
        out.append((a[9].to_host(), a[8].to_host(), a[6].to_host()))
        gr.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    ok = out[0][0] == 0
    assert np.max(np.abs(out[0][2][ok] - out[1][2][ok])) <= 1e-9
