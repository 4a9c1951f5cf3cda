"""The scalar plan of AC and fast-decoupled grids (the k_nr kernel, and the wide kernel at instances_per_wg = -1), which
serves a grid once its pivots were chosen off J's diagonal: contingencies, chains of time steps and fast-decoupled
solves on re-pivoted grids of 119 and 2001 buses, values in LDS and spilled, one and several instances per workgroup,
distributed and single slack, against the oracle. Bars as elsewhere: FP64 form equal flags and iterations and
|V - V_oracle| <= 1e-8; FP32 form equal flags, iterations within one and 5e-8."""
import sys

import numpy as np
import pytest

from conftest import zero_diagonal_grid

pytestmark = pytest.mark.gpu

FP64, FP32_STRICT = 0, 2
ENDS = {"case118_synth": (65, 117), "case2000_synth": (147, 1074)}  # buses of many lines: the new bus goes before them


def _say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


def _args(d):
    return d["slack_ids"], d["slack_weights"], d["pv"], d["pq"]


def _repivoted(ctx, oracle_mod, name, single=False):
    """A grid whose first solve has chosen its pivots, and the oracle's solution."""
    from lightsim2grid_amd import abi
    d = zero_diagonal_grid(*ENDS[name], name=name)
    o = oracle_mod.OracleNR(single)
    assert o.compute_pf(d["Ybus"], d["V0"], d["Sbus"], *_args(d), 10, 1e-8)
    gr = abi.Grid(ctx, d["Ybus"], *_args(d), single_slack=single)
    Yx = gr.ybus_values(d["Ybus"])
    r = gr.solve(Yx, d["Sbus"], d["V0"], 10, 1e-8, precision=FP64)
    assert r["stats"]["repivot_rows"] == 1 and r["status"][0] == 0 and r["iters"][0] == o.get_nb_iter()
    assert np.max(np.abs(r["V"][0] - o.get_V())) <= 1e-8
    return d, gr, Yx, o.get_V()


def _deltas(g, d, lines):
    """Outages of g's lines on the pattern of the grid with the new bus."""
    dptr, dpos, dval = g.ybus_deltas([[int(k)] for k in lines])
    Y, Y2 = g.ybus(), d["Ybus"]
    col = np.repeat(np.arange(g.n), np.diff(Y.indptr))[dpos]
    row = Y.indices[dpos]
    pos = [Y2.indptr[c] + int(np.searchsorted(Y2.indices[Y2.indptr[c]:Y2.indptr[c + 1]], r)) for r, c in zip(row, col)]
    return dptr, np.array(pos, np.int32), dval


@pytest.mark.parametrize("name,single,G", [("case118_synth", False, G) for G in (0, 1, 2, 8, -1)] +
                         [("case118_synth", True, G) for G in (1, -1)] +
                         [("case2000_synth", False, G) for G in (0, 1, 2, -1)])
@pytest.mark.parametrize("prec", [FP64, FP32_STRICT])
def test_contingencies_on_a_repivoted_plan(gpu_ctx, oracle_mod, name, single, G, prec):
    from lightsim2grid_amd import gridgen
    _say("scalar plan, contingencies", name, single, G, prec)
    g = gridgen.make(name)
    d, gr, Yx, Vb = _repivoted(gpu_ctx, oracle_mod, name, single)
    lines = np.nonzero(~gridgen.bridges(g))[0]
    deltas = _deltas(g, d, np.random.default_rng(1).choice(lines, 11, replace=False))
    Vr, itr, _, conv, _, _ = oracle_mod.contingency(d["Ybus"], d["Sbus"], *_args(d), d["V0"], deltas, 10, 1e-8, True, single, 4)
    r = gr.solve(Yx, d["Sbus"], Vb, 10, 1e-8, precision=prec, deltas=deltas, instances_per_wg=G)
    st = r["stats"]
    assert st["instances_per_wg"] == (G or st["instances_per_wg"]) and st["repivot_rows"] == 0
    if G == -1:
        assert st["workgroups"] > 11  # the wide kernel's, on one instance after the other
    assert np.array_equal(r["status"] == 0, conv)
    assert np.max(np.abs(r["iters"][conv] - itr[conv])) <= (0 if prec == FP64 else 1)
    assert np.max(np.abs(r["V"][conv] - Vr[conv])) <= (1e-8 if prec == FP64 else 5e-8)
    gr.close()


@pytest.mark.parametrize("name,G", [("case118_synth", 0), ("case118_synth", 2), ("case118_synth", -1),
                                    ("case2000_synth", 1), ("case2000_synth", -1)])
@pytest.mark.parametrize("prec,chain_len", [(FP64, None), (FP64, 4), (FP32_STRICT, 4)])
def test_chains_on_a_repivoted_plan(gpu_ctx, oracle_mod, name, G, prec, chain_len):
    from lightsim2grid_amd import gridgen
    _say("scalar plan, chains", name, G, prec, chain_len)
    g = gridgen.make(name)
    d, gr, Yx, _ = _repivoted(gpu_ctx, oracle_mod, name)
    T = 8
    Sb = np.concatenate([gridgen.time_series_sbus(g, T, seed=3), np.zeros((T, 1))], axis=1)
    # (from the flat start: the oracle's chains choose their pivots at their heads)
    Vr, itr, _, conv, _, _ = oracle_mod.time_series(d["Ybus"], Sb, *_args(d), d["V0"], 10, 1e-8, False, T // (chain_len or T))
    assert conv.all()
    r = gr.solve_chains(Yx, Sb, d["V0"], chain_len=chain_len, precision=prec, instances_per_wg=G)
    assert np.all(r["status"] == 0)
    assert np.max(np.abs(r["iters"] - itr)) <= (0 if prec == FP64 else 1)
    assert np.max(np.abs(r["V"] - Vr)) <= (1e-8 if prec == FP64 else 5e-8)
    gr.close()


@pytest.mark.parametrize("G", [0, 1, 4])
def test_fast_decoupled_on_a_repivoted_plan(gpu_ctx, oracle_mod, G):
    from lightsim2grid_amd import abi, gridgen
    _say("scalar plan, fast-decoupled", G)
    g = gridgen.make("case118_synth")
    ends = ENDS["case118_synth"]
    d = zero_diagonal_grid(*ends, name="case118_synth")
    line = lambda v, a, b: np.r_[v, a, b]  # noqa: E731
    Bp, Bpp = oracle_mod.fdpf_matrices(g.n + 1, line(g.f, g.n, g.n), line(g.t, *ends), line(g.r, 0, 0),
                                       line(g.x, 0.05, -0.05), 1j * line(g.b, 0, 0), "XB")
    assert Bp[g.n, g.n] == 0
    gr = abi.Grid(gpu_ctx, d["Ybus"], *_args(d), fdpf=(Bp, Bpp))
    rng = np.random.default_rng(5)
    Sb = d["Sbus"][None, :] * (1 + 0.05 * rng.standard_normal((6, g.n + 1)))
    for again in (False, True):  # the first solve chooses the pivots, the second keeps them
        r = gr.solve(gr.ybus_values(d["Ybus"]), Sb, d["V0"], 30, 1e-8, precision=FP64, instances_per_wg=G)
        assert r["stats"]["repivot_rows"] == (0 if again else 6)
        for k in range(6):
            Vr, itr, err = oracle_mod.fdpf(d["Ybus"], d["V0"], Sb[k], *_args(d), Bp, Bpp, 30, 1e-8)
            assert err == 0 and r["status"][k] == 0 and r["iters"][k] == itr
            assert np.max(np.abs(r["V"][k] - Vr)) <= 1e-8
    gr.close()
