"""What the serving loop reckons for an instance's workspace: requests that a budget holds are run."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


# bytes per instance: Va, Vm and Ibus rows, the FP64 values of the scalar plan (8 bytes a slot: 30 153 slots for the
# 2000-bus grid, 1547 for the 118-bus one, 140 859 for 10 000), flags; buffers of Sbus and V rows, iterations, status
@pytest.mark.parametrize("name,rows,per_instance", [("case2000_synth", 64, 305_288 + 64_012),
                                                    ("case118_synth", 100, 16_216 + 3_788),
                                                    ("case10000_synth", 12, 1_446_936 + 320_012)])
def test_request_that_fills_the_budget_runs(oracle_mod, name, rows, per_instance):
    import lightsim2grid_amd as L
    from lightsim2grid_amd import gridgen
    _say("serving, filled budget", name, rows)
    g = gridgen.make(name)
    d = g.solver_inputs()
    o = oracle_mod.OracleNR(False)
    assert o.compute_pf(d["Ybus"], d["V0"], d["Sbus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], 10, 1e-8)
    S = np.repeat(np.asarray(d["Sbus"])[None, :], rows, axis=0)
    V = []
    for budget in (0, rows * per_instance + 4):  # ample, and filled by the request
        sl = L.lightsim2grid_amd_cpp.ServeLoop(budget, rows, 0)
        gid = sl.add_grid(d["Ybus"], d["Sbus"], o.get_V(), d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], 10, 1e-8)
        r = sl.result(sl.submit_time_series(gid, S), 20.0)
        assert r is not None, "the request was never admitted"
        assert np.all(np.asarray(r["status"]) == 0)
        V.append(np.asarray(r["V"]))
        if budget == 0:
            sl.close()
    assert np.array_equal(V[0], V[1])
    with pytest.raises(RuntimeError):  # half as much again does not fit
        sl.submit_time_series(gid, np.repeat(S, 2, axis=0)[:rows + rows // 2 + 1])
    sl.close()
